"""The block Jacobi eigensolvers (one workgroup and the whole GPU), whose
32-wide subproblems run in one wave each: partial last blocks, odd and even
block counts, against the oracle."""

import numpy as np
import pytest

import oracle.gfn1 as og
from dxtb_amd import workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem
from helpers import TIGHT, TIGHT_ORACLE, run_native

pytestmark = pytest.mark.gpu


# orbitals: 264 (17 blocks, the last half full), 272 (17), 296 (19, half full)
# and 320 (20)
@pytest.mark.parametrize("size", [33, 34, 37, 40])
def test_orbital_energies_from_full_eigensolves(size):
    """Full eigensolves only; the SCF's 1e-11 threshold leaves energies
    quadratic and orbital energies linear in it, so 1e-9 and 1e-8 hold with
    room for ~100 sums of rounding."""
    z, p = workloads.water_cluster(np.random.default_rng(size), size)
    r = og.singlepoint(z, p, opts=TIGHT_ORACLE)
    full = {"eig_inexact": 0.0, "bd_gap_kt": 0.0}
    pipe = run_native([(z, p)], orbital_energies=True, **full)
    n = int(pipe.L.n[0])
    assert abs(float(pipe.energies()[0]) - r["energy"]) < 1e-9
    assert np.abs(pipe.emo[:n].cpu().numpy() - r["emo"].numpy()).max() < 1e-8
    c = pipe.matrix(pipe.C, 0).cpu().numpy()
    s = pipe.matrix(pipe.S, 0).cpu().numpy()
    assert np.abs(c @ s @ c.T - np.eye(n)).max() < 1e-10
    # the whole-GPU path's, small systems too: one and two subproblems a round
    for z, p, e in [(z, p, r["energy"])] + [
        (*w, og.singlepoint(*w, opts=TIGHT_ORACLE)["energy"])
        for w in (workloads.water_cluster(np.random.default_rng(k), k) for k in (1, 6))
    ]:
        g = LargeSystem(z, "cuda:0", opts=ScfOptions(**{**TIGHT, **full})).run(p)
        assert g["converged"] and abs(g["energy"] - e) < 1e-9
