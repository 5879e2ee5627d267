"""The LDS Jacobi eigensolver over its size range against the oracle.

Its rounds hold 1 to 10 blocks per thread (changes at 33, 46, 56, 73 and 85
pairs), its vector pass one ring position per lane up to 64 pairs and two
above, and runs of 4 to 16 columns."""

import numpy as np
import pytest

import oracle.gfn1 as og
from dxtb_amd import workloads
from helpers import TIGHT_ORACLE, run_native

pytestmark = pytest.mark.gpu


def _molecule(kind, size):
    rng = np.random.default_rng(1000 * len(kind) + size)
    if kind == "hydrogen":
        return np.array([1, 1]), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.5]])
    if kind == "water":
        return workloads.water_cluster(rng, size)
    return workloads.chain(rng, size)


# orbitals: 4, 8, 44, 64, 72, 92, 112, 128, 132, 148, 172, 188
@pytest.mark.parametrize("kind,size", [("hydrogen", 2), ("water", 1), ("chain", 5), ("water", 8), ("water", 9),
                                       ("chain", 11), ("water", 14), ("water", 16), ("chain", 16), ("chain", 18),
                                       ("chain", 21), ("chain", 23)])
def test_orbital_energies_over_the_size_range(kind, size):
    """Every step a full eigensolve (no occupation classes, no perturbative
    steps), then the default steps with the classes' own diagonalisation at
    the end: the SCF's 1e-11 threshold leaves energies quadratic and orbital
    energies linear in it, so 1e-9 and 1e-8 hold with room for ~100 sums of
    rounding."""
    z, p = _molecule(kind, size)
    r = og.singlepoint(z, p, opts=TIGHT_ORACLE)
    for opt in ({"eig_inexact": 0.0, "bd_gap_kt": 0.0}, {}):
        pipe = run_native([(z, p)], orbital_energies=True, **opt)
        n = int(pipe.L.n[0])
        assert abs(float(pipe.energies()[0]) - r["energy"]) < 1e-9
        assert np.abs(pipe.emo[:n].cpu().numpy() - r["emo"].numpy()).max() < 1e-8
        c = pipe.matrix(pipe.C, 0).cpu().numpy()
        s = pipe.matrix(pipe.S, 0).cpu().numpy()
        assert np.abs(c @ s @ c.T - np.eye(n)).max() < 1e-10
