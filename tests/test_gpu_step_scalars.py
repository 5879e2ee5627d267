"""The one-workgroup parts of an SCF step (sort, Fermi smearing, Anderson
mixing) where they can go wrong: exactly equal levels, both spin channels,
every history length, one key per thread and more."""

import numpy as np
import pytest

import oracle.gfn1 as og
from dxtb_amd import workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem
from helpers import TIGHT, TIGHT_ORACLE, run_native

pytestmark = pytest.mark.gpu


def _twins():
    """Two identical water molecules 200 bohr apart: every level twice."""
    z, p = workloads.water_cluster(np.random.default_rng(3), 1)
    return np.concatenate([z, z]), np.concatenate([p, p + np.array([200.0, 0.0, 0.0])])


@pytest.mark.parametrize("generations", [1, 2, 3, 4, 5, 6])
def test_history_lengths_and_equal_levels(generations):
    """The fixed point does not depend on the mixer: energies to 1e-9 at the
    1e-11 threshold, on both paths."""
    for z, p in (_twins(), workloads.water_cluster(np.random.default_rng(11), 11)):
        e = og.singlepoint(z, p, opts=TIGHT_ORACLE)["energy"]
        k = run_native([(z, p)], generations=generations, maxiter=200)
        assert abs(float(k.energies()[0]) - e) < 1e-9
        g = LargeSystem(z, "cuda:0", opts=ScfOptions(**{**TIGHT, "generations": generations, "maxiter": 200})).run(p)
        assert g["converged"] and abs(g["energy"] - e) < 1e-9


# orbitals: 512 and 520, on both sides of one key per thread; 672 and 688
@pytest.mark.parametrize("size", [64, 65, 84, 86])
@pytest.mark.parametrize("spin", [0, 2])
def test_large_sorts_and_channels(size, spin):
    """Orbital energies in ascending order; both channels filled with their
    electrons to the Fermi threshold."""
    z, p = workloads.water_cluster(np.random.default_rng(size), size)
    opts = ScfOptions(**{**TIGHT, "orbital_energies": True, "fermi_etemp": 5000.0})
    big = LargeSystem(z, "cuda:0", spin=spin, opts=opts)
    assert big.run(p)["converged"]
    n = int(big.pipe.L.n[0])
    emo = big.pipe.emo[:n].cpu().numpy()
    assert n == 8 * size and (np.diff(emo) >= 0.0).all()
    occ = big.pipe.occ.reshape(2, -1)[:, :n].sum(dim=1).cpu().numpy()
    nel = 8 * size
    assert np.abs(occ - np.array([nel + spin, nel - spin]) / 2).max() < 1e-4
