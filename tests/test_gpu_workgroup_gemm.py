"""The one-workgroup GEMM over the edges of its tiles, through the SCF and the
gradient that are built from it, against the oracle.

Products of a closed-shell molecule with n orbitals, k doubly occupied and m =
n - k virtual ones run as (k, n, n), (k, m, n), (k, n, k), (m, n, k) and as
symmetric n x n and k x k: k, m and n here leave 1, 2, 4 ... 15 of a 16-deep
panel or fragment row, fill one 176-wide tile exactly, need two or three, and
are too thin for the panel loads (one occupied or one virtual orbital)."""

import numpy as np
import pytest

import oracle.gfn1 as og
from dxtb_amd import workloads
from helpers import TIGHT_ORACLE, run_native

pytestmark = pytest.mark.gpu


def _molecule(kind, size):
    rng = np.random.default_rng(77 + size)
    if kind == "hydride":
        return np.array([1]), np.zeros((1, 3)), -1.0
    if kind == "hydrogen":
        return np.array([1, 1]), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.45]]), 0.0
    if kind == "water":
        return (*workloads.water_cluster(rng, size), 0.0)
    return (*workloads.chain(rng, size, p_n=0.0, p_o=0.0), 0.0)


# (n, k, m): (2, 1, 1), (4, 1, 3), (8, 4, 4), (52, 19, 33), (132, 49, 83), (176, 88, 88), (184, 92, 92),
# (188, 70, 118), (356, 133, 223)
@pytest.mark.parametrize("kind,size", [("hydride", 1), ("hydrogen", 2), ("water", 1), ("chain", 6), ("chain", 16),
                                       ("water", 22), ("water", 23), ("chain", 23), ("chain", 44)])
def test_energy_and_forces_at_tile_edges(kind, size):
    """At a 1e-11 threshold energies are quadratic and forces linear (with a
    factor below 40) in it: 1e-9 Eh and 1e-8 Eh/bohr."""
    z, p, q = _molecule(kind, size)
    r = og.singlepoint(z, p, chrg=q, opts=TIGHT_ORACLE, with_forces=True)
    pipe = run_native([(z, p)], forces=True, fused=True, chrg=[q])
    assert abs(float(pipe.energies()[0]) - r["energy"]) < 1e-9
    assert np.abs(-pipe.gradient().cpu().numpy() - r["forces"].numpy()).max() < 1e-8
    assert np.abs(pipe.orbital_charges(0).cpu().numpy() - r["charges_orbital"].numpy()).max() < 1e-8
