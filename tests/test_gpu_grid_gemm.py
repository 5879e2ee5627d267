"""The whole-GPU path's grid GEMM over its tile choices and edges, through the
single points built from it, against the per-molecule kernel.

With n orbitals, k doubly occupied and m = n - k virtual ones its products are
(k, n, n), (k, m, n), (k, n, k), (m, n, k) and symmetric n x n and k x k: the
sizes leave 1 to 15 of a fragment row or k chunk, give single tiles, and lie
on both sides of the lines between 16-, 32- and 48-wide tiles (the 96-wide
ones run in the 600-water test)."""

import numpy as np
import pytest

from dxtb_amd import workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem
from helpers import TIGHT, run_native

pytestmark = pytest.mark.gpu


# (n, k): (12, 4), (52, 19), (132, 49), (188, 70), (356, 133), (480, 240), (800, 400)
@pytest.mark.parametrize("kind,size", [("chain", 1), ("chain", 6), ("chain", 16), ("chain", 23), ("chain", 44),
                                       ("water", 60), ("water", 100)])
def test_whole_gpu_path_equals_the_per_molecule_kernel(kind, size):
    """Two independent products of the same SCF at a 1e-11 threshold: energies
    to 1e-9 Eh, forces (below 40 times the threshold) to 1e-8 Eh/bohr."""
    rng = np.random.default_rng(500 + size)
    z, p = workloads.water_cluster(rng, size) if kind == "water" else workloads.chain(rng, size, p_n=0.0, p_o=0.0)
    r = LargeSystem(z, "cuda:0", opts=ScfOptions(**TIGHT)).run(p, forces=True)
    assert r["converged"] and r["status"] == 0
    k = run_native([(z, p)], forces=True)
    assert abs(k.energies().item() - r["energy"]) < 1e-9
    assert np.abs(k.gradient().cpu().numpy() - r["gradient"].cpu().numpy()).max() < 1e-8
