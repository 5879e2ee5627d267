"""Molecules just below the per-molecule kernel's limit of 1024 orbitals, whose
vectors leave the least LDS for the matrices: through a batch and through the
server, against the whole-GPU path."""

import numpy as np
import pytest
import torch

from dxtb_amd import GFN1Calculator, workloads
from dxtb_amd.engine import WG_MAX_N, Pipeline, ScfOptions
from dxtb_amd.large import LargeSystem
from dxtb_amd.serving import RaggedServer, Request
from helpers import TIGHT, TIGHT_ORACLE

pytestmark = pytest.mark.gpu


def _hydrogen(count, seed):
    """`count` H2 molecules on a cubic lattice (4 orbitals each), bohr."""
    rng = np.random.default_rng(seed)
    side = int(np.ceil(count ** (1 / 3)))
    sites = 6.5 * np.array([(i, j, k) for i in range(side) for j in range(side) for k in range(side)][:count])
    axis = rng.normal(size=sites.shape)
    axis *= 0.7 / np.linalg.norm(axis, axis=1, keepdims=True)
    return np.ones(2 * count, dtype=np.int64), np.stack([sites - axis, sites + axis], axis=1).reshape(-1, 3)


def _molecules():
    rng = np.random.default_rng(61)
    return [workloads.water_cluster(rng, 115), workloads.water_cluster(rng, 128), workloads.chain(rng, 8),
            _hydrogen(256, 62)]


@pytest.mark.parametrize("pick", [(0, 2), (1, 2), (3, 2)], ids=["920", "1024", "1024-hydrogen"])
def test_batch(pick):
    """One launch of the largest and a small molecule.  Two independent paths
    at a 1e-11 threshold: energies to 1e-9 Eh, forces to 1e-8 Eh/bohr."""
    mols = [_molecules()[i] for i in pick]
    nums, pos = workloads.pad(mols)
    dev = torch.device("cuda:0")
    print(f"case: batch of {[len(z) for z, _ in mols]} atoms", flush=True)
    calc = GFN1Calculator(torch.tensor(nums, device=dev), dtype=torch.float64, device=dev,
                          opts={**TIGHT_ORACLE, "exclude": ["disp"]})
    p = torch.tensor(pos, dtype=torch.float64, device=dev)
    e = calc.get_energy(p).cpu().numpy()
    f = calc.forces_analytical(p).cpu().numpy()
    assert type(calc._pipe) is Pipeline and int(calc._pipe.L.n.max()) <= WG_MAX_N
    for b, (z, x) in enumerate(mols):
        r = LargeSystem(z, "cuda:0", opts=ScfOptions(**TIGHT)).run(x)
        assert r["status"] == 0
        assert abs(e[b] - r["energy"]) < 1e-9
        assert np.abs(f[b, : len(z)] + r["gradient"].cpu().numpy()).max() < 1e-8


def test_server():
    mols = _molecules()[:3]
    print("case: serving requests of 920 and 1024 orbitals", flush=True)
    srv = RaggedServer("cuda:0", opts=ScfOptions(**TIGHT))
    reqs = [Request(i, z, x, arrival=0.0) for i, (z, x) in enumerate(mols)]
    srv.run_stream(reqs, realtime=False)
    assert srv.stats.completed == len(reqs) and srv.stats.large_runs == 0
    for q in reqs:
        r = LargeSystem(q.numbers, "cuda:0", opts=ScfOptions(**TIGHT)).run(q.positions)
        got = srv.results[q.rid]
        assert got.status == 0 and abs(got.energy - r["energy"]) < 1e-9
        assert np.abs(got.forces + r["gradient"].cpu().numpy()).max() < 1e-8
