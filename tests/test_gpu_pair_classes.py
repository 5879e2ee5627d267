"""Integrals and gradient of the one-launch path, whose pairs are dealt by
class, against the batched kernels: no p shells, only atoms with them, one
atom, around a wave's width of shells and of pairs, several rounds."""

import numpy as np
import pytest

from dxtb_amd import workloads
from helpers import block, run_native

pytestmark = pytest.mark.gpu


def _line(z, d):
    return np.array(z), np.stack([np.zeros(len(z)), 0.2 * np.arange(len(z)) % 0.7, d * np.arange(len(z))], axis=1)


MOLECULES = {
    "hydrogens": _line([1] * 4, 1.5),
    "nitrogen": _line([7, 7], 2.1),
    "oxygen": _line([8], 1.0),
    "water": workloads.water_cluster(np.random.default_rng(1), 1),
    "methane": workloads.chain(np.random.default_rng(2), 1),
    "octane": workloads.chain(np.random.default_rng(3), 8),
    "waters": workloads.water_cluster(np.random.default_rng(4), 22),
    "chain": workloads.chain(np.random.default_rng(5), 30),
}


@pytest.mark.parametrize("name", MOLECULES)
def test_one_launch_equals_the_batched_kernels(name):
    """Per pair the same operations: S, H0, gamma, CN and the repulsion to the
    bit.  The gradient's sums run in another order (~1e-12 of terms below 1
    Eh/bohr); with 40 times the SCF threshold of 1e-11 for the states: 1e-9."""
    m = MOLECULES[name]
    a = run_native([m], forces=True, fused=True)
    b = run_native([m], forces=True, fused=False)
    nsh = int(a.L.nsh[0])
    for k in ("S", "H0"):  # (the buffers are larger than the matrices)
        assert np.array_equal(block(a, getattr(a, k), 0), block(b, getattr(b, k), 0)), k
    for k, size in (("gamma", nsh * nsh), ("cn", len(m[0]))):
        assert np.array_equal(getattr(a, k)[:size].cpu().numpy(), getattr(b, k)[:size].cpu().numpy()), k
    from dxtb_amd import _lib

    assert a.records()[0, _lib.OUT_EREP] == b.records()[0, _lib.OUT_EREP]
    assert (a.gradient() - b.gradient()).abs().max() < 1e-9
