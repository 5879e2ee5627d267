"""Cholesky orthogonalisation by register-held 32-wide diagonal blocks: one
partial, one full and several blocks, cold and warm, on both SCF paths."""

import numpy as np
import pytest

import oracle.gfn1 as og
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem
from helpers import TIGHT, TIGHT_ORACLE, run_native

pytestmark = pytest.mark.gpu


def _hydrogen(k):
    """k H2 molecules on a square grid, 4 orbitals each."""
    rng = np.random.default_rng(k)
    c = 5.0 * np.array([[i % 4, i // 4, 0] for i in range(k)], dtype=float)
    d = rng.normal(size=(k, 3))
    d *= 0.72 / np.linalg.norm(d, axis=1, keepdims=True)
    return np.ones(2 * k, dtype=np.int64), np.stack([c - d, c + d], axis=1).reshape(-1, 3)


# 4, 28, 32, 36, 64 and 68 orbitals
@pytest.mark.parametrize("k", [1, 7, 8, 9, 16, 17])
def test_orthonormal_orbitals_and_energy(k):
    """C S C^T = 1 to ~n roundings of well-conditioned hydrogens; the SCF's
    1e-11 threshold leaves the energy below 1e-9."""
    z, p = _hydrogen(k)
    e = og.singlepoint(z, p, opts=TIGHT_ORACLE)["energy"]
    pipe = run_native([(z, p)])
    n = int(pipe.L.n[0])
    assert n == 4 * k and abs(float(pipe.energies()[0]) - e) < 1e-9
    c = pipe.matrix(pipe.C, 0).cpu().numpy()
    s = pipe.matrix(pipe.S, 0).cpu().numpy()
    assert np.abs(c @ s @ c.T - np.eye(n)).max() < 1e-12
    g = LargeSystem(z, "cuda:0", opts=ScfOptions(**TIGHT)).run(p)
    assert g["converged"] and abs(g["energy"] - e) < 1e-9
