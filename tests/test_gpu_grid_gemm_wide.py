"""The grid GEMM's 96-wide tiles at sizes that fill none of their fragments or k
chunks: a chain of 540 carbons, n = 4324 orbitals, k = 1621 of them occupied
(4324 = 45 x 96 + 4 = 270 x 16 + 4, 1621 = 202 x 8 + 5).  From about 1000 tiles
on they carry the products (n, n, n), plain, transposed and symmetric, (m, n, k)
added to C, and both series side by side (k, 2 n, k)."""

import numpy as np
import pytest
import torch

from dxtb_amd import _lib, workloads
from dxtb_amd.engine import ScfOptions
from dxtb_amd.large import LargeSystem

pytestmark = pytest.mark.gpu


def test_self_consistent_solution_of_a_long_chain():
    """What the SCF's result has to satisfy, formed with torch in FP64 from the
    returned S, H0, potential, P and W.  Sums of n terms of order 1 leave
    ~1e-12; the final coupling (a tenth of the threshold) bounds the
    commutator.  Products that lost a remainder would be off by ~1e-3."""
    z, p = workloads.chain(np.random.default_rng(29), 540, p_n=0.0, p_o=0.0)
    print("case: chain of 540 carbons on the whole GPU", flush=True)
    ls = LargeSystem(z, "cuda:0", opts=ScfOptions(x_atol=1e-9, x_atol_max=1e-9, maxiter=100))
    r = ls.run(p, forces=True)
    assert r["converged"] and r["status"] == 0 and r["records"][_lib.OUT_PD_STEPS] > 0
    pipe = ls.pipe
    n = int(pipe.L.n[0])
    assert n == 4324
    S, H0, P, W = (pipe.matrix(b, 0) for b in (pipe.S, pipe.H0, pipe.P, pipe.T))
    v = pipe.vnew[:n]  # the final step's input potential
    F = H0 - 0.5 * S * (v[:, None] + v[None, :])
    PS = P @ S
    assert abs(float(torch.diagonal(PS).sum()) - 3242.0) < 1e-8
    assert float((PS @ P - 2.0 * P).abs().max()) < 1e-9
    FP = F @ P
    assert float((FP @ S - (FP @ S).T).abs().max()) < 1e-8
    assert float((W - 0.5 * P @ FP).abs().max()) < 1e-8
    assert abs(float((P * H0).sum()) / float(r["records"][_lib.OUT_EH0]) - 1.0) < 1e-12
