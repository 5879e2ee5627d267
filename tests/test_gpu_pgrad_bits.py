"""Exponent gradients of molecules of at most 16 atoms (one tile of atom pairs):
the same bits on every run."""

import numpy as np
import pytest
import torch

from dxtb_amd import workloads
from dxtb_amd.param import SpeciesTables
from helpers import run_native

pytestmark = pytest.mark.gpu


def test_small_molecules_have_the_same_bits_on_every_run():
    """64 molecules of 5 to 16 atoms, one that fills the tile among them."""
    rng = np.random.default_rng(17)
    mols = [workloads.chain(rng, 1 + k % 4) for k in range(62)]
    mols += [workloads.water_cluster(rng, 5), (np.ones(16, dtype=np.int64), 3.0 * np.stack(
        np.meshgrid(np.arange(4), np.arange(2), np.arange(2), indexing="ij"), -1).reshape(-1, 3) + 0.0)]
    assert max(len(z) for z, _ in mols) == 16
    pipe = run_native(mols, forces=True)
    tables = SpeciesTables(np.unique(np.concatenate([z for z, _ in mols])))
    first = pipe.param_grad_basis(tables)
    assert torch.isfinite(first).all()
    for _ in range(20):
        assert torch.equal(pipe.param_grad_basis(tables), first)
