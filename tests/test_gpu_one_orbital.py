"""A padded molecule of one orbital, which the C interface takes though no
supported element has so few: products over one orbital in a perturbative
step."""

import ctypes as ct

import numpy as np
import pytest
import torch

from dxtb_amd import _lib
from dxtb_amd.engine import ScfOptions
from helpers import run_native

pytestmark = pytest.mark.gpu

OUT_EFERMI_A = 7  # slot of the result record (include/xtb_hip.h)


def _fermi_levels(pd_kmax):
    mols = [(np.array([1]), np.zeros((1, 3))), (np.array([1, 1]), np.array([[0.0, 0.0, 0.0], [0.0, 0.0, 1.5]]))]
    pipe = run_native(mols, padded=True)
    n = int(pipe.L.n[0])
    assert n == 4 and int(pipe.L.vec0[0]) == 0 and int(pipe.L.atom0[0]) == 0
    # the first molecule cut to its lower shell: one orbital, two electrons
    for name, at, value in (("mol_nao", 0, 1), ("mol_nsh", 0, 1), ("atom_nsh", 0, 1), ("ao_sh", 1, -1),
                            ("mol_nel", 0, 1.0), ("mol_nel", 1, 1.0), ("n0", 0, 1.0), ("n0", 1, 0.0)):
        pipe.d[name][at] = value
    pipe.matrix(pipe.S, 0).copy_(torch.eye(n, dtype=torch.float64))
    pipe.matrix(pipe.H0, 0).zero_()[0, 0] = -0.5
    pipe.gamma[int(pipe.L.gam0[0])] = 0.4
    o = ScfOptions(x_atol=1e-10, x_atol_max=1e-10, pd_kmax=pd_kmax).to_struct(want_w=False, padded=True)
    s = ct.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(pipe.lib.xtb_scf(ct.byref(pipe.batch), ct.byref(pipe.dt.s), pipe.S.data_ptr(), pipe.H0.data_ptr(),
                                pipe.gamma.data_ptr(), ct.byref(o), ct.byref(pipe.state), s), "xtb_scf")
    torch.cuda.synchronize()
    rec = pipe.records()[0]
    assert rec[_lib.OUT_STATUS].item() == 0
    return float(rec[_lib.OUT_PD_STEPS]), float(rec[OUT_EFERMI_A]), float(rec[_lib.OUT_ESCF])


def test_perturbative_steps_of_one_orbital():
    """The orbital's energy follows its potential in perturbative steps as in
    full eigensolves: the same Fermi level, with no rounding but the sums'."""
    steps, ef, e = _fermi_levels(0.2)
    none, ref, eref = _fermi_levels(0.0)
    assert steps > 0 and none == 0
    assert abs(ef - ref) < 1e-12 and abs(e - eref) < 1e-12
