"""The per-molecule kernels' LDS over the sizes that are sent to them (host-only
query): every molecule up to WG_MAX_N orbitals has a layout that fits a CU,
also those of hydrogen alone, with the most shells and atoms per orbital."""

import ctypes as ct

import pytest

from dxtb_amd import _lib
from dxtb_amd.engine import WG_MAX_N

CU_LDS = 160 * 1024


# orbitals, shells and atoms of a unit
@pytest.mark.parametrize("unit", [(8, 6, 3), (2, 2, 1), (4, 2, 1)], ids=["water", "hydrogen", "carbon"])
def test_every_size_has_a_layout(unit):
    lib = _lib.load()
    nbytes, cap = ct.c_int32(0), ct.c_int32(0)
    for u in range(1, WG_MAX_N // unit[0] + 1):
        n, nsh, nat = (u * x for x in unit)
        b = _lib.XtbBatch(nmol=1, max_n=n, max_nsh=nsh, max_nat=nat)
        rc = lib.xtb_scf_lds_bytes(ct.byref(b), ct.byref(nbytes), ct.byref(cap))
        assert rc == _lib.XTB_OK, f"{n} orbitals: status {rc}"
        # the vectors of a step (2 per orbital, 3 per shell, 1 per atom) lie
        # beside the matrix stage
        assert cap.value + 2 * n + 3 * nsh + nat <= nbytes.value // 8 and nbytes.value <= CU_LDS, n
