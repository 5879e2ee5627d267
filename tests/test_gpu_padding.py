"""Padded batches: the products leave the padding orbitals out and an
eigensolve puts them at their place in the spectrum.  A call that keeps its
state for the next one runs over all orbitals instead; both must agree."""

import numpy as np
import pytest

from dxtb_amd import workloads
from helpers import run_native

pytestmark = pytest.mark.gpu

# closed shells, radicals (an eigensolve in every step), and anions whose
# electrons reach levels above 0, where padding orbitals get occupied
CASES = {
    "closed": ([0, 0, 0, 0], None, {}),
    "orbitals": ([0, 0, 0, 0], None, {"orbital_energies": True}),
    "cations": ([1, 1, 1, 1], None, {"fermi_etemp": 3000.0}),
    "anions": ([-2, -2, -2, -2], None, {"fermi_etemp": 3000.0}),
    "loewdin": ([0, 0, 0, 0], None, {"ortho": 0}),
}


# the largest decides the layout: 52 orbitals, 100 (two eigenvalue counts per
# lane), 204 (block Jacobi, most molecules with blocks of padding only)
@pytest.mark.parametrize("largest", [6, 12, 25])
@pytest.mark.parametrize("case", CASES)
def test_padded_products_equal_the_general_ones(case, largest):
    """Two runs of the same SCF at a 1e-11 threshold: energies to 1e-9,
    forces (below 40 times the threshold) to 1e-8; one more sum over the
    occupations, the -TS term, to 1e-9."""
    chrg, spin, opt = CASES[case]
    mols = [workloads.chain(np.random.default_rng(70 + k), k, p_n=0.0, p_o=0.0) for k in (1, 3, largest - 1, largest)]
    a, b = (run_native(mols, padded=True, forces=True, chrg=chrg, spin=spin, warm_start=w, **opt) for w in (False, True))
    ra, rb = a.records().cpu().numpy(), b.records().cpu().numpy()
    assert (a.energies() - b.energies()).abs().max() < 1e-9
    assert (a.gradient() - b.gradient()).abs().max() < 1e-8
    from dxtb_amd import _lib

    assert (ra[:, _lib.OUT_STATUS] == rb[:, _lib.OUT_STATUS]).all()
    assert np.abs(ra[:, _lib.OUT_FENERGY] - rb[:, _lib.OUT_FENERGY]).max() < 1e-9
    if opt.get("orbital_energies"):
        assert np.abs(a.emo.cpu().numpy() - b.emo.cpu().numpy()).max() < 1e-8
