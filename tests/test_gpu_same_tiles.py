"""The FP64 same-spin terms on tiles with ket lists, and in one launch for
small sets, over their edges: the last small size (na + nb = 1200) and the
first tiled one, string counts around a tile of 32 or 64 rows and a chunk of
128 or 256 columns, odd and even columns, equal and different sets, sets of
the Hartree-Fock string's excitations and scattered ones (mostly empty tiles,
short lists), one string.  Against the sparse row kernels, which add the same
terms in another order: at most some 1e4 per element, random in sign, so the
results differ by about 1e-16 sqrt(1e4) = 1e-14 of the largest value; 1e-12
of it.  The spin-flip symmetric product (one term and its transpose) likewise
against the general one."""
import os

import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings
from test_gpu_symmetry import symmetric_part

pytestmark = pytest.mark.gpu


def _sigma(inst, v, form):
    import sbdx
    old = os.environ.get("SBDX_SAME_SPIN")
    if form:
        os.environ["SBDX_SAME_SPIN"] = form
    try:
        op = sbdx.TPBOperator.from_instance(inst)
        s, again = op.sigma(v), op.sigma(v)
    finally:
        os.environ.pop("SBDX_SAME_SPIN", None)
        if old is not None:
            os.environ["SBDX_SAME_SPIN"] = old
    assert np.array_equal(s, again)
    return op, s


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb", [
    ("blocks", 12, 3, 1, 3, 1),
    ("blocks", 12, 3, 2, 3, 3),
    ("blocks", 12, 4, 17, 3, 130),
    ("blocks", 18, 5, 601, 4, 599),      # the last one-launch size
    ("blocks", 18, 5, 600, 4, 601),      # the first tiled one
    ("blocks", 24, 5, 1, 5, 1500),
    ("blocks", 24, 5, 1500, 5, 1),
    ("blocks", 24, 5, 2, 5, 1300),
    ("blocks", 24, 5, 1300, 5, 2),
    ("blocks", 24, 5, 1217, 4, 129),
    ("blocks", 24, 5, 1023, 4, 255),
    ("scattered", 40, 5, 700, 5, 613),
    ("blocks", 30, 6, 2881, 5, 2999),    # 64 x 64 tiles, odd columns
    ("blocks", 29, 6, 3000, 6, 3000),    # ... of one set, even columns
])
def test_same_spin_tiles(kind, norb, ea, na, eb, nb):
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 21)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 22)
    inst = dict(norb=norb, I0=I0, I1=I1, I2=I2, astr=a, bstr=b)
    print(f"[same tiles] {kind} norb {norb} {na} x {nb}", flush=True)
    v = random_vector(na * nb, 5)
    if np.array_equal(a, b):
        v = symmetric_part(inst, v)
    op, s = _sigma(inst, v, "dense")
    if np.array_equal(a, b):
        assert np.max(np.abs(op.sigma_sym(v) - s)) <= 1e-12 * max(np.max(np.abs(s)), 1e-300)
    op.close()
    op, ref = _sigma(inst, v, "sparse")
    op.close()
    assert np.max(np.abs(s - ref)) <= 1e-12 * max(np.max(np.abs(ref)), 1e-300)
