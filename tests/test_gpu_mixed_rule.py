"""The form of the FP64 mixed term that the rule takes: the block kernel (width
32) where blocks of singles fill its steps, where a short set or one long bra
makes it the faster one; the signed-triangle kernel (width 16) on sets whose
blocks are thin and on few bras.  Each against the other form, whose sums are
the same terms in another order (at most some 1e5 per element): 1e-12 of the
largest value."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb,width", [
    ("blocks", 16, 5, 300, 4, 297, 32),        # a short set
    ("scattered", 24, 5, 500, 4, 512, 32),
    ("blocks", 28, 6, 1900, 5, 1997, 32),      # full steps
    ("blocks", 36, 8, 600, 8, 597, 32),        # one long bra
    ("blocks", 34, 6, 2500, 4, 900, 32),       # many bras, a short set
    ("scattered", 28, 6, 2000, 5, 1997, 32),   # no blocks
    ("scattered", 16, 5, 600, 4, 597, 16),     # thin blocks
    ("scattered", 24, 5, 2000, 4, 3997, 16),
    ("scattered", 34, 6, 90, 4, 3000, 16),     # few bras
    ("blocks", 30, 6, 10, 6, 3000, 16),
    ("blocks", 24, 5, 100, 4, 1100, 32),       # few bras, full steps in four groups
    ("blocks", 30, 6, 300, 5, 3000, 16),       # one long bra, rows split instead
])
def test_mixed_form_by_the_sets(kind, norb, ea, na, eb, nb, width, monkeypatch):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a, b = _strings(kind, norb, ea, na, 3), _strings(kind, norb, eb, nb, 5)
    v = random_vector(na * nb, 9)
    print(f"[mixed rule] {kind} norb {norb} {na} x {nb}", flush=True)
    out = []
    for fixed in (None, "16" if width == 32 else "2"):
        if fixed:
            monkeypatch.setenv("SBDX_MIXED_EB", fixed)
        op = sbdx.TPBOperator(norb, I0, I1, I2, a, b)
        out.append(op.sigma(v))
        assert op.same_spin_forms()["fp64"]["mixed_width"] == (int(fixed) if fixed else width)
        op.close()
    assert np.max(np.abs(out[0] - out[1])) <= 1e-12 * np.max(np.abs(out[1]))
