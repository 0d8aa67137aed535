"""The form of the FP64 same-spin terms that the rule takes for small sets:
the dense blocks in one launch where the sets have excitations or are small,
the row kernels for random strings that have few.  The products of both forms
add the same terms in another order: 1e-12 of the largest value."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb,form", [
    ("scattered", 40, 5, 100, 5, 100, "dense"),
    ("scattered", 40, 5, 600, 5, 600, "sparse"),
    ("scattered", 40, 5, 900, 4, 300, "sparse"),
    ("scattered", 40, 5, 100, 4, 1100, "dense"),
    ("blocks", 18, 5, 600, 5, 600, "dense"),
    ("blocks", 24, 5, 900, 4, 300, "dense"),
])
def test_small_sets_by_their_entries(kind, norb, ea, na, eb, nb, form, monkeypatch):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 21)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 22)
    v = random_vector(na * nb, 5)
    print(f"[same rule] {kind} norb {norb} {na} x {nb}", flush=True)
    out = []
    for fixed in (None, "sparse" if form == "dense" else "dense"):
        if fixed:
            monkeypatch.setenv("SBDX_SAME_SPIN", fixed)
        op = sbdx.TPBOperator(norb, I0, I1, I2, a, b)
        out.append(op.sigma(v))
        if not fixed:
            assert op.same_spin_forms()["fp64"]["form"] == form
        op.close()
    assert np.max(np.abs(out[0] - out[1])) <= 1e-12 * np.max(np.abs(out[1]))
