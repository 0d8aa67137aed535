"""Slots per thread and pairs a round that the rule takes for the symmetric
products: a row of 1100 strings over two blocks where the Hartree-Fock bra's
rounds are most of the launch, over one where they are not, and two pairs a
round where no bra has more than a single.  The symmetric product against the
general one (the same terms in another order: 1e-12 of the largest value; in
FP32 2e-6 of the norm)."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings
from test_gpu_symmetry import symmetric_part

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,e,n,width,slots", [
    ("blocks", 28, 6, 1100, 16, 1),
    ("blocks", 20, 5, 1100, 16, 2),
    ("blocks", 16, 5, 275, 4, 1),
    ("scattered", 36, 6, 275, 16, 1),
])
def test_symmetric_configuration_by_the_sets(kind, norb, e, n, width, slots):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, e, n, 3)
    inst = dict(norb=norb, I0=I0, I1=I1, I2=I2, astr=a, bstr=a.copy())
    v = symmetric_part(inst, random_vector(n * n, 9))
    print(f"[mixed slots] {kind} norb {norb} {n}", flush=True)
    op = sbdx.TPBOperator.from_instance(inst)
    s, ss, s32 = op.sigma(v), op.sigma_sym(v), op.sigma_sym(v, fp32=True)
    forms = op.same_spin_forms()
    op.close()
    assert forms["fp64"]["sym_mixed_width"] == width
    assert forms["fp64"]["sym_mixed_slots_per_thread"] == slots
    assert forms["fp32"]["sym_mixed_width"] == 16 and forms["fp32"]["sym_mixed_slots_per_thread"] == slots
    assert np.max(np.abs(ss - s)) <= 1e-12 * np.max(np.abs(s))
    assert np.linalg.norm(s32 - s) <= 2e-6 * np.linalg.norm(s)


@pytest.mark.parametrize("kind,norb,na,nb,slots", [
    ("blocks", 34, 60, 5000, 1),         # one long bra of few
    ("blocks", 30, 130, 3000, 1),
    ("blocks", 30, 900, 3000, 2),        # from here on FP64 takes the block kernel
    ("scattered", 30, 900, 3000, 4),     # CUs filled by the bras alone
    ("scattered", 34, 900, 5000, 8),
])
def test_general_configuration_by_the_sets(kind, norb, na, nb, slots, monkeypatch):
    """The general form's slots where the sets differ: more blocks a bra for
    few bras and for long ones.  Against the entry-list kernel (the same terms
    in another order, the tolerances above)."""
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a, b = _strings(kind, norb, 6, na, 3), _strings(kind, norb, 5, nb, 5)
    v = random_vector(na * nb, 9)
    out = []
    for eb in (None, "2"):
        if eb:
            monkeypatch.setenv("SBDX_MIXED_EB", eb)
        print(f"[mixed slots] {kind} norb {norb} {na} x {nb} pairs {eb}", flush=True)
        op = sbdx.TPBOperator(norb, I0, I1, I2, a, b)
        out.append((op.sigma(v), op.sigma_fp32(v), op.same_spin_forms()))
        op.close()
    for p in ("fp64", "fp32"):
        forms = out[0][2][p]
        if p == "fp64" and na == 900:
            assert forms["mixed_width"] == 32
            continue
        assert forms["mixed_width"] == 16 and forms["mixed_slots_per_thread"] == slots
    (s, s32, _), (r, _, _) = out
    assert np.max(np.abs(s - r)) <= 1e-12 * np.max(np.abs(r))
    assert np.linalg.norm(s32 - r) <= 2e-6 * np.linalg.norm(r)
