"""What a context's first products launch: where a rule gives the mixed term's
configuration, one mixed launch per product, the first included, and no time
is reported for it."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings
from test_gpu_symmetry import symmetric_part

pytestmark = pytest.mark.gpu


def test_a_rule_takes_no_product_of_its_own():
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(18, 3, 11)
    I0, I1, I2 = instances.pack_integrals(18, h, eri)
    a = _strings("blocks", 18, 5, 700, 3)
    inst = dict(norb=18, I0=I0, I1=I1, I2=I2, astr=a, bstr=a.copy())
    v = symmetric_part(inst, random_vector(a.size ** 2, 9))
    print("[first product] 700 x 700", flush=True)
    op = sbdx.TPBOperator.from_instance(inst)
    s, s32 = op.sigma(v), op.sigma_fp32(v)
    y, y32 = op.sigma_sym(v), op.sigma_sym(v, fp32=True)
    forms = op.same_spin_forms()
    assert np.max(np.abs(y - s)) <= 1e-12 * np.max(np.abs(s))
    for w in (s32, y32):
        assert np.linalg.norm(w - s) <= 2e-6 * np.linalg.norm(s)
    for k in ("fp64", "fp32"):
        assert forms[k]["mixed_ms"] == 0 and forms[k]["sym_mixed_ms"] == 0, forms
        assert forms[k]["mixed_width"] in (16, 32) and forms[k]["sym_mixed_width"] == 16
    op.close()
