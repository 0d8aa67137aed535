"""The RDM's two-spin kernel at the length of beta rows where they no longer
fit in LDS twice (8191 | 8192 strings) and beyond, rows read in place, against
the oracle; |w| = 1, so 1e-12 as in the tests of the columns."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb", [
    ("blocks", 36, 8, 3, 8, 8191),
    ("blocks", 36, 8, 3, 8, 8192),
    ("blocks", 16, 3, 4, 8, 9001),
    ("scattered", 30, 4, 3, 5, 12345),
])
def test_rdm_long_rows(kind, norb, ea, na, eb, nb, oracle_mod):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    inst = dict(norb=norb, nelec=ea + eb, I0=I0, I1=I1, I2=I2, astr=_strings(kind, norb, ea, na, 3),
                bstr=_strings(kind, norb, eb, nb, 5))
    print(f"[rdm long rows] {kind} norb {norb} {na} x {nb}", flush=True)
    op = sbdx.TPBOperator.from_instance(inst)
    W = random_vector(op.ndet, 9)
    one, two = op.correlation(W)
    op.close()
    orc = oracle_mod.Oracle.from_instance(inst)
    r1, r2 = (np.asarray(r).reshape(-1) for r in orc.rdm(W))
    orc.close()
    assert np.max(np.abs(one - r1)) < 1e-12
    assert np.max(np.abs(two - r2)) < 1e-12
