"""A string set that lists some strings twice: the copies are rows of their
own that do not couple to each other, in every form of the products and in
the density matrices, as the oracle has it (it sums over the pairs of listed
strings).  Sets of blocks, so that the copies lie in the blocks of singles,
for one and two tiles of orbitals, and a scattered set.

The sums have at most some 1e4 terms per element, random in sign: 1e-14 of
the largest value, 1e-12 allowed; density matrices of |w| = 1 likewise."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb", [
    ("blocks", 14, 4, 60, 4, 60),
    ("blocks", 16, 4, 90, 3, 80),
    ("blocks", 20, 3, 40, 4, 200),
    ("scattered", 14, 4, 70, 4, 111),
])
def test_repeated_strings(kind, norb, ea, na, eb, nb, oracle_mod):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 3)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 5)
    a, b = np.concatenate([a, a[:5]]), np.concatenate([b, b[3:9]])
    inst = dict(norb=norb, nelec=ea + eb, I0=I0, I1=I1, I2=I2, astr=a, bstr=b)
    print(f"[repeated strings] {kind} norb {norb} {na} x {nb}", flush=True)
    op = sbdx.TPBOperator.from_instance(inst)
    v = random_vector(op.ndet, 9)
    s = op.sigma(v)
    one, two = op.correlation(v)
    op.close()
    orc = oracle_mod.Oracle.from_instance(inst)
    o = orc.sigma(v, orc.diag())
    r1, r2 = (np.asarray(r).reshape(-1) for r in orc.rdm(v))
    orc.close()
    assert np.max(np.abs(s - o)) < 1e-12 * np.max(np.abs(o))
    assert np.max(np.abs(one - r1)) < 1e-12
    assert np.max(np.abs(two - r2)) < 1e-12
