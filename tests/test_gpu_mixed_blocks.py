"""The FP64 mixed term by blocks of beta singles (width 32) over its edges: one
and two tiles of orbitals (and orbital counts at a tile's end and at the
largest triangle), sets made of blocks, of scattered strings (everything
outside the blocks) and of one string, string counts around a slice of 64 and
around the widths of a staged element (8191 | 8192 strings), more tasks than
the matrix waves hold (further launches), and a lowered LDS budget.

Against the form without blocks (one alpha single per round), whose sums are
the same terms in another order: at most some 1e5 terms per element, so their
rounding differs by 1e-16 sqrt(1e5) ~ 3e-14 of the largest value when the
terms are random in sign: 1e-12 of it.  The small ones also against the
oracle."""
import os

import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


def _sigma(inst, v, env):
    import sbdx
    old = {k: os.environ.get(k) for k in env}
    os.environ.update(env)
    try:
        op = sbdx.TPBOperator.from_instance(inst)
        s, again = op.sigma(v), op.sigma(v)
        width = op.same_spin_forms()["fp64"]["mixed_width"]
        op.close()
    finally:
        for k, o in old.items():
            os.environ.pop(k, None)
            if o is not None:
                os.environ[k] = o
    assert np.array_equal(s, again)
    return s, width


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb,lds", [
    ("blocks", 15, 4, 90, 4, 90, None),
    ("blocks", 16, 4, 120, 3, 131, None),
    ("blocks", 17, 5, 150, 4, 129, None),
    ("blocks", 33, 3, 70, 4, 300, None),
    ("blocks", 44, 3, 60, 3, 64, None),
    ("scattered", 14, 4, 70, 4, 111, None),
    ("scattered", 40, 3, 50, 3, 65, None),
    ("blocks", 12, 3, 1, 3, 1, None),
    ("blocks", 12, 3, 1, 4, 40, None),
    ("blocks", 18, 5, 300, 5, 1025, None),
    ("blocks", 14, 3, 4, 7, 3432, None),      # the whole space: 188 tasks
    ("blocks", 36, 8, 3, 8, 8191, None),      # the last of 16-byte elements
    ("blocks", 36, 8, 3, 8, 8192, None),
    ("blocks", 17, 5, 150, 4, 129, 9000),     # one group, a pass per task
])
def test_mixed_blocks(kind, norb, ea, na, eb, nb, lds, oracle_mod):
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 3)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 5)
    inst = dict(norb=norb, nelec=ea + eb, I0=I0, I1=I1, I2=I2, astr=a, bstr=b)
    print(f"[mixed blocks] {kind} norb {norb} {na} x {nb} lds {lds}", flush=True)
    v = random_vector(na * nb, 9)
    s, width = _sigma(inst, v, {"SBDX_LDS_LIMIT": str(lds)} if lds else {})
    assert width == 32
    ref, other = _sigma(inst, v, {"SBDX_MIXED_EB": "1"})
    assert other != 32
    tol = 1e-12 * np.max(np.abs(ref))
    assert np.max(np.abs(s - ref)) < tol
    if na * nb <= 50000:
        orc = oracle_mod.Oracle.from_instance(inst)
        o = orc.sigma(v, orc.diag())
        orc.close()
        assert np.max(np.abs(s - o)) < tol


def test_too_many_orbitals_keep_the_other_form(oracle_mod):
    """45 orbitals: the signed triangles pass the index field of an entry."""
    from sbdx import instances
    h, eri = instances.make_integrals(45, 3, 11)
    I0, I1, I2 = instances.pack_integrals(45, h, eri)
    inst = dict(norb=45, nelec=6, I0=I0, I1=I1, I2=I2, astr=_strings("blocks", 45, 3, 40, 3),
                bstr=_strings("blocks", 45, 3, 50, 5))
    v = random_vector(2000, 9)
    s, width = _sigma(inst, v, {})
    assert width != 32
    orc = oracle_mod.Oracle.from_instance(inst)
    o = orc.sigma(v, orc.diag())
    orc.close()
    assert np.max(np.abs(s - o)) < 1e-12 * np.max(np.abs(o))
