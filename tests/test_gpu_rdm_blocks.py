"""The RDM's two-spin kernel over its edges: one to four tiles of 16 orbitals
(and orbital counts at a tile's end), sets made of blocks, of scattered
strings (everything outside the blocks) and of one string, string counts
around the staged row's halves, and rows read in place (lowered LDS budget),
against the oracle.

|w| = 1, so every element of the RDMs is a sum of products bounded by 1 in
total magnitude; with at most 1e6 rounded terms its error is below
1e6 x 2^-53 ~ 1e-10 in the worst case and near sqrt of that, 1e-13, in a
random one: 1e-12."""
import os

import numpy as np
import pytest

from conftest import random_vector

pytestmark = pytest.mark.gpu


def _strings(kind, norb, n, nstr, seed):
    from sbdx import instances, io
    if kind == "blocks":
        return instances.make_strings(norb, n, nstr, seed)
    rng = np.random.default_rng(seed)
    out = set()
    while len(out) < nstr:
        out.add(sum(1 << int(b) for b in rng.choice(norb, size=n, replace=False)))
    return io.sort_unique(np.array(sorted(out), dtype=np.uint64))


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb,lds", [
    ("blocks", 15, 4, 90, 4, 90, None),
    ("blocks", 16, 4, 120, 3, 131, None),
    ("blocks", 17, 5, 150, 4, 129, None),
    ("blocks", 32, 3, 100, 3, 100, None),
    ("blocks", 33, 3, 90, 2, 64, None),
    ("blocks", 49, 2, 60, 2, 97, None),
    ("blocks", 64, 2, 40, 3, 63, None),
    ("scattered", 14, 4, 70, 4, 111, None),
    ("scattered", 40, 3, 50, 3, 65, None),
    ("blocks", 12, 3, 1, 3, 1, None),
    ("blocks", 12, 3, 1, 4, 40, None),
    ("blocks", 18, 5, 20, 5, 513, None),      # one string past a thread's first value
    ("blocks", 36, 8, 4, 8, 4096, None),      # a whole half row, its zero in the second
    ("blocks", 36, 8, 3, 8, 4097, None),
    ("blocks", 17, 5, 150, 4, 129, 6000),     # rows read in place
    ("scattered", 50, 3, 50, 3, 65, 24000),
])
def test_rdm_blocks(kind, norb, ea, na, eb, nb, lds, oracle_mod):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 3)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 5)
    inst = dict(norb=norb, nelec=ea + eb, I0=I0, I1=I1, I2=I2, astr=a, bstr=b)
    print(f"[rdm blocks] {kind} norb {norb} {na} x {nb} lds {lds}", flush=True)
    old = os.environ.pop("SBDX_LDS_LIMIT", None)
    if lds:
        os.environ["SBDX_LDS_LIMIT"] = str(lds)
    try:
        op = sbdx.TPBOperator.from_instance(inst)
    finally:
        os.environ.pop("SBDX_LDS_LIMIT", None)
        if old is not None:
            os.environ["SBDX_LDS_LIMIT"] = old
    W = random_vector(op.ndet, 9)
    one, two = op.correlation(W)
    op.close()
    orc = oracle_mod.Oracle.from_instance(inst)
    r1, r2 = (np.asarray(r).reshape(-1) for r in orc.rdm(W))
    orc.close()
    assert np.max(np.abs(one - r1)) < 1e-12
    assert np.max(np.abs(two - r2)) < 1e-12
