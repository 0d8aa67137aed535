"""The RDM's Gram matrices (lower triangles by tiles) over their edges: rows
around a tile of 32 and 64 and a block of 128, the 64 x 64 tiles (from some
4000 rows on) and the halved 32 x 32 ones, columns fewer than a stage of 8,
odd, and not a multiple of it.  Against the path without them (a dot product
per pair of strings): sums of the same terms in another order, of a normalized
vector, so the elements agree to some 1e-16 sqrt(1e4) of at most 1."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings
from test_zz_no_alloc import _noalloc_rdm

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norb,ea,na,eb,nb", [
    (10, 3, 1, 3, 9),
    (10, 3, 33, 3, 64),
    (12, 3, 65, 3, 127),
    (14, 4, 129, 4, 7),
    (24, 5, 1543, 4, 321),
    (30, 6, 3969, 5, 13),
    (30, 6, 4001, 5, 203),
    (30, 6, 4096, 5, 4),
])
def test_rdm_gram(norb, ea, na, eb, nb):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a, b = _strings("blocks", norb, ea, na, 3), _strings("blocks", norb, eb, nb, 5)
    print(f"[rdm gram] norb {norb} {na} x {nb}", flush=True)
    op = sbdx.TPBOperator(norb, I0, I1, I2, a, b)
    W = random_vector(op.ndet, 9)
    W = W / np.linalg.norm(W)
    one, two = op.correlation(W)
    rc, msg, r1, r2 = _noalloc_rdm(op, W)
    op.close()
    assert rc == 0, msg
    assert np.max(np.abs(one - r1)) < 1e-12
    assert np.max(np.abs(two - r2)) < 1e-12
