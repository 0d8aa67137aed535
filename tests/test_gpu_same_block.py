"""The FP64 same-spin terms of several vectors in one launch: the one-launch
form, the tiles with a last group of fewer vectors, odd rows and columns, sets
of one string, vectors too long to be grouped, and the row kernels, against
one product per vector (the same terms, in another order where the form
differs: at most some 1e4 per element, 1e-12 of the largest value)."""
import numpy as np
import pytest

from conftest import random_vector
from test_gpu_rdm_blocks import _strings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind,norb,ea,na,eb,nb,k", [
    ("blocks", 12, 3, 17, 3, 33, 5),
    ("blocks", 12, 3, 1, 3, 40, 3),
    ("blocks", 18, 5, 301, 5, 301, 3),
    ("blocks", 18, 5, 501, 4, 499, 7),
    ("blocks", 24, 5, 1217, 4, 129, 30),       # groups of 26 and 4
    ("blocks", 24, 5, 1501, 4, 1501, 2),       # two vectors do not make a group
    ("scattered", 40, 5, 600, 5, 600, 3),
])
def test_block_products(kind, norb, ea, na, eb, nb, k):
    import sbdx
    from sbdx import instances
    h, eri = instances.make_integrals(norb, 3, 11)
    I0, I1, I2 = instances.pack_integrals(norb, h, eri)
    a = _strings(kind, norb, ea, na, 21)
    b = a.copy() if (ea, na) == (eb, nb) else _strings(kind, norb, eb, nb, 22)
    print(f"[same block] {kind} norb {norb} {na} x {nb} k {k}", flush=True)
    op = sbdx.TPBOperator(norb, I0, I1, I2, a, b)
    V = np.stack([random_vector(na * nb, 5 + v) for v in range(k)])
    B, again = op.sigma_block(V), op.sigma_block(V)
    S = np.stack([op.sigma(v) for v in V])
    op.close()
    assert np.array_equal(B, again)
    assert np.max(np.abs(B - S)) <= 1e-12 * np.max(np.abs(S))
