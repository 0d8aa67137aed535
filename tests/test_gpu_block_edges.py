"""The block solver's reductions at the edges of their tiles: vectors shorter
than one chunk of a Gram pass, lengths that leave a remainder, odd lengths,
one to three tiles of 16 columns and blocks at the template sizes.

The roots come from a basis whose residuals |r| are below eps = 1e-9 and
whose columns are FP64, so each lies within |r| of an eigenvalue (Weinstein's
bound) plus the rounding of the dense diagonalization, 1e-13 |H|."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# FP32 corrections ("block") cannot span a space of a few dimensions to 1e-9:
# the solver ends with an exhausted basis there, so 20 and 15 are FP64 only.
@pytest.mark.parametrize("na,nb,nroots,block,solver", [
    (4, 5, 1, 1, "thick"),  # 20 elements: one whole chunk and a remainder
    (3, 5, 1, 1, "thick"),  # 15: no whole chunk
] + [c + (s,) for s in ("thick", "block") for c in [
    (7, 9, 2, 3),      # 63, odd
    (16, 20, 4, 4),    # 320: no remainder
    (17, 19, 3, 5),    # 323, the second template size
    (23, 21, 5, 9),    # 483, the third
    (40, 33, 6, 16),   # the largest block
]])
def test_roots_at_tile_edges(na, nb, nroots, block, solver, oracle_mod):
    import sbdx
    from sbdx import instances
    base = instances.make_instance(norb=9, nelec_half=3, nstr=max(na, nb), nchol=12, seed=7)
    inst = dict(base, astr=base["astr"][:na], bstr=base["bstr"][:nb])
    op = sbdx.TPBOperator.from_instance(inst)
    op.configure(solver)
    orc = oracle_mod.Oracle.from_instance(inst)
    n = op.ndet
    H = np.stack([orc.sigma(e) for e in np.eye(n)], axis=1)
    orc.close()
    ref = np.linalg.eigvalsh(0.5 * (H + H.T))
    print(f"[block edges] {na} x {nb} roots {nroots} block {block} {solver}", flush=True)
    E, W, _, ok = op.davidson_block(nroots, block, max_it=300, eps=1e-9)
    op.close()
    assert ok
    tol = 1e-9 + 1e-13 * np.abs(H).max() * n
    for e, w in zip(E, W):
        assert np.min(np.abs(ref - e)) < tol
        assert abs(np.linalg.norm(w) - 1.0) < 1e-10
        assert np.linalg.norm(H @ w - e * w) < 1e-8
    assert np.max(np.abs(W @ W.T - np.eye(nroots))) < 1e-7
