"""The block solver with one vector of its start block not finite: that vector
alone is dropped, as a linearly dependent one is, and the others, which come
after it in the Gram-Schmidt order, find the roots.  Every root returned lies
within its residual of an eigenvalue (Weinstein's bound), so 1e-8 of the
dense ones."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("solver", ["thick", "block"])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
@pytest.mark.parametrize("whole", [True, False])
def test_a_vector_that_is_not_finite_is_dropped(solver, bad, whole, oracle_mod):
    import sbdx
    from sbdx import instances
    inst = instances.make_instance(norb=9, nelec_half=3, nstr=23, nchol=12, seed=7)
    op = sbdx.TPBOperator.from_instance(inst)
    op.configure(solver)
    orc = oracle_mod.Oracle.from_instance(inst)
    n = op.ndet
    H = np.stack([orc.sigma(e) for e in np.eye(n)], axis=1)
    orc.close()
    ref = np.linalg.eigvalsh(0.5 * (H + H.T))
    W0 = np.zeros((2, n))
    W0[0, 5] = bad
    if whole:
        W0[0] = bad
    W0[1, 0] = 1.0
    print(f"[block nonfinite] {solver} {bad} whole {whole}", flush=True)
    E, W, _, ok = op.davidson_block(2, 5, W0=W0, max_it=300, eps=1e-9)
    op.close()
    assert ok and np.all(np.isfinite(W))
    assert np.max(np.abs(np.sort(E) - ref[:2])) < 1e-8
