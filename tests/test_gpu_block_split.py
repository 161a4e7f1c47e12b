"""The block engine's Gram products, cut into more workgroups while few
instances are live, and its small factor kernels, at the sizes where they
differ: one chunk, a ragged last chunk, at most and more than 64 chunks an entry
(partial sums added up by the consumer, or by a launch of their own), the narrow
and the matrix-core widths, each storage type.

V is a sum of one function per axis, so the exact levels of the discretised H
are sums of 1-D eigenvalues, found densely on the host.  A Ritz value lies within
||H u - theta u|| of a level of the symmetric H, and the solver's residuals are
FP64 and below 1e-8 at convergence; the levels are further apart than that, so
the bound is 1e-8, plus FP64 rounding of H X (1e-13 of its largest eigenvalue,
~50 Eh).  The returned vectors' residuals are checked against 1.01e-8."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x2"])
@pytest.mark.parametrize("n,nroots,block", [
    ((9, 10, 11), 2, 2),       # 990 rows: one ragged chunk
    ((17, 13, 12), 3, 4),      # 2652: three chunks, narrow blocks
    ((40, 33, 31), 4, 5),      # 40920: 40 chunks, summed by the consumer
    ((47, 45, 32), 3, 3),      # 67680: 67 chunks, narrow, a reduction launch
    ((48, 48, 47), 5, 12),     # 108288: 106 chunks, wide
])
def test_block_solve_separable(pisces, oracle_mod, n, nroots, block, precision):
    print("block split", n, nroots, block, precision, flush=True)
    L = (14.0, 15.5, 17.25)
    g = oracle_mod.Grid(n, L)
    T = g.T
    w = [0.02 * (d + 1) * np.linspace(-1.0, 1.0, n[d]) ** 2 for d in range(3)]
    ax = [np.linalg.eigvalsh(T[d] + np.diag(w[d])) for d in range(3)]
    levels = np.sort((ax[2][:, None, None] + ax[1][:, None] + ax[0]).ravel())[:nroots]
    V = (w[2][:, None, None] + w[1][:, None] + w[0]).ravel()
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(V)
        start = pisces.start_vectors(ctx, nroots, seed=4)
        r = ctx.solve_block(nroots, start, block=block, maxsub=5 * block, max_iter=2000, ptol=8,
                            precision=pisces.PRECISIONS[precision])
        HU = ctx.apply_h(r["vecs"])
    assert r["nconv"] == nroots, r
    np.testing.assert_allclose(r["evals"], levels, rtol=0, atol=1e-8 + 5e-12)
    res = np.linalg.norm(HU - r["evals"][:, None] * r["vecs"], axis=1)
    assert np.all(res < 1.01e-8), res
    np.testing.assert_allclose(r["vecs"] @ r["vecs"].T, np.eye(nroots), rtol=0, atol=1e-6)
