"""The one-root form of the FP64 solve at the edges of its kernels: fewer points
than a workgroup, 256 workgroups of one and of four rows a thread, more partial
sums than a kernel adds itself; the smallest and largest subspaces; an exhausted
iteration count."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _well(g, depth=2.0, width=2.5):
    x, y, z = g.x
    r2 = x[None, None, :] ** 2 + y[None, :, None] ** 2 + z[:, None, None] ** 2
    return (-depth * np.exp(-r2 / (2 * width ** 2))).reshape(-1)


@pytest.mark.parametrize("n,maxsub", [((5, 4, 3), 2), ((6, 6, 6), 64), ((40, 41, 40), 20),
                                      ((41, 40, 40), 5), ((67, 64, 62), 12)])
def test_one_root(pisces, oracle_mod, n, maxsub):
    print("one root", n, maxsub, flush=True)
    L = tuple(0.55 * (v + 1) for v in n)
    g = oracle_mod.Grid(n, L)
    V = _well(g)
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(V)
        r = ctx.solve(1, pisces.start_vectors(ctx, 1), maxsub=maxsub, maxmacro=4000, ptol=8)
        H = ctx.apply_h(r["vecs"])
    assert r["nconv"] == 1 and r["resid"][0] < 1e-8
    u = r["vecs"][0]
    assert abs(u @ u - 1) < 1e-13
    assert np.linalg.norm(H[0] - r["evals"][0] * u) < 1.01e-8 + 1e-12
    if g.ngp < 300:  # the whole spectrum
        dense = np.stack([g.apply_h(V, e) for e in np.eye(g.ngp)])
        assert abs(r["evals"][0] - np.linalg.eigvalsh(dense)[0]) < 1e-12
    else:
        ro = g.solve(V, 1, 20, 4000, 8, 1, u[None])
        assert abs(r["evals"][0] - ro["evals"][0]) < 1e-10


def test_one_root_not_converged(pisces, oracle_mod):
    n, L = (16, 16, 16), (20.0,) * 3
    g = oracle_mod.Grid(n, L)
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(_well(g))
        r = ctx.solve(1, pisces.start_vectors(ctx, 1), maxsub=4, maxmacro=3, ptol=12)
    assert r["nconv"] == 0 and r["n_macro"] == 3 and r["evals"][0] == 0.0
    assert abs(r["vecs"][0] @ r["vecs"][0] - 1) < 1e-13
