"""FP64 and FP32 plane kernels (H*X, preconditioner) at the edges of their tile
forms: axes one below, at and one above multiples of 16 and 32, every tile
form (32, 64, 96, 128 points), planes whose two axes take different paddings,
and, up to 32 points, both sides of the line between one launch and two (1000
tiles: 8 vectors of 32^3 are beyond it)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(2, 3, 2), (15, 17, 16), (32, 32, 32), (5, 32, 31), (16, 2, 29), (33, 31, 32), (47, 49, 64), (65, 9, 48), (80, 81, 3),
          (96, 33, 97), (97, 16, 5), (128, 4, 113)]


@pytest.mark.parametrize("n", SHAPES)
@pytest.mark.parametrize("nvec", [1, 3, 8])
def test_apply_h_tile_edges(pisces, oracle_mod, n, nvec):
    print("hx edges", n, nvec, flush=True)
    L = tuple(0.6 * (v + 1) for v in n)
    g = oracle_mod.Grid(n, L)
    rng = np.random.default_rng(sum(n))
    V, X = rng.uniform(-1.0, 0.5, g.ngp), rng.uniform(-1.0, 1.0, (nvec, g.ngp))
    X = X.astype(np.float32).astype(np.float64)  # exact in both precisions
    Yo = g.apply_h(V, X)
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(V)
        # sums of at most 3 * 128 products: a few hundred ulps of the largest
        # entry at the very worst, in either precision
        for precision, eps in ((pisces.FP64, 2.0 ** -53), (pisces.FP32, 2.0 ** -24)):
            Y = ctx.apply_h_ex(X, precision)
            assert np.abs(Y - Yo).max() <= 100 * eps * np.abs(Yo).max(), precision


@pytest.mark.parametrize("n", SHAPES[1:])
def test_precond_fp64_tile_edges(pisces, oracle_mod, n):
    """(T - shift) t = scale r with the shift below the kinetic spectrum."""
    print("precond edges", n, flush=True)
    L = tuple(0.6 * (v + 1) for v in n)
    g = oracle_mod.Grid(n, L)
    r = np.random.default_rng(sum(n)).uniform(-1, 1, (2, g.ngp))
    with pisces.Context(n, L) as ctx:
        t = ctx.kinetic_precond(r, shift=-0.05, scale=-1.0, floor=1e-3)
    lhs = g.apply_h(np.zeros(g.ngp), t) + 0.05 * t
    np.testing.assert_allclose(lhs, -r, rtol=0, atol=1e-10)


@pytest.mark.parametrize("n", [(33, 40, 35), (64, 9, 50)])
@pytest.mark.parametrize("nvec", [5, 13, 30, 70])
def test_bf16x2_launch_shapes_agree(pisces, n, nvec):
    """The split-BF16 kernels choose waves and planes per workgroup by the
    number of planes; a plane's arithmetic is the same in every form, so each
    vector comes out bit for bit as it does alone."""
    print("bf16x2 shapes", n, nvec, flush=True)
    L = tuple(0.6 * (v + 1) for v in n)
    rng = np.random.default_rng(nvec)
    ngp = int(np.prod(n))
    X = rng.uniform(-1, 1, (nvec, ngp))
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(rng.uniform(-1.0, 0.5, ngp))
        Y = ctx.apply_h_ex(X, pisces.BF16X2)
        T = ctx.kinetic_precond(X, shift=-0.05, precision=pisces.BF16X2)
        for v in (0, nvec // 2, nvec - 1):
            np.testing.assert_array_equal(Y[v], ctx.apply_h_ex(X[v], pisces.BF16X2))
            np.testing.assert_array_equal(T[v], ctx.kinetic_precond(X[v], shift=-0.05,
                                                                    precision=pisces.BF16X2)[0])
