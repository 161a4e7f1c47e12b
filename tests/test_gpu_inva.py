"""The polarization matrix inverse behind PolType 3, by the GPU's blocked
elimination (16-point blocks, 64-point workgroup tiles: sizes at, below and above
their multiples): the potential against -E^T InvA E / 2 formed in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _matrix(r, alpha):
    n = len(r)
    A = np.zeros((3 * n, 3 * n))
    for i in range(n):
        A[3 * i:3 * i + 3, 3 * i:3 * i + 3] = np.eye(3) / alpha[i]
        for j in range(n):
            if i != j:
                d = r[i] - r[j]
                R = np.linalg.norm(d)
                x = 0.3 * R ** 3 / np.sqrt(alpha[i] * alpha[j])
                f3, f5 = 1 - np.exp(-x), 1 - (1 + x) * np.exp(-x)
                A[3 * i:3 * i + 3, 3 * j:3 * j + 3] = \
                    f3 / R ** 3 * np.eye(3) - 3 * f5 * np.outer(d, d) / R ** 5
    return A


def _grid_field(xs, sites, ip, epc, rdamp):
    """E + Epc at the polarizable sites, a row per grid point (DampType 2)."""
    g = np.stack([a.reshape(-1) for a in np.meshgrid(xs[2], xs[1], xs[0], indexing="ij")][::-1], 1)
    d = g[:, None] - sites[ip][None]
    R = np.linalg.norm(d, axis=2)
    t = R / rdamp
    re = np.where(R < rdamp, rdamp * (0.5 + t ** 3 * (1 - 0.5 * t)), R)
    return (d / re[..., None] ** 3 + np.asarray(epc).reshape(-1, 3)[None]).reshape(len(g), -1)


@pytest.mark.parametrize("nw,scale", [(1, 1.0), (5, 1.0), (7, 1.0), (8, 1.0), (16, 1.0), (64, 1.0),
                                      (6, 40.0)])
def test_inverse(pisces, oracle_mod, nw, scale):
    import workload
    print("inva", nw, scale, flush=True)
    xyz, _ = workload.water_cluster(nw, max(3.0, 2.3 * nw ** (1 / 3)), 700 + nw)
    cl = oracle_mod.Cluster(xyz)
    sites = np.asarray(cl.sites).reshape(-1, 3)
    alpha, ip, epc, e_pol = cl.pol3_lists()
    alpha = scale * np.asarray(alpha)
    A = _matrix(sites[ip], alpha)
    w = np.linalg.eigvalsh(A)
    assert w[0] > 0
    n, L = (5, 4, 4), (24.0, 25.0, 26.0)
    pp = pisces.default_potpara()
    with pisces.Context(n, L) as ctx:
        ctx.build_potential((3, 2, 0, 0, 0, 0), pp, sites, cl.q, cl.iq, np.zeros(3), np.zeros(0))
        V0 = ctx.get_potential()
        ctx.build_potential_scp((3, 2, 0, 3, 0, 0), pp, sites, cl.q, cl.iq, alpha, ip, epc, 0.25)
        V = ctx.get_potential()
        xs, _ = ctx.grid()
    E = _grid_field(xs, sites, ip, epc, pp[1])
    ref = -0.5 * np.sum(E * np.linalg.solve(A, E.T).T, axis=1) - 0.25
    # a backward-stable inverse: the condition number times a few hundred ulps
    tol = 1e-13 * np.abs(w).max() / np.abs(w).min() + 1e-12
    assert np.abs(V - V0 - ref).max() <= tol * np.abs(ref).max()


def _star(first, n=120):
    """One site of very large polarizability at the front or the back of a shell of
    small ones, each pair's damped coupling near its maximum: the only way to an
    indefinite matrix with positive polarizabilities is through many sites, so the
    first pivot that is not positive lies in a later 16-point block."""
    k = np.arange(n - 1) + 0.5
    th, ph = np.arccos(1 - 2 * k / (n - 1)), np.pi * (1 + 5 ** 0.5) * k
    shell = 4.6 * np.stack([np.cos(ph) * np.sin(th), np.sin(ph) * np.sin(th), np.cos(th)], 1)
    c = np.array([[0.1, -0.2, 0.15]])
    sites = np.concatenate([c, shell] if first else [shell, c])
    alpha = np.full(n, 0.01)
    alpha[0 if first else -1] = 1e4
    return sites, alpha


@pytest.mark.parametrize("first", [True, False])
def test_not_positive_definite(pisces, first):
    """A regular matrix that is not positive definite: the elimination on the GPU
    flags it and the host's pivoted one takes its place, for the potential and for
    the gradient sums after it."""
    print("not positive definite", first, flush=True)
    sites, alpha = _star(first)
    n = len(sites)
    ip = np.arange(n)
    A = _matrix(sites, alpha)
    sc = np.sqrt(np.repeat(alpha, 3))
    w = np.linalg.eigvalsh(A * np.outer(sc, sc))
    assert w[0] < -1e-2 and np.abs(w).min() > 1e-3
    L = A.copy()
    piv = []
    for k in range(3 * n):
        piv.append(L[k, k])
        L[k + 1:, k + 1:] -= np.outer(L[k + 1:, k], L[k, k + 1:]) / L[k, k]
    assert np.argmax(np.array(piv) <= 0) >= 16
    rng = np.random.default_rng(3)
    epc = rng.normal(size=3 * n) * 0.01
    q = np.where(np.arange(n) % 4 == 3, -0.4, 0.2)
    iq = np.arange(n)
    pp = pisces.default_potpara()
    grid, box = (5, 4, 6), (24.0, 25.0, 26.0)
    psi = rng.normal(size=int(np.prod(grid)))
    with pisces.Context(grid, box) as ctx:
        ctx.build_potential((3, 2, 0, 0, 0, 0), pp, sites, q, iq, np.zeros(3), np.zeros(0))
        V0 = ctx.get_potential()
        ctx.build_potential_scp((3, 2, 0, 3, 0, 0), pp, sites, q, iq, alpha, ip, epc, 0.25)
        V = ctx.get_potential()
        _, tmu, mcm = ctx.gradient_terms(psi, n, n)
        xs, _ = ctx.grid()
    E = _grid_field(xs, sites, ip, epc, pp[1])
    mu = np.linalg.solve(A, E.T).T
    ref = -0.5 * np.sum(E * mu, axis=1) - 0.25
    # pivoted elimination: the condition number (scaled by the polarizabilities,
    # and of E^T mu itself) times a few hundred ulps
    grow = 0.5 * np.sum(np.abs(E * mu), axis=1).max() / np.abs(ref).max()
    cond = np.abs(w).max() / np.abs(w).min()
    tol = 1e-13 * cond * max(grow, 1.0) + 1e-12
    assert np.abs(V - V0 - ref).max() <= tol * np.abs(ref).max()
    w2 = psi ** 2
    t, M = w2 @ mu, (w2[:, None] * mu).T @ mu
    assert np.abs(tmu - t).max() <= 10 * tol * np.abs(t).max()
    assert np.abs(mcm - M).max() <= 10 * tol * np.abs(M).max()


@pytest.mark.parametrize("at", [0, 11])
def test_zero_pivot(pisces, at):
    """An infinite polarizability makes three rows of zeros, in the first 16-point
    block or in a later one: both eliminations refuse it."""
    import workload
    print("zero pivot", at, flush=True)
    xyz, _ = workload.water_cluster(4, 4.0, 31)
    with pisces.Context((4, 4, 4), (24.0,) * 3) as ctx:
        sites, _, _ = ctx.build_cluster_potential(xyz)
        sites = np.asarray(sites).reshape(-1, 3)
        alpha = np.full(16, 1.5)
        alpha[at] = np.inf
        lib_args = ((3, 2, 0, 3, 0, 0), pisces.default_potpara(), sites, np.full(16, 0.1), np.arange(16), alpha,
                    np.arange(16), np.zeros(48), 0.0)
        with pytest.raises(pisces.PiscesError, match="singular polarization matrix"):
            ctx.build_potential_scp(*lib_args)
        # the context goes on
        V = ctx.build_cluster_potential(xyz) and ctx.get_potential()
    assert np.all(np.isfinite(V))
