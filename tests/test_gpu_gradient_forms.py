"""Gradient sums at the edges of the kernels' forms: one water, 16 and 17 column
blocks (64- and 32-point tiles), 33 and 36 (three rounds of column blocks), grids
that end inside a tile and a chunk of points; against the same sums in numpy."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CORES = {0: ((9.98526, 192.608), (1.67075, 13.8937)), 1: ((1.64121, 1.7643),),
         2: ((1.64121, 1.7643),), 3: ()}


def _reff(R, r0):
    t = R / r0
    return (np.where(R < r0, r0 * (0.5 + t ** 3 * (1 - 0.5 * t)), R),
            np.where(R < r0, 3 * t ** 2 - 2 * t ** 3, 1.0))


@pytest.mark.parametrize("nw,n", [(1, (3, 3, 2)), (3, (17, 8, 9)), (28, (9, 8, 7)), (29, (9, 8, 7)),
                                  (57, (7, 5, 3)), (64, (8, 4, 4))])
def test_gradient_forms(pisces, oracle_mod, nw, n):
    import workload
    print("gradient forms", nw, n, flush=True)
    xyz, _ = workload.water_cluster(nw, max(3.0, 2.3 * nw ** (1 / 3)), 900 + nw)
    cl = oracle_mod.Cluster(xyz)
    s = np.asarray(cl.sites).reshape(-1, 3)
    alpha, ip, epc, _ = cl.pol3_lists()
    ip = np.asarray(ip)
    pp = pisces.default_potpara()
    L = (18.0, 19.0, 20.0)
    psi = np.random.default_rng(nw).normal(size=int(np.prod(n)))
    with pisces.Context(n, L) as ctx:
        ctx.build_cluster_potential(xyz, (3, 2, 0, 3, 0, 0))
        gel, tmu, mcm = ctx.gradient_terms(psi, 4 * nw, 3 * nw)
        xs, _ = ctx.grid()
    g = np.stack([a.reshape(-1) for a in np.meshgrid(xs[2], xs[1], xs[0], indexing="ij")][::-1], 1)
    w = psi ** 2
    # polarization matrix and mu
    r = s[ip]
    d = r[:, None] - r[None]
    R = np.linalg.norm(d, axis=2) + np.eye(len(r))
    x = 0.3 * R ** 3 / np.sqrt(np.outer(alpha, alpha))
    f3, f5 = 1 - np.exp(-x), 1 - (1 + x) * np.exp(-x)
    T = 3 * (f5 / R ** 5)[..., None, None] * d[..., :, None] * d[..., None, :] \
        - (f3 / R ** 3)[..., None, None] * np.eye(3)
    off = 1 - np.eye(len(r))
    A = -T * off[..., None, None] + (np.eye(len(r)) / np.asarray(alpha)[:, None])[..., None, None] * np.eye(3)
    A = A.transpose(0, 2, 1, 3).reshape(3 * len(r), -1)
    D = g[:, None] - r[None]
    RD = np.linalg.norm(D, axis=2)
    re, dre = _reff(RD, pp[1])
    E = D / re[..., None] ** 3
    mu = np.linalg.solve(A, (E + np.asarray(epc).reshape(-1, 3)).reshape(len(g), -1).T).T
    m3 = mu.reshape(len(g), -1, 3)
    ref = np.zeros((4 * nw, 3))
    h = -3 * dre / re ** 4 / RD * np.sum(D * m3, axis=2)
    np.add.at(ref, ip, np.sum(w[:, None, None] * (h[..., None] * D + m3 / re[..., None] ** 3), axis=0))
    q = np.zeros(4 * nw)
    np.add.at(q, np.asarray(cl.iq), np.asarray(cl.q))
    for k in range(4 * nw):
        D = g - s[k]
        RD = np.linalg.norm(D, axis=1)
        re, dre = _reff(RD, pp[3])
        f = -q[k] * dre / re ** 2
        for z, c in CORES[k % 4]:
            f = f + c / pp[2] * z * np.exp(-z * RD)
        ref[k] += np.sum((w * f / RD)[:, None] * D, axis=0)
    # Epc of the two dipole solves agrees to about 1e-12; sums over a few hundred points
    assert np.abs(tmu - w @ mu).max() <= 1e-10 * np.abs(w @ mu).max()
    M = (w[:, None] * mu).T @ mu
    assert np.abs(mcm - M).max() <= 1e-10 * np.abs(M).max()
    assert np.abs(gel.reshape(-1, 3) - ref).max() <= 1e-10 * np.abs(ref).max()
