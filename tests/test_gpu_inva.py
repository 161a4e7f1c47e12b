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
    g = np.stack([a.reshape(-1) for a in np.meshgrid(xs[2], xs[1], xs[0], indexing="ij")][::-1], 1)
    d = g[:, None] - sites[ip][None]
    R = np.linalg.norm(d, axis=2)
    t = R / pp[1]
    re = np.where(R < pp[1], pp[1] * (0.5 + t ** 3 * (1 - 0.5 * t)), R)
    E = (d / re[..., None] ** 3 + np.asarray(epc).reshape(-1, 3)[None]).reshape(len(g), -1)
    ref = -0.5 * np.sum(E * np.linalg.solve(A, E.T).T, axis=1) - 0.25
    # a backward-stable inverse: the condition number times a few hundred ulps
    tol = 1e-13 * np.abs(w).max() / np.abs(w).min() + 1e-12
    assert np.abs(V - V0 - ref).max() <= tol * np.abs(ref).max()
