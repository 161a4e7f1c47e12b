"""The induced-dipole kernel at the edges of its forms: pairs held in registers
(up to 24 waters), in LDS, streamed from memory, and the 1024-thread form above
640 sites; the lanes per site change at 10, 20, 40, 80 and 160 sites and more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nw", [1, 3, 4, 7, 13, 14, 24, 25, 27, 53, 54, 107, 214])
def test_induced_dipoles(pisces, oracle_mod, nw):
    import workload
    print("dipoles", nw, flush=True)
    xyz, _ = workload.water_cluster(nw, max(3.0, 2.3 * nw ** (1 / 3)), 500 + nw)
    cl = oracle_mod.Cluster(xyz)
    with pisces.Context((4, 4, 4), (40.0,) * 3) as ctx:
        _, mu, rc = ctx.build_cluster_potential(xyz)
    assert rc == 0
    # both iterations stop at a mean change of 1e-12 per component
    assert np.abs(mu - cl.mu).max() <= 1e-9 * max(np.abs(cl.mu).max(), 1e-3)


@pytest.mark.parametrize("gap", [1e-3, 1.3e-3, 1.7e-3, 2.3e-3, 3e-3, 5e-3, 8e-3, 2e-2, 1e-1])
def test_nearly_coincident_hydrogens(pisces, oracle_mod, gap):
    """Hydrogens of two waters `gap` bohr apart, where the dipole tensor's damping
    factor 1 - (1 + x) exp(-x) is below the rounding of its terms."""
    import workload
    a = np.asarray(workload.water_cluster(1, 3.0, 5)[0]).reshape(3, 3)
    b = 2 * a[1] - a + 0.52917720859 * gap * np.array([0.6, -0.64, 0.48])  # reflected through H1
    xyz = np.concatenate([a, b]).reshape(2, 9)
    print("overlap", gap, flush=True)
    cl = oracle_mod.Cluster(xyz)
    s = np.asarray(cl.sites).reshape(-1, 3)
    r = np.linalg.norm(s[1] - s[5])
    assert 0.5 * gap < r < 2 * gap
    with pisces.Context((4, 4, 4), (40.0,) * 3) as ctx:
        _, mu, rc = ctx.build_cluster_potential(xyz)
    assert rc == 0
    # the factor's rounding, a few 2^-53, over r^3, on top of the iteration's bound
    alpha = 0.28 / 0.52917720859 ** 3
    tol = 1e-9 + 3 * 4 * 2.0 ** -53 / r ** 3 * alpha
    assert np.abs(mu - cl.mu).max() <= tol * np.abs(cl.mu).max()
