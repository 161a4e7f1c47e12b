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
