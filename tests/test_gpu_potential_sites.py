"""The grid potential's merge of the cluster's lists by site and its one- and
two-point forms: several charges and dipoles on one site, lists in a mixed order,
sites that carry nothing, and grids on both sides of the size (524288 points)
from which a thread takes two points of a column, with an odd number of planes
(the last one has no partner).  Bound: the sums have the oracle's terms in another
order, each a few roundings off, so 1e-13 of the largest value, the bound that the
other tests of this pass use for reordered lists."""
import numpy as np
import pytest

from conftest import golden

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("flagset", ["default", "gaussdamp", "gto12", "adiabatic"])
@pytest.mark.parametrize("n", [(16, 15, 3), (17, 9, 10), (90, 80, 75)])
def test_shared_sites(pisces, oracle_mod, flagset, n):
    print("potential sites", flagset, n, flush=True)
    f = golden("potential_c1.npz")
    cl = oracle_mod.Cluster(f["xyz"])
    L = (31.0, 30.0, 32.5)
    g = oracle_mod.Grid(n, L)
    rng = np.random.RandomState(3)
    # every charge in two parts, one site with three more; the dipoles likewise,
    # those of the first water left out
    q, iq = np.asarray(cl.q), np.asarray(cl.iq)
    q, iq = np.concatenate([0.3 * q, 0.7 * q, [0.2, -0.1, 0.05]]), np.concatenate([iq, iq, [iq[2]] * 3])
    d, idd = np.asarray(cl.d).reshape(-1, 3)[3:], np.asarray(cl.id)[3:]
    d, idd = np.concatenate([0.25 * d, 0.75 * d]), np.concatenate([idd, idd])
    a, b = rng.permutation(len(iq)), rng.permutation(len(idd))
    cl.q, cl.iq = np.ascontiguousarray(q[a]), np.ascontiguousarray(iq[a], dtype=np.int32)
    cl.d, cl.id = np.ascontiguousarray(d[b]), np.ascontiguousarray(idd[b], dtype=np.int32)
    flags, pp = f["flags_" + flagset], f["potpara_" + flagset]
    Vo = cl.potential_grid(g, flags, pp)
    with pisces.Context(n, L) as ctx:
        ctx.build_potential(flags, pp, cl.sites, cl.q, cl.iq, cl.d, cl.id)
        V = ctx.get_potential()
    assert np.abs(V - Vo).max() <= 1e-13 * np.abs(Vo).max()
