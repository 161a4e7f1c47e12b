"""Block solves at block sizes on both sides of the factor kernels' code sizes (4,
8 and 16 columns), against the dense spectrum."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "bf16x2"])
@pytest.mark.parametrize("block", [1, 3, 4, 5, 8, 9, 16])
def test_block_sizes(pisces, oracle_mod, block, precision):
    import workload
    print("block size", block, precision, flush=True)
    n, L = (11, 10, 9), (22.0, 21.0, 20.0)
    xyz, _ = workload.water_cluster(4, 3.4, 77)
    g = oracle_mod.Grid(n, L)
    V = oracle_mod.Cluster(xyz).potential_grid(g)
    ref = np.linalg.eigvalsh(g.apply_h(V, np.eye(g.ngp)))
    nroots = max(1, block - 1)
    start = np.random.default_rng(block).uniform(-1, 1, (nroots, g.ngp))
    with pisces.Context(n, L) as ctx:
        ctx.set_potential(V)
        r = ctx.solve_block(nroots, start, block=block, maxsub=min(64, 4 * block + 4), max_iter=2000, ptol=7,
                            precision=pisces.PRECISIONS[precision])
    assert r["nconv"] == nroots
    # residuals below 1e-7 bound every eigenvalue's error by that
    assert np.abs(r["evals"] - ref[:nroots]).max() <= 1e-7
