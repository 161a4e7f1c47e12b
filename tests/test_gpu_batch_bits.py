"""A served request gives the same bits whatever else is in the batch.  Requests
are matched by their id, which seeds the start block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# sizes on both sides of the Gram kernels' chunk counts (one chunk; up to 64 and
# more of 1024 rows), and as many 64^3 as change the launches' shapes
SIZES = [((32, 32, 32), 30.0, 6, 3.5, 4100, 2), ((48, 48, 48), 36.0, 12, 4.5, 4101, 4),
         ((17, 15, 13), 24.0, 4, 3.2, 4105, 1), ((9, 8, 10), 20.0, 3, 3.2, 4106, 1),
         ((41, 39, 41), 34.0, 8, 4.0, 4102, 3)] + \
        [((64, 64, 64), 40.0, 24, 6.0, 4200 + i, 1) for i in range(4)]


def _submit(sv, i):
    import workload
    n, L, nw, rad, seed, nr = SIZES[i]
    return sv.submit(n, (L,) * 3, workload.water_cluster(nw, rad, seed)[0], nr, want_vectors=True)


@pytest.mark.parametrize("precision", ["fp64", "fp32", "bf16x2"])
def test_same_bits_alone_and_in_the_mix(pisces, precision):
    prec = pisces.PRECISIONS[precision]
    sv = pisces.Server(hbm_cap_bytes=64 << 30, max_slots=32, precision=prec)
    ids = [_submit(sv, i) for i in range(len(SIZES))]
    mix = {r["id"]: r for r in sv.run_until_done()}
    vecs = {i: sv.vectors(i) for i in ids}
    sv.close()
    assert ids == list(range(len(SIZES)))
    sv = pisces.Server(hbm_cap_bytes=64 << 30, max_slots=1, precision=prec)
    for i in ids:  # one at a time, under the same ids
        print(precision, SIZES[i], flush=True)
        assert _submit(sv, i) == i
        (r,) = sv.run_until_done()
        assert r["n_iter"] == mix[i]["n_iter"]
        np.testing.assert_array_equal(r["evals"], mix[i]["evals"])
        np.testing.assert_array_equal(r["resid"], mix[i]["resid"])
        np.testing.assert_array_equal(sv.vectors(i), vecs[i])
    sv.close()


@pytest.mark.parametrize("large", [214, 250])
def test_small_clusters_beside_a_large_one(pisces, large):
    """Dipoles of a batch whose largest cluster takes the 1024-thread form (above
    640 sites): the others keep theirs, with pairs in registers, LDS and memory,
    and give the bits they give without it; each agrees with its own potential
    built and solved singly."""
    import workload
    n, L = (12, 11, 12), (44.0, 44.0, 44.0)
    nws = [3, 27, 107, 213]
    xyz = {nw: workload.water_cluster(nw, max(3.0, 2.3 * nw ** (1 / 3)), 900 + nw)[0] for nw in nws + [large]}

    def serve(sizes):
        sv = pisces.Server(hbm_cap_bytes=8 << 30, max_slots=8, precision=pisces.FP64, ptol=9)
        for nw in sizes:
            sv.submit(n, L, xyz[nw], 1)
        res = {r["id"]: r for r in sv.run_until_done()}
        sv.close()
        return [res[i] for i in range(len(sizes))]

    print("batch", nws, large, flush=True)
    without, with_large = serve(nws), serve(nws + [large])
    for nw, r in zip(nws + [large], with_large):
        assert r["status"] == 1
        with pisces.Context(n, L) as ctx:
            _, _, rc = ctx.build_cluster_potential(xyz[nw])
            assert rc == 0
            one = ctx.solve(1, pisces.start_vectors(ctx, 1), maxsub=20, maxmacro=200, ptol=9, corrflag=1)
        assert one["nconv"] == 1
        # residuals of 1e-9 put either eigenvalue within 1e-9 of the level
        assert abs(r["evals"][0] - one["evals"][0]) <= 2e-9
    for a, b in zip(without, with_large):
        assert a["n_iter"] == b["n_iter"]
        np.testing.assert_array_equal(a["evals"], b["evals"])
        np.testing.assert_array_equal(a["resid"], b["resid"])
