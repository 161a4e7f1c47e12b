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
