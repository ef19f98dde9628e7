"""GPU kNN lists of whole-number data, on both sides of the rule that takes it
to the bf16 product: values up to 256 and past it, signed values, norms up to
2^22 and 2^23, repeated points (distance 0), sizes at the edges of the 64-point
tiles and 256-row workgroups, row ranges.  Every FP32 term is exact, so ids and
distances must equal the FP64 lists."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(kind, n, d, rng):
    if kind == "bytes":
        return rng.integers(0, 256, size=(n, d))
    if kind == "copies":
        return np.repeat(rng.integers(0, 256, size=(-(-n // 5), d)), 5, axis=0)[rng.permutation(n)]
    if kind == "top":  # the largest norms: 128 * 255^2 is just below 2^23
        return rng.integers(250, 256, size=(n, d))
    if kind == "signed":  # below 2^22
        return rng.integers(-100, 101, size=(n, d))
    if kind == "signed_large":  # norms of both sides of 2^22
        return rng.integers(-256, 257, size=(n, d))
    return rng.integers(0, 2, size=(n, d)) * 257  # no bf16 value


def _lists(X, k):
    """Every row's whole order by (distance, id) in FP64 (data.knn_exact looks at
    k + 9 candidates only, which equal distances may fill by any of their ids)."""
    x = X.astype(np.float64)
    nn = (x * x).sum(1)
    d2 = nn[:, None] + nn[None, :] - 2.0 * x @ x.T
    np.fill_diagonal(d2, np.inf)
    ids = np.argsort(d2, axis=1, kind="stable")[:, :k].astype(np.int32)
    return ids, np.take_along_axis(d2, ids, 1)


@pytest.mark.parametrize("n,d,k", [(2, 32, 1), (64, 64, 63), (65, 128, 64), (257, 96, 10), (1023, 128, 64),
                                   (4097, 32, 33)])
@pytest.mark.parametrize("kind", ["bytes", "copies", "top", "signed", "signed_large", "257"])
def test_lists_equal_fp64(ctx, kind, n, d, k):
    X = np.ascontiguousarray(_data(kind, n, d, np.random.default_rng(n + d))[:n], dtype=np.float32)
    print(f"[knn] {kind} n={n} d={d} k={k}", flush=True)
    ref_ids, ref_d = _lists(X, k)
    ids, dists = ctx.knn(X, k, with_dists=True)
    np.testing.assert_array_equal(ids, ref_ids)
    np.testing.assert_array_equal(dists.view(np.int32), ref_d.astype(np.float32).view(np.int32))
    r0, nr = n // 3, max(1, n // 2)
    ids, dists = ctx.knn(X, k, with_dists=True, rows=(r0, nr))
    np.testing.assert_array_equal(ids, ref_ids[r0:r0 + nr])
    np.testing.assert_array_equal(dists.view(np.int32), ref_d[r0:r0 + nr].astype(np.float32).view(np.int32))
