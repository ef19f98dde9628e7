"""GPU kNN lists of whole-number data over many cells, where most tiles are left
out by their distance ranges: clusters far apart, clusters too small to fill a
list, lone points, a line, many equal distances, repeated points, and row ranges.
Sampled rows against FP64 lists; every term is exact, so ids and distances must be
equal."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(kind, n, d, rng):
    cen = rng.integers(0, 256, size=(40, d))
    near = lambda c, s: np.clip(np.rint(c + s * rng.standard_normal((len(c), d))), 0, 255)  # noqa: E731
    if kind == "clusters":
        return near(cen[rng.integers(0, 40, n)], 4.0)
    if kind == "small":  # clusters of about 20, most without a pivot and with less than a list's points
        many = rng.integers(0, 256, size=(n // 20, d))
        return near(many[rng.integers(0, n // 20, n)], 3.0)
    if kind == "lone":  # 300 points away from everything, spread over the rows
        x = near(cen[rng.integers(0, 40, n)], 4.0)
        x[rng.choice(n, 300, replace=False)] = rng.integers(0, 256, size=(300, d))
        return x
    if kind == "line":
        return np.repeat(rng.integers(0, 256, size=(n, 1)), d, axis=1)
    if kind == "binary":  # few distinct distances
        return rng.integers(0, 2, size=(n, d))
    return cen[rng.integers(0, 40, n)]  # copies


@pytest.mark.parametrize("n,d,k,r0,nr", [(20011, 64, 64, 0, 20011), (12801, 128, 10, 7000, 3333),
                                         (30000, 32, 33, 29999, 1)])
@pytest.mark.parametrize("kind", ["clusters", "small", "lone", "line", "binary", "copies"])
def test_sampled_rows_equal_fp64(ctx, kind, n, d, k, r0, nr):
    rng = np.random.default_rng(n + k)
    X = np.ascontiguousarray(_data(kind, n, d, rng), dtype=np.float32)
    print(f"[knn cells] {kind} n={n} d={d} k={k} rows {r0}+{nr}", flush=True)
    ids, dists = ctx.knn(X, k, with_dists=True, rows=(r0, nr))
    x = X.astype(np.float64)
    nn = (x * x).sum(1)
    rows = np.unique(rng.integers(r0, r0 + nr, 150))
    d2 = nn[rows, None] + nn[None, :] - 2.0 * x[rows] @ x.T
    d2[np.arange(len(rows)), rows] = np.inf
    want = np.argsort(d2, axis=1, kind="stable")[:, :k]
    np.testing.assert_array_equal(ids[rows - r0], want)
    np.testing.assert_array_equal(dists[rows - r0], np.take_along_axis(d2, want, 1).astype(np.float32))
