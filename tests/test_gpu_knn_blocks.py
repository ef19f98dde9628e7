"""GPU kNN lists of whole-number data at the edges of the kernel's blocks of 128 rows (32 a
wave) and of its tiles, in every dimension it is compiled for: one tile, two, a last
block of one row, row ranges that end inside a block."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 64, 96, 128])
@pytest.mark.parametrize("n", [31, 33, 127, 128, 129, 321, 641])
def test_block_edges(ctx, n, d):
    x = np.random.default_rng(n * d).integers(0, 256, size=(n, d)).astype(np.float64)
    d2 = ((x[:, None, :] - x[None, :, :]) ** 2).sum(2)
    np.fill_diagonal(d2, np.inf)
    k = min(64, n - 1)
    order = np.argsort(d2, axis=1, kind="stable")[:, :k]
    for row0, rows in ((0, n), (n - 1, 1), (0, min(n, 32)), (n // 5, n - n // 5)):
        print(f"[knn blocks] n={n} d={d} rows={row0}+{rows}", flush=True)
        ids, dists = ctx.knn(x.astype(np.float32), k, with_dists=True, rows=(row0, rows))
        np.testing.assert_array_equal(ids, order[row0:row0 + rows])
        np.testing.assert_array_equal(
            dists, np.take_along_axis(d2, order, 1)[row0:row0 + rows].astype(np.float32))
