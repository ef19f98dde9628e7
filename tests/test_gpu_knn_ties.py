"""GPU kNN lists where most distances are equal, at the sizes between which such bases take
the FP32 kernel: equal points, sparse zeros and ones, points repeated next to each
other (varied data all the same).  Lists are by (distance, id)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d", [32, 128])
@pytest.mark.parametrize("n", [767, 768, 1024, 32768, 32769])
def test_equal_points(ctx, n, d):
    import torch
    x = torch.full((n, d), 7.0, device="cuda")
    ids, dists = ctx.knn(x, 64, with_dists=True)
    ctx.synchronize()
    i = torch.arange(64, dtype=torch.int32, device="cuda")[None, :]
    row = torch.arange(n, dtype=torch.int32, device="cuda")[:, None]
    assert torch.equal(ids, torch.where(i < row, i, i + 1))
    assert not dists.any()


@pytest.mark.parametrize("kind", ["sparse", "sparse_tail", "repeat"])
@pytest.mark.parametrize("n", [767, 769, 1500])
def test_few_distances(ctx, n, kind):
    r = np.random.default_rng(n)
    x = (r.random((n, 32)) < 0.03).astype(np.float64)
    if kind == "repeat":
        x = np.repeat(r.integers(0, 256, size=(-(-n // 5), 32)), 5, axis=0)[:n].astype(np.float64)
    elif kind == "sparse_tail":  # one varied block of rows among them
        x[64:128] = r.integers(0, 256, size=(64, 32))
    d2 = (x * x).sum(1)[:, None] + (x * x).sum(1)[None, :] - 2.0 * x @ x.T
    np.fill_diagonal(d2, np.inf)
    order = np.argsort(d2, axis=1, kind="stable")[:, :33]
    ids, dists = ctx.knn(x.astype(np.float32), 33, with_dists=True)
    np.testing.assert_array_equal(ids, order)
    np.testing.assert_array_equal(dists, np.take_along_axis(d2, order, 1).astype(np.float32))
