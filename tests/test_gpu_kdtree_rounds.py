"""GPU kd-tree build where its rounds do not go as halving does: skewed values that
split off a few points at a time (many more rounds than are queued at first), sizes
at the edges of the small nodes and of the workgroups' chunks, searches that end at
once or never, against the host build."""
import numpy as np
import pytest

from rt_entry_amd import RteError, build_kdtree

pytestmark = pytest.mark.gpu


def _points(kind, n, rng):
    if kind == "skewed":
        return np.exp(3.0 * rng.standard_normal((n, 3)))
    if kind == "thin":  # one wide axis, two with no width
        return np.stack([rng.permutation(n), np.full(n, 7.0), np.zeros(n)], 1)
    return rng.standard_normal((n, 3)) * [5, 1, 9]


@pytest.mark.parametrize("kind", ["plain", "skewed", "thin"])
@pytest.mark.parametrize("n,cap", [(1, 1), (2048, 64), (2049, 64), (4097, 2048), (30011, 200)])
def test_equals_host(ctx, kind, n, cap):
    pts = np.ascontiguousarray(_points(kind, n, np.random.default_rng(n)), dtype=np.float32)
    print(f"[kdtree rounds] {kind} n={n} cap={cap}", flush=True)
    hb, hp = build_kdtree(pts, cap)
    boxes, pids = ctx.build_kdtree(pts, cap)
    np.testing.assert_array_equal(boxes, hb)
    np.testing.assert_array_equal(pids, hp)


def test_refused(ctx):
    """Equal points cannot be split; whole numbers near 2^24 leave the search on two
    neighbouring floats (the host build would not return)."""
    rng = np.random.default_rng(3)
    same = np.ones((5000, 3), np.float32)
    with pytest.raises(RteError) as host:
        build_kdtree(same, 64)
    for pts in (same, (1.6e7 + rng.integers(0, 9, (5000, 3))).astype(np.float32)):
        with pytest.raises(RteError) as gpu:
            ctx.build_kdtree(pts, 64)
        assert gpu.value.code == host.value.code
