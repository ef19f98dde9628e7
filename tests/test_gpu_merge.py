"""GPU parity of the batch merge where it can go wrong: equal distances (within
a batch, between batch and beam, at the beam's last slot), repeated points and
repeated graph entries, beams that are not full, distances at and past the empty
slot's 536870912, infinities; on the kernels with whole 32-dim groups and on
those with a remainder, for beams held in VGPRs and in LDS and for several
waves per query.  Ids, distances and statistics must equal the oracle's."""
import numpy as np
import pytest

import oracle as O
from conftest import assert_same

pytestmark = pytest.mark.gpu


def _space(kind, n, d, degree, cap, seed):
    r = np.random.default_rng(seed)
    if kind == "ties":  # few distinct distances
        x = r.integers(0, 3, size=(n, d))
    elif kind == "copies":  # every point four times
        x = np.repeat(r.normal(0, 30, size=(n // 4, d)), 4, axis=0)[r.permutation(n)]
    elif kind == "far":  # about half of the distances past the empty slot's
        x = r.normal(0, 3000, size=(n, d)) * np.sqrt(32.0 / d)
    elif kind == "inf":
        x = r.normal(0, 30, size=(n, d))
        x[r.integers(0, n, n // 3)] *= 1e19
    else:
        x = r.normal(0, 30, size=(n, d))
    x = x.astype(np.float32)
    g = r.integers(0, n, size=(n, degree)).astype(np.int32)
    g[:, 1] = g[:, 0]  # one neighbour listed twice
    g[r.random((n, degree)) < 0.05] = n  # short rows
    pids = np.full((n // (cap // 2), cap), n, np.int32)  # half-filled leaves
    order = r.permutation(n)[:pids.shape[0] * (cap // 2)].reshape(pids.shape[0], -1)
    pids[:, :cap // 2] = np.sort(order, axis=1)
    q = x[r.integers(0, n, 96)] + (0 if kind == "ties" else r.normal(0, 5, size=(96, d)))
    return x, g, pids, q.astype(np.float32), r.integers(0, pids.shape[0], 96).astype(np.int32)


@pytest.mark.parametrize("kind", ["plain", "ties", "copies", "far", "inf"])
@pytest.mark.parametrize("d,degree,beam,width", [
    (32, 32, 32, 1), (64, 32, 64, 1), (64, 64, 128, 1), (96, 16, 8, 1), (96, 32, 256, 1),
    (128, 32, 64, 1), (128, 32, 512, 1), (256, 32, 128, 1), (960, 32, 64, 1), (100, 32, 256, 1),
    (128, 32, 128, 4), (64, 32, 16, 2)])
def test_merge_parity(ctx, kind, d, degree, beam, width):
    from rt_entry_amd import make_params
    x, g, pids, q, hits = _space(kind, 2000, d, degree, 64, seed=d + beam)
    boxes = np.zeros((pids.shape[0], 6), np.float32)
    ctx.set_base(x)
    ctx.set_graph(g)
    ctx.set_leaves(boxes, pids)
    for mode in (0, 1):
        bw, bh = O.default_bloom(mode, 1 << (beam - 1).bit_length())
        k = min(10, beam)
        io, do, so = O.search(x, g, q, pids, hits,
                              O.make_params(k=k, beam=beam, width=width, max_iter=40, mode=mode,
                                            bloom_words=bw, bloom_hashes=bh), with_stats=True)
        for kw in (dict(), dict(queue=1), dict(wpq=2)):
            print(f"[merge] {kind} d={d} beam={beam} width={width} mode={mode} {kw}", flush=True)
            ig, dg, sg = ctx.search(q, hits, make_params(k=k, beam=beam, width=width, max_iter=40,
                                                         mode=mode, **kw), with_stats=True)
            assert_same(ig, io, "ids")
            assert_same(dg.view(np.int32), do.view(np.int32), "dists")
            assert_same(sg, so.astype(np.int32), "stats")
