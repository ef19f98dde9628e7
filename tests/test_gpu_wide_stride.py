"""Search on a base whose rows lie far apart: a row's byte offset must not be formed from
24-bit factors once the row size needs more bits.  Strides on both sides of 2^22 floats
(2^24 bytes); ids, distances and statistics must equal the oracle's on the packed rows."""
import numpy as np
import pytest

import oracle as O
from conftest import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,stride", [
    (64, (1 << 22) - 32), (64, 1 << 22), (128, (1 << 22) + 32), (64, (1 << 24) + 64)])
def test_rows_far_apart(ctx, d, stride):
    import torch
    from rt_entry_amd import make_params
    r = np.random.default_rng(stride)
    n, cap = (40 if stride < 1 << 23 else 16), 8
    x = r.normal(0, 30, size=(n, d)).astype(np.float32)
    g = r.integers(0, n, size=(n, 16)).astype(np.int32)
    pids = r.permutation(n).astype(np.int32).reshape(-1, cap)
    q = (x[r.integers(0, n, 32)] + r.normal(0, 5, size=(32, d))).astype(np.float32)
    hits = r.integers(0, pids.shape[0], 32).astype(np.int32)
    base = torch.empty((n, stride), dtype=torch.float32, device="cuda:0")
    base[:, :d] = torch.from_numpy(x)
    ctx.set_base(base, d)
    ctx.set_graph(g)
    ctx.set_leaves(np.zeros((pids.shape[0], 6), np.float32), pids)
    bw, bh = O.default_bloom(0, 16)
    kw = dict(k=8, beam=16, max_iter=20)
    io, do, so = O.search(x, g, q, pids, hits, O.make_params(bloom_words=bw, bloom_hashes=bh, **kw),
                          with_stats=True)
    ig, dg, sg = ctx.search(torch.from_numpy(q).cuda(), torch.from_numpy(hits).cuda(),
                            make_params(**kw), with_stats=True)
    assert_same(ig.cpu().numpy(), io, "ids")
    assert_same(dg.cpu().numpy().view(np.int32), do.view(np.int32), "dists")
    assert_same(sg.cpu().numpy(), so.astype(np.int32), "stats")
