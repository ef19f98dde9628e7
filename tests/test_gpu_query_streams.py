"""rte_query's outputs while several contexts' queries are in flight: results
that are dropped give their memory back at once, and no later query of any
context, on its own stream, the caller's or torch's default one, may be handed
memory that is still being written."""
import numpy as np
import pytest

from conftest import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", [1, 0])
@pytest.mark.parametrize("streams", ["own", "caller", "mixed"])
def test_dropped_results_do_not_disturb_others(int_workload, algo, streams):
    import torch
    from rt_entry_amd import Context, make_params
    w = int_workload
    p = make_params(k=10, beam=64, max_iter=30, algo=algo)
    ctxs, want, Qs, ss = [], [], [], []
    for i in range(3):
        c = Context(0)
        c.set_base(torch.from_numpy(w.base).cuda())
        c.set_graph(torch.from_numpy(w.graph_raw).cuda())
        c.set_leaves(w.aabbs, w.pids)
        c.set_pca(w.R, w.mu, w.R.shape[1])
        s = torch.cuda.Stream()
        if streams == "caller":
            c.set_stream(s.cuda_stream)
        Q = torch.from_numpy(np.ascontiguousarray(np.roll(w.raw_queries, i, axis=0))).cuda()
        torch.cuda.synchronize()
        r = c.query(Q, p)
        torch.cuda.synchronize()  # a caller's stream is ordered by the caller alone
        want.append([t.cpu().numpy() for t in r])
        ctxs.append(c)
        Qs.append(Q)
        ss.append(s)
    torch.cuda.synchronize()
    kept = []
    for i in range(120):
        j = i % 3
        cur = ss[j] if streams != "own" and (streams == "caller" or i % 2) else torch.cuda.current_stream()
        with torch.cuda.stream(cur):
            r = ctxs[j].query(Qs[j], p)
        if i % 7 == 0:
            kept.append((j, r))
        del r
    torch.cuda.synchronize()
    for j, r in kept:
        for name, got, ref in zip(("ids", "dists", "pq", "leaf"), r, want[j]):
            assert_same(got.cpu().numpy().view(np.int32), ref.view(np.int32), f"{streams} {name}")
    for c in ctxs:
        c.close()
