"""rte_query on the caller's stream, read on torch's default stream: outputs that are
dropped while a reader is pending there must not be overwritten by the next query,
which is ordered behind the first one but not behind the reader."""
import numpy as np
import pytest

from conftest import assert_same

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("algo", [1, 0])
def test_reader_on_default_stream(int_workload, algo):
    import torch
    from rt_entry_amd import Context, make_params
    w = int_workload
    p = make_params(k=10, beam=64, max_iter=30, algo=algo)
    c = Context(0)
    c.set_base(torch.from_numpy(w.base).cuda())
    c.set_graph(torch.from_numpy(w.graph_raw).cuda())
    c.set_leaves(w.aabbs, w.pids)
    c.set_pca(w.R, w.mu, w.R.shape[1])
    Q = torch.from_numpy(w.raw_queries).cuda()
    Q2 = torch.from_numpy(np.ascontiguousarray(w.raw_queries[::-1])).cuda()
    s = torch.cuda.Stream()
    default = torch.cuda.default_stream()
    slow = torch.zeros((4096, 4096), device="cuda")
    torch.mm(slow, slow)  # the library's own first-call work
    torch.cuda.synchronize()
    want = [t.cpu().numpy() for t in c.query(Q, p)]
    c.set_stream(s.cuda_stream)
    torch.cuda.synchronize()
    assert torch.cuda.current_stream() == default
    for _ in range(3):
        r = c.query(Q, p)
        default.wait_stream(s)  # the caller orders its reader behind the query
        for _ in range(20):  # the reader waits its turn
            torch.mm(slow, slow)
        got = [t.clone() for t in r]
        del r
        r2 = c.query(Q2, p)  # behind the first query on s, not behind the reader
        torch.cuda.synchronize()
        for name, a, b in zip(("ids", "dists", "pq", "leaf"), got, want):
            assert_same(a.cpu().numpy().view(np.int32), b.view(np.int32), name)
        for name, a, b in zip(("dists", "pq"), r2[1:3], want[1:3]):
            if algo == 1:
                assert_same(a.cpu().numpy()[::-1].view(np.int32), b.view(np.int32), name)
        del r2
    c.close()
