"""kNN lists while one context's calls change between whole numbers and other values, and
between bases whose scratch the context keeps and larger ones: the test of a call's
values must not see an earlier call's, and neither path may run on the other's data."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

KEPT = 20_000    # rows of 128: about 80 MB of scratch with the whole-number kernel
LARGE = 420_000  # more than the 256 MiB that a context keeps


def _data(kind, n, d, seed):
    import torch
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randint(0, 256, (n, d), generator=g, device="cuda").float()
    if kind == "one_half":  # whole numbers but for one value
        x[n // 2, d - 1] += 0.5
    elif kind == "large":  # norms too large by one row
        x[n - 1] = 256.0
        x[n - 1, 0] = -1.0
    elif kind == "float":
        x += torch.rand((n, d), generator=g, device="cuda")
    return x


def _check(x, row0, rows, k, ids, dists, exact):
    import torch
    xd = x.double()
    q = xd[row0:row0 + rows]
    nn = (xd * xd).sum(1)
    d2 = nn[row0:row0 + rows, None] + nn[None, :] - 2.0 * q @ xd.T
    d2[torch.arange(rows), row0 + torch.arange(rows)] = float("inf")
    if exact:
        order = torch.sort(d2, dim=1, stable=True).indices[:, :k]
        assert torch.equal(ids.long(), order)
        assert torch.equal(dists, torch.gather(d2, 1, order).float())
    else:  # FP32 sums: 128 products of up to 2^16 and two norms of up to 2^23
        want = torch.sort(d2, dim=1).values[:, :k]
        tol = 130 * 2.0 ** -24 * 2.0 ** 25
        assert (dists.double() - torch.gather(d2, 1, ids.long())).abs().max() <= tol
        assert (dists.double() - want).abs().max() <= tol


@pytest.mark.parametrize("order", [
    ["whole", "float", "whole", "one_half", "large", "whole"],
    ["float", "whole", "large", "float"]])
@pytest.mark.parametrize("sizes", [(KEPT,), (LARGE,), (KEPT, LARGE, 65)])
def test_changing_values(order, sizes):
    from rt_entry_amd import Context
    c = Context(0)
    for i, kind in enumerate(order):
        n = sizes[i % len(sizes)]
        print(f"[knn values] {kind} n={n}", flush=True)
        x = _data(kind, n, 128, seed=i)
        rows = min(n, 40)
        row0 = (n - rows) // 2
        ids, dists = c.knn(x, 16, with_dists=True, rows=(row0, rows))
        c.synchronize()
        _check(x, row0, rows, 16, ids, dists, exact=kind in ("whole", "large"))
    c.close()
