"""The work that programs on this library have it do, as measurable cases.

A case is a dict of plain values; `kind` says which calls a pass makes:

  query    rte_query: projection, entry leaves (or random entries) and the plain search in one call
  batched  projection, kd-tree entry leaves, uniform batched search (the serving loop)
  learned  the same with the entry network in place of the kd-tree walk
  uneven   the same with a k and a beam per query
  rerank   search on the leading PCA columns, whole beam, rerank on the original vectors
  predict  the entry network alone
  train    steps of the entry network's training, then its weights to the host
  knn      exact kNN lists and the search graph made of them
  setup    PCA fit, base rotation and kd-tree of a new base

Data are mixtures around centres, as in rt_entry_amd/data.py's workloads: "int" whole numbers 0..255, "float"
unrounded, "unit" normalised, "lowrank" a 64-dimensional signal in `d` dimensions plus noise.  Everything is made
from the seed on the GPU.  The index that a program holds before its queries come (base, graph, leaves, network) is
made in prepare(); its neighbour lists are exact within each centre's points, which is where nearly all true
neighbours are.
"""
from __future__ import annotations

import math

import numpy as np
import torch

from rt_entry_amd import Context, expand_aabbs, make_params

DEV = "cuda:0"
MODES = {"ref": 0, "tuned": 1}


# ---- cases ---------------------------------------------------------------
def listed():
    return [
        # one user's request: nothing but launches and the search's serial chain
        dict(name="query_one", kind="query", data="float", np=100_000, nq=1, d=128, degree=32, leaf=128, k=10,
             beam=64, iters=33, width=1, mode="ref", algo=1, wpq=0),
        # the small configuration's whole batch: too few queries to fill the card
        dict(name="query_1k", kind="query", data="float", np=100_000, nq=1_000, d=128, degree=32, leaf=128, k=10,
             beam=64, iters=33, width=1, mode="ref", algo=1, wpq=0),
        # random entries and four rows an iteration, as without an entry table; sizes that nothing divides
        dict(name="query_wide_odd", kind="query", data="float", np=150_001, nq=3_001, d=100, degree=30, leaf=150,
             k=100, beam=128, iters=20, width=4, mode="tuned", algo=0, wpq=0),
        # the headline batch from kd-tree leaves, at the setting that reaches recall 0.95
        dict(name="kdtree_10k", kind="batched", data="int", np=1_000_000, nq=10_000, d=128, degree=32, leaf=256,
             k=10, beam=256, iters=51, mode="ref"),
        # the headline batch from the learned entry, at its setting
        dict(name="learned_10k", kind="learned", data="int", np=1_000_000, nq=10_000, d=128, degree=32, leaf=256,
             k=10, beam=64, iters=33, mode="ref"),
        # requests of many sizes in one launch: k 1/10/100, beams 32..256
        dict(name="uneven_20k", kind="uneven", data="unit", np=1_000_000, nq=20_000, d=96, degree=32, leaf=256,
             k=100, beam=256, iters=100, mode="ref"),
        # high-dimensional vectors searched whole, four waves a query
        dict(name="query_960", kind="query", data="lowrank", np=200_000, nq=2_000, d=960, degree=48, leaf=100, k=10,
             beam=64, iters=27, width=1, mode="ref", algo=1, wpq=4),
        # high-dimensional vectors searched on 64 columns, the beam reranked on all 960
        dict(name="rerank_960", kind="rerank", data="lowrank", np=200_000, nq=10_000, d=960, ds=64, degree=48,
             leaf=100, k=10, beam=64, iters=28, mode="ref"),
        # entries of a large batch from a network with many leaves
        dict(name="predict_100k", kind="predict", data="int", np=400_000, nq=100_000, d=128, leaf=28),
        # the inner loop of training the entry network
        dict(name="train_1k", kind="train", batch=1_024, steps=8, d=128, h1=256, h2=256, leaves=4_096),
        # the graph of a new base of whole numbers (images' descriptors are bytes)
        dict(name="graph_160k", kind="knn", data="int", np=160_000, d=128, k=64, degree=32),
        # everything else that a new base needs before it can be searched
        dict(name="setup_1m", kind="setup", data="int", np=1_000_000, d=128, leaf=256),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["query", "query", "query", "batched", "learned", "uneven", "rerank", "predict", "train", "knn",
                       "setup"])
    c = dict(kind=kind)
    if kind == "query":
        width = rng.choice([1, 1, 2, 4])
        degree = rng.choice([16, 24, 32, 32, 48, 64]) if width == 1 else rng.choice([16, 24, 30, 32])
        beam = rng.choice([32, 64, 64, 100, 128, 256])
        c.update(data=rng.choice(["float", "int", "unit"]), np=_log(rng, 20_000, 300_000), nq=_log(rng, 1, 4_000),
                 d=rng.choice([32, 50, 64, 96, 100, 128, rng.randint(65, 128), 200]), degree=degree,
                 leaf=rng.randint(60, 256), k=rng.choice([1, 10, 10, min(100, beam)]), beam=beam,
                 iters=rng.randint(16, 60) // width + 4, width=width, mode=rng.choice(["ref", "tuned"]),
                 algo=rng.choice([1, 1, 1, 0]), wpq=rng.choice([0, 0, 2, 4]))
    elif kind in ("batched", "learned"):
        c.update(data=rng.choice(["int", "float", "unit"]), np=_log(rng, 200_000, 1_000_000), nq=_log(rng, 1_500, 10_000),
                 d=rng.choice([64, 96, 128]), degree=rng.choice([24, 32]), leaf=rng.randint(100, 256), k=10,
                 beam=rng.choice([64, 128, 256]), iters=rng.randint(24, 51), mode=rng.choice(["ref", "tuned"]))
    elif kind == "uneven":
        c.update(data=rng.choice(["unit", "int"]), np=_log(rng, 200_000, 1_000_000), nq=_log(rng, 2_000, 20_000),
                 d=rng.choice([64, 96]), degree=32, leaf=rng.randint(100, 256), k=100, beam=256,
                 iters=rng.randint(40, 100), mode=rng.choice(["ref", "tuned"]))
    elif kind == "rerank":
        c.update(data="lowrank", np=_log(rng, 50_000, 200_000), nq=_log(rng, 500, 10_000),
                 d=rng.choice([256, 512, 768, 960, 8 * rng.randint(32, 120)]), ds=rng.choice([32, 64, 96]), degree=48,
                 leaf=rng.randint(60, 200), k=10, beam=rng.choice([64, 128]), iters=rng.randint(20, 40), mode="ref")
    elif kind == "predict":
        c.update(data=rng.choice(["int", "unit"]), np=_log(rng, 60_000, 400_000), nq=_log(rng, 1_000, 100_000),
                 d=rng.choice([64, 96, 128]), leaf=rng.randint(28, 128))
    elif kind == "train":
        c.update(batch=_log(rng, 256, 2_048), steps=rng.randint(4, 8), d=rng.choice([64, 96, 128]),
                 h1=rng.choice([128, 256]), h2=rng.choice([128, 256]), leaves=_log(rng, 500, 4_096))
    elif kind == "knn":
        c.update(data=rng.choice(["int", "int", "float", "unit"]), np=_log(rng, 20_000, 150_000),
                 d=rng.choice([32, 64, 96, 128]), k=rng.choice([32, 48, 64]), degree=rng.choice([16, 24, 32]))
    else:
        c.update(data=rng.choice(["int", "float", "unit"]), np=_log(rng, 50_000, 1_000_000),
                 d=rng.choice([64, 96, 100, 128]), leaf=rng.randint(100, 400))
    return c


# ---- data ----------------------------------------------------------------
def _gen(seed, what):
    g = torch.Generator(device=DEV)
    g.manual_seed(1_000_003 * int(seed) + what)
    return g


def _n_centres(case):
    return max(4, round(case["np"] / (2_000 if case["data"] == "lowrank" else 1_000)))


def _points(case, seed, what, n):
    """n points of the case's mixture (stream `what`) and the centre each was drawn around."""
    nc, d = _n_centres(case), case["d"]
    g0, g = _gen(seed, 0), _gen(seed, what)
    z = torch.randperm(n, generator=g, device=DEV) % nc  # every centre has as many points as the others, or one more
    if case["data"] == "lowrank":
        basis = torch.linalg.qr(torch.randn((d, 64), generator=g0, device=DEV))[0]
        mu = torch.randn((nc, 64), generator=g0, device=DEV)
        lat = mu[z] + 0.25 * torch.randn((n, 64), generator=g, device=DEV)
        x = lat @ basis.T + 0.05 * torch.randn((n, d), generator=g, device=DEV)
    elif case["data"] == "unit":
        cen = torch.randn((nc, d), generator=g0, device=DEV)
        cen /= cen.norm(dim=1, keepdim=True)
        x = cen[z] + 0.15 * torch.randn((n, d), generator=g, device=DEV)
        x /= x.norm(dim=1, keepdim=True)
    else:
        hi, sigma = (255.0, 20.0) if case["data"] == "int" else (100.0, 8.0)
        cen = torch.rand((nc, d), generator=g0, device=DEV) * hi
        x = cen[z] + sigma * torch.randn((n, d), generator=g, device=DEV)
        if case["data"] == "int":
            x = x.round().clamp(0.0, 255.0)
    return x.contiguous(), z


def _knn_by_centre(x, z, nc, k):
    """The k nearest of every row among the rows of its own centre (int32 ids)."""
    n = x.shape[0]
    order = torch.argsort(z, stable=True)
    m = -(-n // nc)
    count = torch.bincount(z, minlength=nc)
    start = torch.cumsum(count, 0) - count
    slot = torch.arange(m, device=DEV)
    there = slot[None, :] < count[:, None]
    rows = order[(start[:, None] + slot[None, :]).clamp(max=n - 1)]  # nc x m
    knn = torch.empty((n, k), dtype=torch.int32, device=DEV)
    step = max(1, (1 << 27) // (m * m))
    for c in range(0, nc, step):
        r, ok = rows[c:c + step], there[c:c + step]
        p = x[r]
        nn = (p * p).sum(2)
        d2 = nn[:, :, None] + nn[:, None, :] - 2.0 * torch.bmm(p, p.transpose(1, 2).contiguous())
        d2.masked_fill_(~ok[:, None, :], float("inf"))
        d2.diagonal(dim1=1, dim2=2).fill_(float("inf"))
        near = torch.topk(d2, k, dim=2, largest=False, sorted=True).indices
        ids = torch.gather(r[:, None, :].expand(-1, m, -1), 2, near)
        knn[r[ok]] = ids[ok].int()
    return knn


def _leaves(ctx, pbase, cap):
    boxes, pids = ctx.build_kdtree(pbase, cap)
    aabbs = expand_aabbs(boxes.cpu().numpy(), 0.2)
    ctx.set_leaves(aabbs, pids.cpu().numpy())
    return pids


def _index(case, seed, graph=True):
    """A context that holds the case's base (rotated), graph and leaves, and what it was made of."""
    x, z = _points(case, seed, 1, case["np"])
    ctx = Context(0)
    d_out = case.get("ds", case["d"])
    R, mu, _ = ctx.pca_fit(x)
    ctx.set_pca(R, mu, d_out)
    pbase = ctx.pca_rotate(x, R, mu, d_out)
    pids = _leaves(ctx, pbase, case["leaf"])
    if graph:
        ctx.set_base(pbase)
        knn = _knn_by_centre(x, z, _n_centres(case), 48)
        g = ctx.graph_from_knn(knn, case["degree"], case["degree"])
        if case["data"] == "unit":  # overlapping centres: links between them
            ctx.graph_add_entry_links(g, 8)
        ctx.set_graph(g)
    return ctx, x, z, pbase, pids


def _runs_by_centre(z, size):
    n = z.shape[0] // size
    return torch.argsort(z, stable=True)[:n * size].view(n, size)


def _network_of(xb, z, pids, seed):
    """An entry network as training leaves one: random-feature hidden layers, and for every leaf the mean feature of
    the points of its commonest centre, so that a query's own centre decides and the confidence varies.  Plain
    torch.  Returns (weights, biases, input mean, input 1/std)."""
    g, d = _gen(seed, 5), xb.shape[1]
    mean, std = xb.mean(0), xb.std(0).clamp_min(1e-6)
    W1 = torch.randn((d, 256), generator=g, device=DEV) * math.sqrt(2.0 / d)
    W2 = torch.randn((256, 256), generator=g, device=DEV) * math.sqrt(2.0 / 256)
    n = xb.shape[0]
    leaf_z = torch.where(pids < n, z[pids.clamp(max=n - 1).long()], -1)
    protos = []
    for s in range(0, pids.shape[0], 512):
        p, lz = pids[s:s + 512].long(), leaf_z[s:s + 512]
        common = torch.where(lz >= 0, lz, lz[:, :1]).mode(dim=1).values
        w = (lz == common[:, None]).float()
        h = torch.relu(torch.relu(((xb[p.clamp(max=n - 1)] - mean) / std) @ W1) @ W2)
        protos.append((h * w[:, :, None]).sum(1) / w.sum(1, keepdim=True).clamp_min(1.0))
    P = torch.cat(protos)
    centred = P - P.mean(0)
    s = 150.0 / (centred * centred).sum(1).mean()
    W3 = (s * centred).T.contiguous()
    b3 = -0.5 * s * (P * P).sum(1) + s * 0.5 * (P.mean(0) ** 2).sum()
    zero = torch.zeros(256, device=DEV)
    host = lambda t: t.float().cpu().numpy()  # noqa: E731
    return [host(W1), host(W2), host(W3)], [host(zero), host(zero), host(b3)], host(mean), host(1.0 / std)


def _shapes(case, seed):
    """k and beam of every query of an uneven batch."""
    g = _gen(seed, 4)
    k = torch.tensor([1, 10, 100], device=DEV)[torch.randint(0, 3, (case["nq"],), generator=g, device=DEV)]
    b = torch.tensor([32, 64, 128, 256], device=DEV)[torch.randint(0, 4, (case["nq"],), generator=g, device=DEV)]
    return k.int(), torch.maximum(b, torch.where(k > 10, 128, 16)).int()


def _batch(case, seed):
    g = _gen(seed, 6)
    x = torch.randn((case["batch"] * case["steps"], case["d"]), generator=g, device=DEV)
    # labels follow the input through a fixed random map, as leaves follow regions
    m = torch.randn((case["d"], 12), generator=g, device=DEV)
    bits = ((x @ m) > 0).long()
    y = (bits * (2 ** torch.arange(12, device=DEV))).sum(1) % case["leaves"]
    return x, y.int()


def _start_weights(case, seed):
    g = _gen(seed, 7)
    dims = [case["d"], case["h1"], case["h2"], case["leaves"]]
    W = [((torch.rand((a, b), generator=g, device=DEV) * 2 - 1) * math.sqrt(6.0 / a)) for a, b in zip(dims, dims[1:])]
    return W, [torch.zeros(b, device=DEV) for b in dims[1:]]


# ---- one pass ------------------------------------------------------------
def prepare(case, seed):
    kind = case["kind"]
    s = dict(case=case, kind=kind)
    if kind == "train":
        ctx = Context(0)
        W, b = _start_weights(case, seed)
        ctx.mlp_create(case["d"], case["h1"], case["h2"], case["leaves"], seed=1)
        ctx.mlp_set([w.cpu().numpy() for w in W], [t.cpu().numpy() for t in b])
        x, y = _batch(case, seed)
        n = case["batch"]
        s.update(ctx=ctx, parts=[(x[i * n:(i + 1) * n], y[i * n:(i + 1) * n]) for i in range(case["steps"])])
        return s
    if kind in ("knn", "setup"):
        s.update(ctx=Context(0), x=_points(case, seed, 1, case["np"])[0])
        return s
    ctx, x, z, pbase, pids = _index(case, seed, graph=kind != "predict")
    nq, d_out = case["nq"], case.get("ds", case["d"])
    Q = _points(case, seed, 2, nq)[0]
    s.update(ctx=ctx, Q=Q)
    new = lambda *shape, dtype=torch.float32: torch.zeros(shape, dtype=dtype, device=DEV)  # noqa: E731
    if kind != "query":
        s.update(pq=new(nq, d_out), leaf=new(nq, dtype=torch.int32))
    if kind in ("learned", "predict"):
        # alone, the network's classes are runs of points by centre; before a search they are the kd-tree's leaves
        classes = pids if kind == "learned" else _runs_by_centre(z, case["leaf"])
        W, b, mean, inv = _network_of(pbase, z, classes, seed)
        ctx.mlp_create(case["d"], 256, 256, classes.shape[0])
        ctx.mlp_set(W, b)
        ctx.mlp_set_input_norm(mean, inv)
        s.update(conf=new(nq))
    if kind == "predict":
        ctx.project(Q, out=s["pq"])
        return s
    mode = MODES[case["mode"]]
    if kind == "query":
        s["p"] = make_params(k=case["k"], beam=case["beam"], width=case["width"], max_iter=case["iters"], mode=mode,
                             algo=case["algo"], wpq=case["wpq"])
    else:  # batched launches in leaf order; one query a workgroup where their lengths differ
        k = case["beam"] if kind == "rerank" else case["k"]
        s["p"] = make_params(k=k, beam=case["beam"], max_iter=case["iters"], mode=mode, order=1,
                             wg_waves=1 if kind == "uneven" else 4)
        s.update(ids=new(nq, k, dtype=torch.int32), dists=new(nq, k))
    if kind == "uneven":
        s["k_q"], s["b_q"] = _shapes(case, seed)
    if kind == "rerank":
        ctx.set_rerank_base(x)
        s.update(top=new(nq, case["k"], dtype=torch.int32), top_d=new(nq, case["k"]))
    return s


def run(s):
    ctx, kind = s["ctx"], s["kind"]
    if kind == "query":
        ids, dists, pq, leaf = ctx.query(s["Q"], s["p"])
        return dict(ids=ids, dists=dists, pq=pq, leaf=leaf)
    if kind == "train":
        for x, y in s["parts"]:
            ctx.mlp_train_step(x, y, lr=2e-3, want_loss=False)
        W, b = ctx.mlp_get()
        return dict(W=W, b=b)
    if kind == "knn":
        ids, dists = ctx.knn(s["x"], s["case"]["k"], with_dists=True)
        graph = ctx.graph_from_knn(ids, s["case"]["degree"])
        return dict(ids=ids, dists=dists, graph=graph)
    if kind == "setup":
        R, mu, eig = ctx.pca_fit(s["x"])
        pbase = ctx.pca_rotate(s["x"], R, mu)
        boxes, pids = ctx.build_kdtree(pbase, s["case"]["leaf"])
        return dict(R=R, mu=mu, eig=eig, pbase=pbase, boxes=boxes, pids=pids)
    pq, leaf = s["pq"], s["leaf"]
    if kind == "predict":
        ctx.predict_entry(pq, 0.3, out=leaf, conf=s["conf"])
        return dict(leaf=leaf, conf=s["conf"])
    ctx.project(s["Q"], out=pq)
    if kind == "learned":
        ctx.predict_entry(pq, 0.3, out=leaf, conf=s["conf"])
    else:
        ctx.select_entry(pq, out=leaf)
    out = dict(pq=pq, leaf=leaf, ids=s["ids"], dists=s["dists"])
    if kind == "uneven":
        ctx.search_batched(pq, leaf, s["k_q"], s["b_q"], s["p"], k_stride=s["case"]["k"], out=(s["ids"], s["dists"]),
                           beam_bound=s["case"]["beam"])
        return out
    ctx.search_batched(pq, leaf, None, None, s["p"], out=(s["ids"], s["dists"]))
    if kind == "learned":
        out["conf"] = s["conf"]
    if kind == "rerank":
        ctx.rerank(s["Q"], s["ids"], k=s["case"]["k"], out=(s["top"], s["top_d"]))
        out.update(top=s["top"], top_d=s["top_d"])
    return out


# ---- what a pass cannot do without ---------------------------------------
def work(case):
    """Every input row that a pass has to look at, once, and its outputs; the arithmetic of the distances, products
    and sums that its results are made of."""
    kind = case["kind"]
    if kind == "train":
        w = case["d"] * case["h1"] + case["h1"] * case["h2"] + case["h2"] * case["leaves"]
        rows = case["batch"] * case["steps"]
        # parameters, two moments: read and written by every step; weights to the host
        return dict(bytes=24.0 * w * case["steps"] + 4.0 * w + 4.0 * rows * (case["d"] + 1), flops=6.0 * w * rows)
    n, d = case["np"], case["d"]
    if kind == "knn":
        return dict(bytes=4.0 * n * d + 8.0 * n * case["k"] + 4.0 * n * case["degree"], flops=2.0 * n * n * d)
    if kind == "setup":
        return dict(bytes=4.0 * n * d * 3 + 4.0 * n, flops=1.0 * n * d * d + 2.0 * n * d * d)
    nq, ds = case["nq"], case.get("ds", d)
    net = d * 256 + 256 * 256 + 256 * (n // case["leaf"])
    if kind == "predict":
        return dict(bytes=4.0 * nq * (d + 2) + 2.0 * net, flops=2.0 * nq * net)
    k = case["beam"] if kind == "rerank" else case["k"]
    beam = 128 if kind == "uneven" else case["beam"]
    width = case.get("width", 1)
    rows = case["iters"] * width  # graph rows expanded by a query
    evals = beam + 0.75 * case["degree"] * rows  # about three of four neighbours are new to it
    b = 4.0 * nq * (d + ds) + 8.0 * nq * k
    b += 4.0 * ds * min(n, nq * evals) + 4.0 * case["degree"] * min(n, nq * rows)
    f = 2.0 * nq * d * ds + 3.0 * ds * nq * evals
    if kind == "learned":
        b, f = b + 2.0 * net, f + 2.0 * nq * net
    if kind == "rerank":
        b, f = b + 4.0 * d * min(n, nq * beam) + 8.0 * nq * case["k"], f + 3.0 * d * nq * beam
    return dict(bytes=b, flops=f)


# ---- 64-bit results ------------------------------------------------------
def _pca64(x):
    """Mean and eigenvectors by descending eigenvalue (largest component positive) in 64 bits."""
    x = x.double()
    mu = x.mean(0)
    c = torch.zeros((x.shape[1],) * 2, dtype=torch.float64, device=DEV)
    for part in (x - mu).split(1 << 17):
        c += part.T.contiguous() @ part
    w, v = np.linalg.eigh((c / (x.shape[0] - 1)).cpu().numpy())
    v, w = v[:, ::-1], w[::-1]
    sign = np.sign(v[np.abs(v).argmax(0), np.arange(v.shape[1])])
    return v * sign, mu.cpu().numpy(), w


def _conf64(pq, net):
    """Softmax maximum of the network: bf16 operands (as the network is defined), sums in 64 bits."""
    r = lambda t: t.float().bfloat16().double()  # noqa: E731
    W, b, mean, inv = ([torch.from_numpy(w).to(DEV) for w in net[0]], [torch.from_numpy(t).to(DEV).double() for t in net[1]],
                       torch.from_numpy(net[2]).to(DEV), torch.from_numpy(net[3]).to(DEV))
    conf = []
    for x in pq.float().split(8192):
        h = r((x - mean) * inv)
        for l in range(2):
            h = r(torch.relu(h @ r(W[l]) + b[l]))
        z = h @ r(W[2]) + b[2]
        conf.append(1.0 / torch.exp(z - z.max(1, keepdim=True).values).sum(1))
    return torch.cat(conf)


def _train64(case, seed):
    r = lambda t: t.float().bfloat16().double()  # noqa: E731
    W, b = _start_weights(case, seed)
    W, b = [w.double() for w in W], [t.double() for t in b]
    mom = [[torch.zeros_like(t), torch.zeros_like(t)] for t in W + b]
    x_all, y_all = _batch(case, seed)
    n = case["batch"]
    for i in range(case["steps"]):
        x, y = r(x_all[i * n:(i + 1) * n]), y_all[i * n:(i + 1) * n].long()
        Wr = [r(w) for w in W]
        h1 = torch.relu(x @ Wr[0] + b[0])
        h2 = torch.relu(r(h1) @ Wr[1] + b[1])
        dz = torch.softmax(r(h2) @ Wr[2] + b[2], 1)
        dz[torch.arange(n, device=DEV), y] -= 1.0
        dz /= n
        d2 = (r(dz) @ Wr[2].T.contiguous()) * (h2 > 0)
        d1 = (r(d2) @ Wr[1].T.contiguous()) * (h1 > 0)
        grads = [x.T @ r(d1), r(h1).T @ r(d2), r(h2).T @ r(dz), d1.sum(0), d2.sum(0), dz.sum(0)]
        for t, g, (m, v) in zip(W + b, grads, mom):
            m.mul_(0.9).add_(g, alpha=0.1)
            v.mul_(0.999).add_(g * g, alpha=0.001)
            t.sub_(2e-3 * (m / (1 - 0.9 ** (i + 1))) / (torch.sqrt(v / (1 - 0.999 ** (i + 1))) + 1e-8))
    return dict(W=W, b=b)


def exact(case, seed):
    """64-bit values of the projections, confidences, weights, PCA results and kNN distances.  Ids, leaves and
    boxes are whole numbers or copies of inputs; the distances of a search belong to the ids that its walk ends at
    and have no value apart from them."""
    kind = case["kind"]
    if kind == "train":
        return _train64(case, seed)
    x, z = _points(case, seed, 1, case["np"])
    if kind == "knn":
        x = x.double()
        nn, best = (x * x).sum(1), []
        for i in range(0, x.shape[0], 2048):
            q = x[i:i + 2048]
            d2 = nn[i:i + 2048, None] + nn[None, :] - 2.0 * (q @ x.T)
            at = torch.arange(q.shape[0], device=DEV)
            d2[at, i + at] = float("inf")
            best.append(torch.topk(d2, case["k"], dim=1, largest=False, sorted=True).values)
        return dict(ids=None, dists=torch.cat(best), graph=None)
    R, mu, w = _pca64(x)
    if kind == "setup":
        R32, mu32 = (torch.from_numpy(np.ascontiguousarray(t.astype(np.float32))).to(DEV).double() for t in (R, mu))
        pbase = torch.cat([(p.double() - mu32) @ R32 for p in x.split(1 << 17)])
        return dict(R=R.copy(), mu=mu, eig=w.copy(), pbase=pbase, boxes=None, pids=None)
    d_out = case.get("ds", case["d"])
    R32, mu32 = (torch.from_numpy(np.ascontiguousarray(t.astype(np.float32))).to(DEV).double() for t in (R[:, :d_out], mu))
    Q = _points(case, seed, 2, case["nq"])[0]
    if kind == "predict":
        pbase = torch.cat([((p.double() - mu32) @ R32).float() for p in x.split(1 << 17)])
        net = _network_of(pbase, z, _runs_by_centre(z, case["leaf"]), seed)
        return dict(leaf=None, conf=_conf64((Q.double() - mu32) @ R32, net))
    out = dict(ids=None, dists=None, leaf=None, pq=(Q.double() - mu32) @ R32)
    if kind == "learned":
        out["conf"] = None
    if kind == "rerank":
        out.update(top=None, top_d=None)
    return out
