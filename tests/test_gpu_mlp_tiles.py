"""GPU training step of the entry network at the edges of its tiles: batches
and widths of one, of whole and of cut 32- and 64-row tiles and 128-deep
stages, widths that break 16-byte loads, every register form of the softmax.

The network is made so that every FP32 sum is exact: small whole weights, equal
logits (hidden units in pairs of equal activation whose output weights cancel)
and power-of-two batches and class counts.  The gradients must then equal the
FP64 oracle's (same bf16 roundings) bit for bit, whatever the order of the
sums.  The Adam step is checked against its formula on those gradients."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _network(rng, d0, d1, d2, C):
    """Pairs (2i, 2i + 1) of both hidden layers have equal activations; the two
    units of an output pair read different units of the first layer's pairs."""
    W1, W2, W3 = np.zeros((d0, d1)), np.zeros((d1, d2)), np.zeros((d2, C))
    for i in range(d1 // 2):
        W1[:, 2 * i] = W1[:, 2 * i + 1] = rng.choice([-1, 0, 0, 0, 1], size=d0) * (rng.random(d0) < 8 / d0)
    for i in range(d2 // 2):
        for j in rng.choice(max(1, d1 // 2), size=3):
            if d1 >= 2:
                W2[2 * j, 2 * i] = W2[2 * j + 1, 2 * i + 1] = rng.choice([-1, 1])
        W3[2 * i] = rng.choice([-1, 0, 1], size=C)
        W3[2 * i + 1] = -W3[2 * i]
    f = lambda a: a.astype(np.float32)  # noqa: E731
    return [f(W1), f(W2), f(W3)], [np.ones(d1, np.float32), np.ones(d2, np.float32), np.zeros(C, np.float32)]


@pytest.mark.parametrize("n,shape", [
    (1, (1, 2, 2, 2)), (1, (32, 32, 32, 64)), (2, (31, 65, 130, 256)), (32, (33, 64, 96, 64)),
    (64, (128, 128, 127, 64)), (128, (40, 72, 136, 64)), (256, (100, 97, 34, 64)),
    (1024, (64, 128, 256, 64)), (2048, (128, 258, 256, 64)), (8, (128, 256, 256, 2048)),
    (4, (129, 256, 256, 4096)), (8, (40, 72, 24, 16384)), (4, (40, 72, 24, 32768))])
def test_gradients_and_step_at_tile_edges(ctx, n, shape):
    import torch
    from oracle import mlp as M
    rng = np.random.default_rng(n + sum(shape))
    W, b = _network(rng, *shape)
    ctx.mlp_create(*shape, seed=3)
    ctx.mlp_set(W, b)
    X = rng.choice([-1, 0, 1], size=(n, shape[0])).astype(np.float32)
    y = rng.integers(0, shape[3], size=n).astype(np.int32)
    Xd, yd = torch.from_numpy(X).cuda(), torch.from_numpy(y).cuda()
    print(f"[mlp] n={n} shape={shape}", flush=True)
    oW, ob, oloss = M.grads(W, b, X, y)
    gW, gb, loss = ctx.mlp_grad(Xd, yd)
    assert abs(loss - oloss) < 1e-5 * oloss
    for l in range(3):
        assert np.array_equal(gW[l], oW[l].astype(np.float32)), f"gW{l + 1}"
        assert np.array_equal(gb[l], ob[l].astype(np.float32)), f"gb{l + 1}"
    assert n == 1 or any(np.abs(g).max() > 0 for g in oW[:2])
    # first Adam step: m / (1 - b1) = g and v / (1 - b2) = g^2
    lr = 1e-2
    ctx.mlp_train_step(Xd, yd, lr=lr)
    W1, b1 = ctx.mlp_get()
    for p0, p1, g in list(zip(W, W1, gW)) + list(zip(b, b1, gb)):
        g = g.astype(np.float64)
        want = p0 - lr * g / (np.abs(g) + 1e-8)
        # FP32 rounding of the parameter (up to 1 in magnitude) and of the
        # ratio: 1 - 0.999f carries 2^-24 / 0.001 = 6e-5 into v / (1 - b2),
        # half of it into the root
        assert np.abs(p1 - want).max() < 2.0**-23 + lr * 4e-5
