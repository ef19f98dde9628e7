"""PCA rotation to few columns, at the edges of the four or eight columns a wave, the 16
and 32 of the kernels, their 64 rows and their 64 columns of X: bit equality with the
ascending FP64 multiply-then-add."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d_out", [1, 3, 4, 5, 12, 13, 16, 17, 24, 25, 32, 33])
@pytest.mark.parametrize("n,d", [(1, 33), (64, 64), (65, 65), (191, 129), (1000, 200)])
def test_rotate_narrow(ctx, n, d, d_out):
    import torch
    r = np.random.default_rng(n + d + d_out)
    x = r.normal(0, 50, (n, d)).astype(np.float32)
    R = r.normal(0, 1, (d, d)).astype(np.float32)
    mu = r.normal(0, 50, d).astype(np.float32)
    want = np.zeros((n, d_out))
    for j in range(d):
        want = want + (x[:, j].astype(np.float64) - np.float64(mu[j]))[:, None] \
            * R[j, :d_out].astype(np.float64)
    out = ctx.pca_rotate(torch.from_numpy(x).cuda(), R, mu, d_out)
    np.testing.assert_array_equal(out.cpu().numpy(), want.astype(np.float32))
