"""Covariance blocks and rotation strips at the edges of their tiles: columns
around 16, 64 and 128, rows around 32 and 64, one row range and several."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,d", [(2, 1), (31, 15), (33, 17), (1025, 127), (2100, 144),
                                 (1500, 129), (700, 260)])
def test_covariance_blocks(n, d):
    """R diag(eig) R^T is the covariance.  R is rounded to FP32 from an
    orthonormal matrix, so the product is off by at most 2 * 2^-24 * ||R||_F *
    max(eig) = 2^-23 sqrt(d) max(eig) in norm (FP64 errors are far below; the
    factor 2 left is for the second-order term)."""
    import rt_entry_amd as rt
    X = np.random.default_rng(1000 * n + d).normal(size=(n, d)).astype(np.float32)
    X *= np.linspace(0.5, 3.0, d).astype(np.float32)
    print(f"[pca edges] n={n} d={d}", flush=True)
    with rt.Context(0) as ctx:
        R, mu, eig = ctx.pca_fit(X)
    X64 = X.astype(np.float64)
    C = np.cov(X64, rowvar=False).reshape(d, d)
    R64 = R.astype(np.float64)
    assert np.abs(R64 @ np.diag(eig) @ R64.T - C).max() <= 2.0 ** -22 * np.sqrt(d) * eig.max()
    np.testing.assert_allclose(mu, X64.mean(0), rtol=1e-6, atol=1e-6)


@pytest.mark.parametrize("device", [False, True])
@pytest.mark.parametrize("n,d,d_out", [(1, 1, 1), (63, 63, 15), (65, 64, 16), (64, 65, 17),
                                       (130, 130, 128), (200, 300, 129), (129, 300, 300)])
def test_rotation_strips(n, d, d_out, device):
    """Bit equality with the ascending FP64 multiply-then-add."""
    import torch
    import rt_entry_amd as rt
    rng = np.random.default_rng(d_out)
    X = rng.normal(size=(n, d)).astype(np.float32) * 7
    R = rng.normal(size=(d, d)).astype(np.float32)
    mu = rng.normal(size=d).astype(np.float32)
    acc = np.zeros((n, d_out))
    for j in range(d):
        acc = acc + (X[:, j].astype(np.float64) - np.float64(mu[j]))[:, None] \
            * R[j, :d_out].astype(np.float64)[None, :]
    print(f"[rotate edges] n={n} d={d} d_out={d_out}", flush=True)
    with rt.Context(0) as ctx:
        out = ctx.pca_rotate(torch.from_numpy(X).cuda() if device else X, R, mu, d_out)
    out = out.cpu().numpy() if device else np.asarray(out)
    np.testing.assert_array_equal(out, acc.astype(np.float32))
