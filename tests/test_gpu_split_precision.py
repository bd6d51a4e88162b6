"""Precision of the split-bfloat16 products.

Inner products: of the nine products of parts six are formed, so a result is
off by the roundings of FP32 sums of 64 values (24 of them, each of at most
2^-23 of |x_i| |y_j| if it truncates, about 2^-23 sqrt(24) / 2 = 3e-7 together)
and, for more than 64 values, by that over sqrt(K / 64).  Twice that is the
bound; without one of the six a host model gives at least 2.7e-6 (K <= 64),
1.9e-7 (2050) and 1.4e-7 (4096).

Rotations: at most 512 terms in an FP32 sum with one rounding for 16 terms, so
the relative error is at most about 2^-24 sqrt(512 / 16 / 2) / sqrt(3) = 1.4e-7
of the norm for any number of bands, and the result's own rounding (2.5e-8)
where the diagonal of C dominates, whose term is formed in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('N', [5, 64, 65, 129])
@pytest.mark.parametrize('K', [15, 16, 64, 2050, 4096])
def test_inner_products(cuda, N, K):
    import torch
    from gpawdft_amd.hs_operators import grid_inner_products

    class gd:
        dv = 1.0
    rng = np.random.default_rng(N + K)
    x, y = (rng.standard_normal((N, K)).astype('f') for _ in range(2))
    tol = 6e-7 / max(1.0, K / 64)**0.5
    for a, b in ((x, x), (y, x)):
        da = torch.from_numpy(a).cuda().view(N, 1, 1, K)
        db = da if b is a else torch.from_numpy(b).cuda().view(N, 1, 1, K)
        a, b = a.astype(float), b.astype(float)
        size = np.outer(np.linalg.norm(a, axis=1), np.linalg.norm(b, axis=1))
        err = grid_inner_products(gd, da, db).cpu().numpy() - a @ b.T
        assert (np.abs(err) / size).max() < tol


def _rotated(C, x):
    import torch
    from gpawdft_amd.hs_operators import rotate
    N, K = x.shape
    C = torch.from_numpy(C).cuda()
    x = torch.from_numpy(x).cuda()
    out = torch.empty_like(x)
    rotate(C, x.view(N, 1, 1, K), out.view(N, 1, 1, K))
    ref = C @ x.double()
    return float((out.double() - ref).norm() / ref.norm())


@pytest.mark.parametrize('N', [17, 128, 257, 512, 513, 1100, 2049])
def test_rotation(cuda, N):
    rng = np.random.default_rng(N)
    x = rng.standard_normal((N, 515)).astype('f')
    C = rng.standard_normal((N, N))
    assert _rotated(C, x) < 1.4e-7
    C *= 0.01 / np.sqrt(N)
    C = np.tril(C, -1) + np.diag(1.0 + np.diag(C))
    assert _rotated(C, x) < 3e-8


@pytest.mark.parametrize('N', [48, 300])
def test_rotation_of_small_values(cuda, N):
    """Values whose parts lie below the least bfloat16."""
    rng = np.random.default_rng(N)
    x = (1e-36 * rng.standard_normal((N, 300))).astype('f')
    C = rng.standard_normal((N, N))
    assert _rotated(C, x) < 1.4e-7
    x = (1e36 * x.astype(float)).astype('f')
    assert _rotated(1e-36 * C, 1e3 * x) < 1.4e-7
