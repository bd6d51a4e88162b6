"""Rotations of bands that hold infinities, NaN or very large values: an
element is what its terms give by themselves, and no other band's or column's
elements are touched."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sum(C, X):
    """The terms' sum, each part by itself (numpy's complex product and a
    matrix product may give NaN where a part is infinite)."""
    if X.dtype != np.complex128:
        return (C[:, :, None] * X[None]).sum(1)
    c, x = C[:, :, None], X[None]
    re = (c.real * x.real).sum(1) + (-c.imag * x.imag).sum(1)
    im = (c.real * x.imag).sum(1) + (c.imag * x.real).sum(1)
    return np.stack([re, im], -1).view(np.complex128)[..., 0]


def _parts(a):
    return a.view(a.real.dtype)


# bands: a slab of terms with and without a remainder, one and two tiles,
# more terms than one FP32 sum takes
@pytest.mark.parametrize('dtype', [np.float32, np.float64, np.complex128])
@pytest.mark.parametrize('N', [3, 16, 50, 64, 70, 129, 520])
def test_rotation(cuda, N, dtype):
    import torch
    from gpawdft_amd.hs_operators import rotate
    K = 150
    rng = np.random.default_rng(N)
    X, C = rng.standard_normal((N, K)), rng.standard_normal((N, N))
    if dtype == np.complex128:
        X = X + 1j * rng.standard_normal(X.shape)
        C = C + 1j * rng.standard_normal(C.shape)
    X = X.astype(dtype)
    C[0, N - 1] = 0.0
    X[N - 1, 1] = np.inf            # the last band
    X[0, 2] = -np.inf
    X[1, 3] = np.nan
    X[0, 4], X[1, 4] = np.inf, -np.inf
    big = np.finfo(dtype).max
    C[:, 1] *= 0.1
    X[1, 5] = big                   # rounds to an infinite bfloat16
    X[1, 6] = -big / 1e5
    x = torch.from_numpy(X).cuda().view(N, 1, 1, K)
    out = torch.empty_like(x)
    rotate(torch.from_numpy(C).cuda(), x, out)
    got = out.cpu().numpy().reshape(N, K)
    with np.errstate(all='ignore'):
        wide = X.astype(np.complex128 if dtype == np.complex128 else float)
        ref = _sum(C, wide).astype(dtype)
    got, ref = _parts(got), _parts(ref)
    assert np.array_equal(np.isnan(got), np.isnan(ref))
    inf = np.isinf(ref)
    assert np.array_equal(got[inf], ref[inf])
    ok = np.isfinite(ref)
    size = np.abs(np.where(np.isfinite(X), X, 0.0)).astype(np.longdouble)
    size = np.sqrt((size**2).sum(0))
    size = np.repeat(np.broadcast_to(size, (N, K)), got.shape[1] // K, axis=1)
    tol = 4e-7 if dtype == np.float32 else 1e-13
    err = np.abs(got[ok].astype(float) - ref[ok])
    assert (err <= tol * N**0.5 * np.maximum(size[ok], 1.0)).all()
