"""The 3x3x3 convolutions bit for bit: an output of the data kernels is one
chain of FMAs over channels and, within them, taps; a weight gradient is the
sum of 256 chains of FMAs a chunk of the points.  A training step takes its
weights from these roundings, so the order is part of the result.  The chains
are formed here with the products exact and each sum rounded to 64 bits
before it is rounded to 24 (the two roundings differ from one in 2^-39 of the
sums)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _fma(a, b, c):
    r = np.multiply(a, b, dtype=np.longdouble)
    r += c
    return r.astype(np.float32)


def _dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a, np.float32)).cuda()


def _arrays(B, Cin, Cout, shape):
    rng = np.random.default_rng(B + 10 * Cin + 100 * Cout)
    x = rng.standard_normal((B, Cin) + shape).astype(np.float32)
    w = (rng.standard_normal((Cout, Cin, 27)) / 5).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    gy = rng.standard_normal((B, Cout) + shape).astype(np.float32)
    return x, w, b, gy


def _tap(t):
    return t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1


def _some_points(B, shape):
    """Flat points: all of a small grid, else the ends and some between."""
    n = B * int(np.prod(shape))
    if n <= 3000:
        return np.arange(n)
    rng = np.random.default_rng(n)
    return np.concatenate([np.arange(600), np.arange(n - 600, n),
                           rng.integers(0, n, 1800)])


def _neighbour(x, q, shape, t, sign):
    """Channels of x at the points q + sign d_t: (channels, points)."""
    b, z, y, c = np.unravel_index(q, x.shape[:1] + shape)
    d = [sign * k for k in _tap(t)]
    return x[b, :, (z + d[0]) % shape[0], (y + d[1]) % shape[1],
             (c + d[2]) % shape[2]].T


# one and two channels on either side, tiles of 8 x 8 x 2 points, and enough
# of them for 8 x 8 x 4 with 16 and 32 channels a workgroup
DATA = [(2, 1, 17, (3, 5, 7)), (1, 2, 16, (9, 10, 33)), (1, 3, 1, (8, 9, 17)),
        (1, 9, 2, (2, 16, 15)), (2, 5, 9, (5, 17, 8)), (1, 17, 33, (4, 7, 8)),
        (32, 5, 13, (13, 17, 30)), (16, 20, 18, (13, 31, 30))]


@pytest.mark.parametrize('B,Cin,Cout,shape', DATA)
def test_data_kernels_are_one_chain(cuda, B, Cin, Cout, shape):
    import torch
    from gpawdft_amd._lib import check, lib
    from gpawdft_amd.device import stream_ptr
    x, w, b, gy = _arrays(B, Cin, Cout, shape)
    dx, dw, db, dgy = _dev(x), _dev(w), _dev(b), _dev(gy)
    y, gx = torch.empty_like(dgy), torch.empty_like(dx)
    check(lib().gpd_conv3d_forward(B, Cin, Cout, *shape, dx.data_ptr(),
                                   dw.data_ptr(), db.data_ptr(), y.data_ptr(),
                                   0, stream_ptr()))
    check(lib().gpd_conv3d_backward_data(B, Cin, Cout, *shape, dgy.data_ptr(),
                                         dw.data_ptr(), gx.data_ptr(), 0,
                                         stream_ptr()))
    q = _some_points(B, shape)
    ref = np.zeros((Cout, len(q)), np.float32)
    taps = [_neighbour(x, q, shape, t, 1) for t in range(27)]
    for i in range(Cin):
        for t in range(27):
            ref = _fma(w[:, i, t, None], taps[t][None, i], ref)
    ref += b[:, None]
    got = y.cpu().numpy().swapaxes(0, 1).reshape(Cout, -1)[:, q]
    assert np.array_equal(got, ref)
    ref = np.zeros((Cin, len(q)), np.float32)
    taps = [_neighbour(gy, q, shape, t, -1) for t in range(27)]
    for o in range(Cout):
        for t in range(27):
            ref = _fma(w[o, :, t, None], taps[t][None, o], ref)
    got = gx.cpu().numpy().swapaxes(0, 1).reshape(Cin, -1)[:, q]
    assert np.array_equal(got, ref)


def _wgrad(x, gy):
    """gW and gb in the kernels' order."""
    B, Cin = x.shape[:2]
    Cout, shape = gy.shape[1], gy.shape[2:]
    npts, pairs = B * int(np.prod(shape)), Cin * Cout
    nchunk = max(1, min((2048 + pairs - 1) // pairs, npts // 4096))
    chunk = -(-npts // nchunk)
    q = np.arange(npts)
    xs = np.stack([_neighbour(x, q, shape, t, 1) for t in range(27)], 1)
    g = gy.swapaxes(0, 1).reshape(Cout, npts)
    gw = np.zeros((Cout, Cin, 27), np.float32)
    gb = np.zeros(Cout, np.float32)
    for q0 in range(0, npts, chunk):
        q1 = min(npts, q0 + chunk)
        acc = np.zeros((Cout, Cin, 27, 256), np.float32)
        accb = np.zeros((Cout, 256), np.float32)
        for p in range(q0, q1, 256):
            n = min(256, q1 - p)
            acc[..., :n] = _fma(g[:, None, None, p:p + n],
                                xs[None, :, :, p:p + n], acc[..., :n])
            accb[:, :n] += g[:, p:p + n]
        for s in (128, 64, 32, 16, 8, 4, 2, 1):
            acc = acc[..., :s] + acc[..., s:]
            accb = accb[:, :s] + accb[:, s:]
        gw += acc[..., 0]
        gb += accb[:, 0]
    return gw, gb


# grids below 256 points (one of one point), lines longer than 256 points,
# blocks of outputs and inputs with a remainder, several chunks that no
# multiple of 256 ends
WEIGHT = [(1, 1, 1, (1, 1, 1)), (3, 1, 2, (2, 3, 4)), (2, 3, 5, (6, 10, 12)),
          (1, 2, 3, (2, 2, 300)), (1, 16, 9, (15, 24, 25)),
          (3, 2, 16, (17, 16, 20)), (2, 16, 1, (12, 16, 25)),
          (1, 9, 2, (5, 4, 100)), (5, 17, 1, (3, 5, 7)),
          (1, 17, 33, (4, 4, 20)), (2, 33, 20, (3, 8, 17))]


@pytest.mark.parametrize('B,Cin,Cout,shape', WEIGHT)
def test_weight_gradient_keeps_its_order(cuda, B, Cin, Cout, shape):
    import torch
    from gpawdft_amd._lib import check, lib
    from gpawdft_amd.device import stream_ptr
    x, _, _, gy = _arrays(B, Cin, Cout, shape)
    dx, dgy = _dev(x), _dev(gy)
    gw = torch.empty((Cout, Cin, 27), dtype=torch.float32, device='cuda')
    gb = torch.empty(Cout, dtype=torch.float32, device='cuda')
    check(lib().gpd_conv3d_backward_weight(
        B, Cin, Cout, *shape, dx.data_ptr(), dgy.data_ptr(), gw.data_ptr(),
        gb.data_ptr(), stream_ptr()))
    rgw, rgb = _wgrad(x, gy)
    assert np.array_equal(gw.cpu().numpy(), rgw)
    assert np.array_equal(gb.cpu().numpy(), rgb)


@pytest.mark.parametrize('Cout', [1, 3])
def test_weight_gradient_of_arrays_above_4_gib(cuda, Cout):
    """Values at the end of a grid of 2^30 points, against the same values in
    a small grid: all other products are zero.  At most 36 products a sum."""
    import torch
    import unet as U
    from gpawdft_amd._lib import check, lib
    from gpawdft_amd.device import stream_ptr
    shape, small = (16, 8192, 8192), (6, 16, 16)
    rng = np.random.default_rng(Cout)
    x = np.zeros((1, 1) + small, np.float32)
    x[..., -2:, -8:, -8:] = rng.standard_normal((2, 8, 8))
    gy = np.zeros((1, Cout) + small, np.float32)
    gy[..., -1:, -6:, -6:] = rng.standard_normal((1, Cout, 1, 6, 6))

    def large(a):
        t = torch.zeros(a.shape[:2] + shape, device='cuda')
        t[..., -6:, -16:, -16:] = torch.from_numpy(a).cuda()
        return t

    dx, dgy = large(x), large(gy)
    gw = torch.empty((Cout, 1, 27), dtype=torch.float32, device='cuda')
    gb = torch.empty(Cout, dtype=torch.float32, device='cuda')
    check(lib().gpd_conv3d_backward_weight(
        1, 1, Cout, *shape, dx.data_ptr(), dgy.data_ptr(), gw.data_ptr(),
        gb.data_ptr(), stream_ptr()))
    rgw, rgb = U.conv3d_backward_weight(x.astype(float), gy.astype(float))
    tol = 36 * 2.0**-24 * np.abs(gy).sum(axis=(0, 2, 3, 4)).max() * 4
    assert np.abs(gw.cpu().numpy() - rgw).max() < tol
    assert np.abs(gb.cpu().numpy() - rgb).max() < tol
    assert np.abs(rgw).max() > 1000 * tol
