"""FP32 inner products: FP32 sums of 64 values of k at most, which begin at
chunks that are multiples of 32 values, then FP64.  The result is FP64, so
where the sums begin is part of it: the groups' products one by one, each a
call of its own, and their FP64 sum give the result of the whole.

Tolerance: both add the same FP32 numbers in FP64, at most K / 32 of them
after the first, in two orders: 2 (K / 32) 2^-53 of the sum of their sizes, so
1e-12 of that covers 10^5 values."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# K: below one chunk, odd (rows not aligned), chunks of an odd multiple of 32
# values, 64 bands and fewer, one tile of 128 and several
@pytest.mark.parametrize('N,K', [(3, 40), (18, 3171), (37, 17766),
                                 (64, 4512), (70, 29700), (95, 14141),
                                 (130, 5003)])
@pytest.mark.parametrize('same', [True, False])
def test_groups_of_64(cuda, N, K, same):
    import torch
    from gpawdft_amd._lib import GPD_F32, check, lib
    from gpawdft_amd.device import stream_ptr

    def products(a, b):
        out = torch.empty((N, N), dtype=torch.float64, device='cuda')
        check(lib().gpd_inner_products(
            GPD_F32, N, a.shape[1], a.data_ptr(), b.data_ptr(), 1.0, 0, None,
            0, out.data_ptr(), stream_ptr()))
        return out

    rng = np.random.default_rng(N + K)
    x = torch.from_numpy(rng.standard_normal((N, K)).astype('f')).cuda()
    y = x if same else torch.from_numpy(
        rng.standard_normal((N, K)).astype('f')).cuda()
    tiles = (N + 127) // 128
    ntile = tiles * (tiles + 1) // 2 if same else tiles**2
    nsplit = max(1, min(512 // ntile, K // 1024))
    chunk = -(-(-(-K // nsplit)) // 32) * 32
    ref = torch.zeros((N, N), dtype=torch.float64, device='cuda')
    size = torch.zeros_like(ref)
    for c in range(0, K, chunk):
        for k in range(c, min(K, c + chunk), 64):
            end = min(K, c + chunk, k + 64)
            a = x[:, k:end].contiguous()
            p = products(a, a if same else y[:, k:end].contiguous())
            ref += p
            size += p.abs()
    err = (products(x, y) - ref).abs()
    assert (err <= 1e-12 * size).all()
