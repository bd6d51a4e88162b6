"""gpd_poisson_vcycle refuses grids that must be distinct before it looks at
anything they point to (no GPU: the pointers are not those of memory)."""
import ctypes

import pytest

from gpawdft_amd import _lib


def _call(phis, rhos, residuals):
    n = len(phis)
    levels = n - 1
    L = _lib.lib()
    vp = ctypes.c_void_p

    def pointers(values):
        return (vp * n)(*values)

    handles = pointers([0x10] * n)
    counts = (ctypes.c_int * n)(*[1] * n)
    weights = (ctypes.c_double * n)(*[0.7] * n)
    rc = L.gpd_poisson_vcycle(levels, handles, handles, handles,
                              pointers(phis), pointers(rhos),
                              pointers(residuals), counts, counts, weights, 2,
                              1.0, vp(0x20), vp(0x30), None)
    return rc, L.gpd_last_error()


A, B, C, D, E, F, G, H, I = range(0x1000, 0xa000, 0x1000)


@pytest.mark.parametrize('phis,rhos,residuals', [
    ([A, B], [C, D], [A, E]),          # phi and residual of a level
    ([A, B], [C, D], [C, E]),          # rho and residual
    ([A, B], [A, D], [C, E]),          # phi and rho
    ([A, B], [C, B], [D, E]),
    ([A, B, C], [D, E, F], [G, E, H]),  # of level 1
    ([A, B], [C, D], [D, E]),          # a residual and the next level's rho
    ([A, B], [C, D], [B, E]),          # and its phi
    ([A, A], [C, D], [B, E]),
    ([A], [B], [B])])
def test_distinct_grids(phis, rhos, residuals):
    rc, message = _call(phis, rhos, residuals)
    assert rc == _lib.GPD_ERR_ARG
    assert b'distinct' in message
