"""A V-cycle whose caller keeps no residual for the coarsest level, on which
none is formed: any array may stand in its place."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# a coarsest level above what the launch of the coarsest levels takes (38 ->
# 19 points an axis), with tiles and with second-order sweeps alone; sweeps
# that take one launch, several, and an odd number of them
@pytest.mark.parametrize('N,pbc', [((38, 38, 38), True),
                                   ((40, 46, 38), (0, 1, 0)),
                                   ((12, 20, 28), True)])
@pytest.mark.parametrize('relax', ['J', 'GS'])
@pytest.mark.parametrize('post', [0, 1, 4, 9])
def test_residual_of_the_coarsest_level(cuda, N, pbc, relax, post):
    import torch
    from gpawdft_amd.grid_descriptor import GridDescriptor
    from gpawdft_amd.poisson import PoissonSolver
    gd = GridDescriptor(N, np.array(N) * 0.4, pbc)
    rho = np.random.default_rng(sum(N)).standard_normal(tuple(gd.n_c))
    res = []
    for stand_in in (False, True):
        ps = PoissonSolver(nn=3, relax=relax)
        ps.set_grid_descriptor(gd)
        ps.initialize()
        assert ps.levels > 0
        ps.postsmooths[ps.levels] = post
        phi = torch.zeros(tuple(gd.n_c), dtype=torch.float64, device='cuda')
        ps.phis[0] = phi
        ps.rhos[0].copy_(torch.from_numpy(rho - rho.mean()))
        if stand_in:
            ps.residuals[ps.levels] = ps.rhos[0]
        res.append((phi, [ps.iterate2(ps.step) for _ in range(2)]))
        assert np.array_equal(ps.rhos[0].cpu().numpy(), rho - rho.mean())
    assert torch.equal(res[0][0], res[1][0])
    assert res[0][1] == res[1][1]
