"""V-cycles of solvers of different sizes in two threads: the coarsest levels'
launch asks for LDS by an attribute of the process."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_two_sizes_in_two_threads(cuda):
    import torch
    from gpawdft_amd.grid_descriptor import GridDescriptor
    from gpawdft_amd.poisson import PoissonSolver
    sizes = [(64, 64, 64), (8, 8, 8)]
    start = threading.Barrier(len(sizes))

    def cycles(N, out, together):
        gd = GridDescriptor(N, np.array(N) * 0.4, True)
        rho = np.random.default_rng(N[0]).standard_normal(N)
        with torch.cuda.stream(torch.cuda.Stream()):
            ps = PoissonSolver(nn=1)
            ps.set_grid_descriptor(gd)
            ps.initialize()
            ps.phis[0] = torch.zeros(N, dtype=torch.float64, device='cuda')
            ps.rhos[0].copy_(torch.from_numpy(rho - rho.mean()))
            if together:
                start.wait(60)
            norms = [ps.iterate2(ps.step) for _ in range(60)]
            out[N] = ps.phis[0].cpu().numpy(), norms

    alone, both = {}, {}
    for N in sizes:
        cycles(N, alone, False)
    threads = [threading.Thread(target=cycles, args=(N, both, True))
               for N in sizes]
    for t in threads:
        t.start()
    for t in threads:
        t.join(100)
    for N in sizes:
        assert np.array_equal(alone[N][0], both[N][0])
        assert alone[N][1] == both[N][1]
