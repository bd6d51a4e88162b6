"""H psi on any stream of the caller's: torch hands its streams out round
robin from a pool, so that one of them is the stream a Hamiltonian keeps for
the projections."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize('dtype', ['float64', 'float32'])
def test_every_stream_of_the_pool(cuda, dtype):
    import torch
    from gpawdft_amd.hamiltonian import Hamiltonian
    from gpawdft_amd.synthetic import System, smooth_bands_numpy
    system = System(24, 0.25, 2, seed=5)
    kin, pt = system.operators()
    ham = Hamiltonian(system.gd, [system.vt_G], system.dH_asp)
    psi = torch.from_numpy(smooth_bands_numpy(3, system.gd.n_c, 1)).cuda()
    psi = psi.to(getattr(torch, dtype))
    ref = torch.empty_like(psi)
    P_ref = ham.apply_fused(psi, ref, kin, pt)
    torch.cuda.synchronize()
    own = ham._side_stream(psi.device).cuda_stream
    met = False
    for _ in range(64):
        stream = torch.cuda.Stream()
        met = met or stream.cuda_stream == own
        with torch.cuda.stream(stream):
            out = torch.zeros_like(psi)
            P = ham.apply_fused(psi, out, kin, pt)
        torch.cuda.synchronize()
        assert torch.equal(out, ref) and torch.equal(P, P_ref)
    assert met
