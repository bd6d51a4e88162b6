"""Benchmark: batched H psi on one MI355X.

Workload (the headline configuration): periodic 96^3 grid, h = 0.18 A,
256 bands of smoothed Gaussian noise, local potential of 32 Gaussian wells,
32 atoms with l = 0..2 Gaussian projectors (9 per atom) and random
symmetric dH.  One step = H psi for all 256 bands in FP64 (the reference's
precision; bit-exact with its C): projections P = <p|psi>, c = P dH, the
stencil with the local potential in its epilogue, then the projector add.
Metric: band * gridpoints / s (higher is better).

Prints one JSON line.  Also reported: the FP32 path with its measured
error against FP64, the multigrid preconditioner on the same grid with its
roofline, the stencil kernel's and the whole step's roofline (HBM bytes /
measured time), the 112^3 x 512 subspace step with MFMA utilisation, and
the CPU baseline on a bounded sample of bands (the reference's own C on
all host cores, next to the C oracle).
"""
import argparse
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
sys.path.insert(0, ROOT)

HBM_PEAK_GBS = 8000.0


def parse():
    p = argparse.ArgumentParser()
    p.add_argument('--gpus', type=int, default=1)
    p.add_argument('--steps', type=int, default=20)
    p.add_argument('--warmup', type=int, default=3)
    p.add_argument('--N', type=int, default=96)
    p.add_argument('--bands', type=int, default=256)
    p.add_argument('--atoms', type=int, default=32)
    p.add_argument('--no-cpu', action='store_true',
                   help='skip the CPU oracle baseline')
    p.add_argument('--cpu-seconds', type=float, default=8.0,
                   help='target length of the CPU baseline sample')
    p.add_argument('--no-ttt', action='store_true',
                   help='skip the time-to-1e-8 comparison of the multigrid '
                        'and learned preconditioners')
    p.add_argument('--ttt-max-iter', type=int, default=400)
    p.add_argument('--learned-c4', action='store_true',
                   help='also run the learned-preconditioner evaluation at '
                        'its stated size (96^3, 256 bands; minutes)')
    p.add_argument('--c4-seconds', type=float, default=150.0,
                   help='wall-clock bound of each C4 run')
    p.add_argument('--no-ragged', action='store_true',
                   help='skip the ragged-batch graph measurement')
    p.add_argument('--ragged-systems', type=int, default=48)
    p.add_argument('--no-kpoint', action='store_true',
                   help='skip the complex (k-point) H psi timing')
    p.add_argument('--no-poisson', action='store_true',
                   help='skip the multigrid Poisson solver timing')
    p.add_argument('--no-subspace', action='store_true',
                   help='skip the 112^3 x 512 subspace-step timing')
    p.add_argument('--copy-calibration', action='store_true',
                   help='also run a plain copy of one band block (for '
                        'counter calibration under rocprofv3 --pmc)')
    return p.parse_args()


def _events_ms(fn, reps):
    """Mean milliseconds of fn() over reps calls, timed with HIP events on
    torch's current stream (the stream every library launch takes)."""
    import torch
    e0 = torch.cuda.Event(enable_timing=True)
    e1 = torch.cuda.Event(enable_timing=True)
    fn()
    e0.record()
    for _ in range(reps):
        fn()
    e1.record()
    e1.synchronize()
    return e0.elapsed_time(e1) / reps


def hpsi_block(sysm, ham, nb, dt, args, dev):
    """H psi of nb bands in dtype dt: whole-step wall time and per-part
    event times; the multigrid preconditioner on the same bands."""
    import numpy as np
    import torch
    from gpawdft_amd._lib import check, lib
    from gpawdft_amd.device import DeviceView, stream_ptr
    from gpawdft_amd.preconditioner import Preconditioner
    from gpawdft_amd.synthetic import smooth_bands_device
    gd = sysm.gd
    G = int(np.prod(gd.n_c))
    kin, pt = sysm.operators()
    psi = smooth_bands_device(nb, gd.n_c, 7, dtype=dt)
    out = torch.empty_like(psi)
    P = torch.zeros((nb, pt.Mmax), dtype=dt, device=dev)
    c = torch.empty_like(P)

    def step():
        ham.apply_fused(psi, out, kin, pt, P_xM=P, c_xM=c)
    step()                                    # device tables, warm caches
    for _ in range(args.warmup):
        step()
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(args.steps):
        step()
    torch.cuda.synchronize()
    ms_step = (time.perf_counter() - t0) / args.steps * 1e3
    # the parts of one step, each timed alone with events
    vt = ham._vt(0, dt, dev)
    code = DeviceView(psi).code

    def projections():
        P.zero_()
        pt.integrate_xM(psi, P)
        ham.projector_coefs(pt, P, 0, c)

    def stencil():
        check(lib().gpd_hamiltonian_apply(
            kin.handle, None, code, nb, psi.data_ptr(), vt.data_ptr(),
            None, out.data_ptr(), stream_ptr()), 'hamiltonian_apply')

    def add():
        pt.add_xM(c, out)
    reps = max(3, args.steps // 2)
    ms_proj = _events_ms(projections, reps)
    ms_stencil = _events_ms(stencil, reps)
    ms_add = _events_ms(add, reps)
    es = psi.element_size()
    stencil_bytes = 2 * es * nb * G + es * G
    res = dict(ms_per_step=ms_step, value=nb * G / (ms_step * 1e-3),
               ms_stencil=ms_stencil, ms_projections=ms_proj,
               ms_projector_add=ms_add,
               stencil_gbs=stencil_bytes / (ms_stencil * 1e-3) / 1e9,
               stencil_alg_bytes=stencil_bytes,
               step_gbs=2 * es * nb * G / (ms_step * 1e-3) / 1e9)
    # the multigrid preconditioner: all bands in one call (the throughput
    # figure) and in blocks of 16 (eigensolver-sized)
    d = torch.empty_like(psi)
    for blk, key in ((nb, 'precond'), (16, 'precond_blocks16')):
        pc = Preconditioner(gd, kin, block=blk)

        def run():
            for b0 in range(0, nb, blk):
                pc(psi[b0:b0 + blk], None, out=d[b0:b0 + blk])
        ms = _events_ms(run, max(2, args.steps // 4))
        res[key + '_ms'] = ms
        res[key + '_value'] = nb * G / (ms * 1e-3)
        del pc
    res['precond_gbs'] = 3.6875 * es * nb * G / (res['precond_ms'] * 1e-3) / 1e9
    res['hpsi_plus_precond_value'] = nb * G / (
        (ms_step + res['precond_ms']) * 1e-3)
    del psi, out, P, c, d
    torch.cuda.empty_cache()
    return res


def fp32_error(sysm, ham, nb, dev):
    """Largest per-band relative 2-norm error of FP32 H psi and of the FP32
    preconditioner against the FP64 device path (bit-exact with the
    reference's C) on the same FP32-representable bands."""
    import torch
    from gpawdft_amd.preconditioner import Preconditioner
    from gpawdft_amd.synthetic import smooth_bands_device
    kin, pt = sysm.operators()
    x32 = smooth_bands_device(nb, sysm.gd.n_c, 7, dtype=torch.float32)
    x64 = x32.double()

    def err(a, b):
        d = (a.double() - b).flatten(1).norm(dim=1)
        return float(torch.max(d / b.flatten(1).norm(dim=1)))
    o32 = torch.empty_like(x32)
    o64 = torch.empty_like(x64)
    ham.apply_fused(x32, o32, kin, pt)
    ham.apply_fused(x64, o64, kin, pt)
    e_h = err(o32, o64)
    pc = Preconditioner(sysm.gd, kin, block=nb)
    e_p = err(pc(x32, None), pc(x64, None))
    del x32, x64, o32, o64, pc
    torch.cuda.empty_cache()
    return {'hpsi_max_band_rel_err': e_h, 'precond_max_band_rel_err': e_p,
            'bands': nb}


def main():
    args = parse()
    if args.gpus != 1:
        print('bench.py: this build runs on one GPU; --gpus %d is not '
              'supported (bands shard across GPUs with no communication for '
              'H psi, see the design notes)' % args.gpus, file=sys.stderr)
        sys.exit(2)

    import numpy as np
    import torch

    from gpawdft_amd.hamiltonian import Hamiltonian
    from gpawdft_amd.synthetic import System

    assert torch.cuda.is_available(), 'bench.py needs a HIP device'
    dev = torch.device('cuda')
    N, nb = args.N, args.bands
    sysm = System(N, 0.18, args.atoms, seed=2024)
    gd = sysm.gd
    G = int(np.prod(gd.n_c))
    ham = Hamiltonian(gd, [sysm.vt_G], sysm.dH_asp)

    if args.copy_calibration:
        copy_calibration(4 * nb * G)

    f64 = hpsi_block(sysm, ham, nb, torch.float64, args, dev)
    f32 = hpsi_block(sysm, ham, nb, torch.float32, args, dev)
    f32['vs_f64'] = fp32_error(sysm, ham, nb, dev)

    subspace = None
    if not args.no_subspace:
        subspace = subspace_step(args.steps)

    kpoint = None
    if not args.no_kpoint:
        kpoint = complex_hpsi(sysm, nb, args.steps)

    ragged = None
    if not args.no_ragged:
        # the single system's FP32 costs per unit: stencil + preconditioner
        # per band*point, projections + projector add per band*atom
        unit_costs = {
            'ms_per_band_point': (f32['ms_stencil'] + f32['precond_ms']) /
                                 (nb * N ** 3),
            'ms_per_band_atom': (f32['ms_projections'] +
                                 f32['ms_projector_add']) / (nb * args.atoms)}
        ragged = ragged_batch(args.ragged_systems, args.steps,
                              f32['hpsi_plus_precond_value'], unit_costs)

    poisson = None
    if not args.no_poisson:
        poisson = poisson_solve(2 * N, args.no_cpu)

    ttt = None
    if not args.no_ttt:
        ttt = time_to_1e8(args.ttt_max_iter)

    c4 = None
    if args.learned_c4:
        c4 = learned_c4(args.c4_seconds)

    # CPU baseline: the reference's own C on all host cores (one process
    # per core) and the C oracle, on a bounded sample of the same system
    cpu = None
    if not args.no_cpu:
        cpu = cpu_baseline(args.cpu_seconds)

    traffic = measured_traffic()
    line = {
        'metric': 'band*gridpts/s for H*psi at 96^3x256',
        'value': f64['value'],
        'unit': 'band*gridpts/s',
        'n_gpus': 1,
        'steps': args.steps,
        'warmup': args.warmup,
        'ms_per_step': f64['ms_per_step'],
        'higher_is_better': True,
        'scaling': 'weak',
        'vs_baseline': None,
        'dtype': 'f64',
        'data': 'synthetic (seeded Gaussian-well potential, Gaussian '
                'projectors, smoothed N(0,1) bands)',
        'config': {'workload': 'H*psi, 96^3 periodic grid, h=0.18 A, %d '
                               'bands, %d atoms x 9 projectors, nn=3 stencil'
                               % (nb, args.atoms),
                   'grid': [N, N, N], 'bands': nb, 'atoms': args.atoms},
        'roofline': {'bound': 'hbm',
                     'kernel': 'fd_axis_mb_kernel<double,3,EPI_POT,1,32> '
                               '(T psi + v psi, %d bands, one per '
                               'workgroup)' % nb,
                     'achieved': f64['stencil_gbs'],
                     'peak': HBM_PEAK_GBS, 'unit': 'GB/s',
                     'frac': f64['stencil_gbs'] / HBM_PEAK_GBS,
                     'traffic': traffic,
                     'alg_bytes_per_launch': f64['stencil_alg_bytes'],
                     'ms_per_launch': f64['ms_stencil']},
        'step_roofline': {'bound': 'hbm', 'bytes_per_band_point': 16,
                          'achieved': f64['step_gbs'], 'peak': HBM_PEAK_GBS,
                          'unit': 'GB/s',
                          'frac': f64['step_gbs'] / HBM_PEAK_GBS},
        'cpu_baseline': cpu,
        'f64': f64,
        'f32': f32,
        'precond_roofline': {
            'bound': 'hbm', 'bytes_per_band_point': '3.6875*sizeof(T)',
            'f64_achieved': f64['precond_gbs'],
            'f32_achieved': f32['precond_gbs'], 'peak': HBM_PEAK_GBS,
            'unit': 'GB/s', 'f64_frac': f64['precond_gbs'] / HBM_PEAK_GBS,
            'f32_frac': f32['precond_gbs'] / HBM_PEAK_GBS},
        'subspace_c3': subspace,
        'time_to_1e-8': ttt,
        'ragged_batch': ragged,
        'poisson': poisson,
        'kpoint_c128': kpoint,
    }
    if c4 is not None:
        line['learned_c4'] = c4
    if cpu and 'value' in cpu:
        line['speedup_vs_cpu'] = {
            'hpsi_f64': f64['value'] / cpu['value'],
            'hpsi_f32': f32['value'] / cpu['value'],
            'hpsi_plus_precond_f64': (f64['hpsi_plus_precond_value'] /
                                      cpu['hpsi_plus_precond_value']),
            'hpsi_plus_precond_f32': (f32['hpsi_plus_precond_value'] /
                                      cpu['hpsi_plus_precond_value'])}
    print(json.dumps(line))


def subspace_step(steps):
    """The mixed-precision subspace step at 112^3 x 512 (64 atoms): FP32
    bands; S = dv psi psi^T and H = dv psi (H psi)^T on split-bfloat16 MFMA
    (six bf16 products per useful one, FP32 then FP64 accumulation), the
    FP64 inverse Cholesky and eigensolve, and the FP32 band rotation on the
    same split products.  MFMA utilisation counts the issued bf16 products
    (6 per multiply-add formed) against the dense bf16 peak."""
    import numpy as np
    import torch
    from gpawdft_amd import hs_operators as hs
    from gpawdft_amd.hamiltonian import Hamiltonian
    from gpawdft_amd.synthetic import System, smooth_bands_device
    sysm = System(112, 0.18, 64, seed=31)
    gd = sysm.gd
    kin, pt = sysm.operators()
    ham = Hamiltonian(gd, [sysm.vt_G], sysm.dH_asp)
    Nb = 512
    K = int(np.prod(gd.n_c))
    psi = smooth_bands_device(Nb, gd.n_c, 4, dtype=torch.float32)
    hpsi = torch.empty_like(psi)
    ham.apply_fused(psi, hpsi, kin, pt)
    S = torch.empty((Nb, Nb), dtype=torch.float64, device='cuda')
    H = torch.empty_like(S)
    reps = max(2, steps // 4)
    t = {}
    t['S'] = _events_ms(lambda: hs.grid_inner_products(
        gd, psi, psi, _transposed_result=S), reps)
    t['H'] = _events_ms(lambda: hs.grid_inner_products(
        gd, psi, hpsi, hermitian=True, _transposed_result=H), reps)
    S0 = S.clone()

    def chol():
        S.copy_(S0)
        hs.inverse_cholesky(S)
    t['inverse_cholesky'] = _events_ms(chol, reps)
    out = torch.empty_like(psi)
    t['rotate'] = _events_ms(lambda: hs.rotate(S, psi, out), reps)
    H0 = 0.5 * (H + H.t())
    w = torch.empty(Nb, dtype=torch.float64, device='cuda')
    H1 = H0.clone()
    t0 = time.perf_counter()
    sweeps = hs.diagonalize(H1, w)
    torch.cuda.synchronize()
    t['eigensolve'] = (time.perf_counter() - t0) * 1e3
    useful_S = Nb * (Nb + 1) * K            # dsyrk flops (one triangle)
    useful_H = 2 * Nb * Nb * K
    issued = lambda n_mac: 6 * 2 * n_mac      # six bf16 products per MAC
    res = {'workload': '112^3 grid x 512 FP32 bands, 64 atoms',
           'ms': t, 'jacobi_sweeps': sweeps,
           'total_ms': sum(t.values()),
           'S_useful_tflops': useful_S / (t['S'] * 1e-3) / 1e12,
           'H_useful_tflops': useful_H / (t['H'] * 1e-3) / 1e12,
           # S: the 128 x 128 tiles on and below the diagonal; H: all
           'S_mfma_util_bf16': issued((Nb // 128) * (Nb // 128 + 1) // 2 *
                                      128**2 * K) / (t['S'] * 1e-3) / 2.5e15,
           'H_mfma_util_bf16': issued(Nb * Nb * K) / (t['H'] * 1e-3) /
           2.5e15,
           'rotate_tflops': 2 * Nb * Nb * K / (t['rotate'] * 1e-3) / 1e12,
           'rotate_mfma_util_bf16': issued(Nb * Nb * K) /
           (t['rotate'] * 1e-3) / 2.5e15,
           'inverse_cholesky_gflops': Nb**3 / 3 / (t['inverse_cholesky'] *
                                                   1e-3) / 1e9}
    del psi, hpsi, out
    torch.cuda.empty_cache()
    return res


def complex_hpsi(sysm, nb, steps):
    """H psi for complex bands at a k-point (Bloch stencil, local
    potential, phased projector integrate / P dH / add) on the same 96^3
    system: the reference's operator sequence (gpaw/hamiltonian.py:
    426-460) in complex128."""
    import types
    import numpy as np
    import torch
    from gpawdft_amd.hamiltonian import FDWaveFunctions, Hamiltonian, KPoint
    from gpawdft_amd.lfc import LFC
    gd = sysm.gd
    k_c = np.array([0.25, 0.0, -0.375])
    phase = np.exp(2j * np.pi * np.array([[1, -1]] * 3) * k_c[:, None])
    pt = LFC(gd, [sysm.splines] * sysm.natoms,
             kd=types.SimpleNamespace(gamma=False, ibzk_qc=k_c[None]),
             dtype=complex)
    pt.set_positions(sysm.spos_ac)
    wfs = FDWaveFunctions(gd, pt, sysm.nn, complex)
    ham = Hamiltonian(gd, [sysm.vt_G], sysm.dH_asp)
    kpt = KPoint(q=0, phase_cd=phase)
    G = int(np.prod(gd.n_c))
    g = torch.Generator(device='cuda')
    g.manual_seed(3)
    psi = torch.randn((nb,) + tuple(int(n) for n in gd.n_c),
                      dtype=torch.complex128, device='cuda', generator=g)
    out = torch.empty_like(psi)
    ham.apply(psi, out, wfs, kpt)
    ev = [torch.cuda.Event(enable_timing=True) for _ in range(2)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        ham.apply(psi, out, wfs, kpt)
    torch.cuda.synchronize()
    ms = (time.perf_counter() - t0) / steps * 1e3
    ev[0].record()
    wfs.kin.apply(psi, out, phase)
    ev[1].record()
    ev[1].synchronize()
    ms_kin = ev[0].elapsed_time(ev[1])
    # the multigrid preconditioner on the same complex bands
    pc = wfs.make_preconditioner(nb)
    pc(psi, kpt, out=out)
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    for _ in range(steps):
        pc(psi, kpt, out=out)
    torch.cuda.synchronize()
    ms_pc = (time.perf_counter() - t0) / steps * 1e3
    res = {'workload': '96^3 periodic grid, %d complex128 bands, k = '
                       '(0.25, 0, -0.375), %d atoms x 9 projectors'
                       % (nb, sysm.natoms),
           'ms_per_step': ms, 'value': nb * G / (ms * 1e-3),
           'unit': 'band*gridpts/s', 'ms_stencil': ms_kin,
           'stencil_gbs': 2 * 16 * nb * G / (ms_kin * 1e-3) / 1e9,
           'precond_ms': ms_pc,
           'precond_gbs': 3.6875 * 16 * nb * G / (ms_pc * 1e-3) / 1e9}
    del psi, out
    torch.cuda.empty_cache()
    return res


def poisson_solve(N, no_cpu):
    """FP64 multigrid Poisson solve (gpaw/poisson.py, Jacobi smoothing,
    nn = 3) of a charged periodic density on the N^3 fine grid of the H psi
    system (twice its points per axis, as GPAW's finegd), tolerance 2e-10;
    the CPU oracle's V-cycle timed on one cycle for comparison."""
    import numpy as np
    import torch
    from gpawdft_amd.grid_descriptor import GridDescriptor
    from gpawdft_amd.poisson import PoissonSolver
    from gpawdft_amd.synthetic import Bohr
    n_c = np.array([N, N, N])
    gd = GridDescriptor(n_c, n_c * 0.09 / Bohr, True)
    x = np.arange(N) * 2 * np.pi / N
    rho = (np.cos(x)[:, None, None] * np.sin(2 * x)[None, :, None] *
           np.cos(3 * x)[None, None, :] + 0.1)
    ps = PoissonSolver()
    ps.set_grid_descriptor(gd)
    ps.initialize()
    drho = torch.from_numpy(rho).cuda()
    phi = torch.zeros_like(drho)
    ps.solve(phi, drho)                      # warm up (tables, scratch)
    times = []
    for _ in range(3):                       # the median of 3 solves
        phi.zero_()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        niter = ps.solve(phi, drho)
        torch.cuda.synchronize()
        times.append(time.perf_counter() - t0)
    t = sorted(times)[1]
    out = {'workload': 'FP64 %d^3 periodic, nn=3, Jacobi, eps 2e-10, '
                       '%d levels' % (N, ps.levels + 1),
           'v_cycles': niter, 'seconds': t, 'seconds_all': times,
           'ms_per_v_cycle': t / niter * 1e3}
    if not no_cpu:
        sys.path.insert(0, os.path.join(ROOT, 'oracle'))
        import poisson as P
        ref = P.Poisson(gd)
        phis = [np.zeros(tuple(n_c))] + [None] * ref.levels
        rhos = [rho - rho.mean()] + [None] * ref.levels
        t0 = time.perf_counter()
        ref.iterate2(phis, rhos)
        tc = time.perf_counter() - t0
        out['cpu_ms_per_v_cycle'] = tc * 1e3
        out['cpu_sample'] = 'one V-cycle of the C oracle (1 thread)'
        out['speedup_per_v_cycle'] = tc / (t / niter)
    return out


def ragged_batch(nsys, steps, single_rate, unit_costs=None):
    """Throughput of one step (H psi + multigrid preconditioner, FP32) over
    nsys independent systems (grids from {32,48,64,80}^3, 16-256 bands, 4-48
    atoms): the step issued eagerly versus one replay of a graph holding the
    same launches in parallel branches, after the launch-shape autotuner.
    Systems on one grid share a preconditioner call over all their bands;
    `vs_single_system` compares the graph with the single-system FP32
    H psi + preconditioner rate at 96^3 x 256 (all bands in one
    preconditioner call).  The batch has several times the single system's
    projector work per band*point (small grids crowded with atoms), so
    `vs_single_system_density_adjusted` prices the batch at the single
    system's own FP32 costs (stencil + preconditioner per band*point,
    projections + projector add per band*atom, run one after the other)
    and divides that time by the graph's."""
    import torch
    from gpawdft_amd.ragged import RaggedBatch, random_specs
    t0 = time.perf_counter()
    rb = RaggedBatch(random_specs(nsys, seed=0), block=None)
    setup = time.perf_counter() - t0
    tuning = rb.autotune(reps=2)
    rb.capture()
    res = {}
    for name, fn in (('sequential', rb.run_sequential), ('graph', rb.replay)):
        fn()
        torch.cuda.synchronize()
        t0 = time.perf_counter()
        for _ in range(steps):
            fn()
        torch.cuda.synchronize()
        dt = (time.perf_counter() - t0) / steps
        res[name] = {'ms_per_step': dt * 1e3,
                     'band_gridpts_per_s': rb.band_points / dt}
    res['graph_speedup'] = (res['sequential']['ms_per_step'] /
                            res['graph']['ms_per_step'])
    res['graph_branches'] = rb.nstreams
    res['systems'] = nsys
    res['grids'] = len(rb.grids)
    res['precond_call'] = 'all bands of a grid in one call'
    # atoms per grid point against the single 96^3 system (32 atoms): the
    # projector share of the work per band*point
    res['projector_density_vs_single'] = (
        rb.band_atoms / rb.band_points) / (32.0 / 96 ** 3)
    if single_rate:
        res['single_system_rate'] = single_rate
        res['vs_single_system'] = res['graph']['band_gridpts_per_s'] / single_rate
    if unit_costs:
        expect = (rb.band_points * unit_costs['ms_per_band_point'] +
                  rb.band_atoms * unit_costs['ms_per_band_atom'])
        res['single_system_costs'] = dict(unit_costs,
                                          batch_ms_at_these_costs=expect)
        res['vs_single_system_density_adjusted'] = (
            expect / res['graph']['ms_per_step'])
    res['band_gridpts_per_step'] = rb.band_points
    res['setup_s'] = setup
    res['wg_targets'] = {'%d pts x %d bands' % k: v for k, v in tuning.items()}
    del rb
    torch.cuda.empty_cache()
    return res


def time_to_1e8(max_iter):
    """Wall-clock seconds for FP64 RMM-DIIS to bring the occupied-band
    residual error below 1e-8 with the multigrid preconditioner and with the
    learned one (multigrid fallback), on a held-out 32^3 system of the same
    generators (h = 0.18 A, 3 wells, unit-norm projectors, 16 bands, 12
    occupied), both from the same Gaussian-orbital start.  Both runs must
    end on the same eigenvalues for the times to compare like with like:
    eps_max_diff is the largest difference of their occupied eigenvalues."""
    import numpy as np
    from gpawdft_amd.learned import UNet
    from gpawdft_amd.precond_training import time_to_tolerance
    from gpawdft_amd.synthetic import System
    net = UNet.load(os.path.join(ROOT, 'gpawdft_amd', 'data',
                                 'unet_precond.npz'))
    sysm = System(32, 0.18, 3, seed=4242, unit_projectors=True)
    out = {'workload': '32^3 periodic grid, h=0.18 A, 3 wells, unit-norm '
                       'projectors, 16 FP64 bands (12 occupied) from '
                       'Gaussian orbitals on the wells, blocksize 8, '
                       'tolerance 1e-8, at most %d iterations' % max_iter}
    for name, n in (('multigrid', None), ('learned', net)):
        out[name] = time_to_tolerance(sysm, n, nbands=16, nocc=12,
                                      max_iter=max_iter)
    e_m = np.array(out['multigrid']['eps_n'][:12])
    e_l = np.array(out['learned']['eps_n'][:12])
    out['eps_max_diff'] = float(np.abs(e_m - e_l).max())
    return out


def learned_c4(max_seconds):
    """The learned preconditioner at its stated evaluation size: FP64
    RMM-DIIS on a held-out 96^3 system (h = 0.18 A, 32 wells, unit-norm
    projectors, 256 bands, 192 occupied, blocks of 16) from Gaussian
    orbitals, with the multigrid and with the learned preconditioner
    (multigrid fallback), each until sum_occ <R|R> < 1e-8 or max_seconds.
    Progress goes to stderr."""
    from gpawdft_amd.learned import UNet
    from gpawdft_amd.precond_training import time_to_tolerance
    from gpawdft_amd.synthetic import System
    net = UNet.load(os.path.join(ROOT, 'gpawdft_amd', 'data',
                                 'unet_precond.npz'))
    sysm = System(96, 0.18, 32, seed=5151, unit_projectors=True)
    out = {'workload': '96^3 periodic grid, h=0.18 A, 32 wells, unit-norm '
                       'projectors, 256 FP64 bands (192 occupied) from '
                       'Gaussian orbitals on the wells, blocksize 16, '
                       'tolerance 1e-8, at most %.0f s per run' % max_seconds}
    for name, n in (('multigrid', None), ('learned', net)):
        def progress(it, err, sec, name=name):
            print('[c4 %s] iteration %d error %.3e %.1f s' % (name, it, err,
                                                               sec),
                  file=sys.stderr, flush=True)
        r = time_to_tolerance(sysm, n, nbands=256, nocc=192, max_iter=10000,
                              blocksize=16, max_seconds=max_seconds,
                              progress=progress)
        r['eps_n'] = r['eps_n'][:8]
        out[name] = r
    return out


def measured_traffic():
    """HBM bytes per launch of the roofline kernel from the committed
    rocprofv3 counter summary (FETCH_SIZE + WRITE_SIZE, scaled by a plain
    copy's counters), or None when absent."""
    import re
    path = os.path.join(ROOT, 'profiles', 'fd_axis_f64_96x256_traffic.md')
    if not os.path.exists(path):
        return None
    with open(path) as fh:
        m = re.search(r'^hbm_bytes_per_launch:\s*([0-9.eE+]+)', fh.read(), re.M)
    return float(m.group(1)) if m else None


def copy_calibration(nbytes, reps=3):
    """A plain device-to-device copy of nbytes: its FETCH_SIZE / WRITE_SIZE
    counters calibrate the stencil's (run under rocprofv3 --pmc)."""
    import torch
    src = torch.ones(nbytes // 4, dtype=torch.float32, device='cuda')
    dst = torch.empty_like(src)
    for _ in range(reps):
        dst.copy_(src)
    torch.cuda.synchronize()


def cpu_baseline(target_s):
    """The CPU leg (rank 0, N = 1): oracle/cpu_baseline.py in a child
    process, which times the reference's own C (built from its sources into
    oracle/_ref; one process per usable core, bands split over them, as
    GPAW runs without GPAW_OMP) and the C oracle on the same 16 bands of the
    same system.  `value` is the reference's H psi throughput on the host
    cores when its build is present, else the oracle's."""
    import subprocess
    cmd = [sys.executable, os.path.join(ROOT, 'oracle', 'cpu_baseline.py'),
           '--seconds', str(target_s), '--bands', '16']
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=900)
    if r.returncode != 0:
        return {'error': r.stderr[-2000:]}
    res = json.loads(r.stdout.strip().splitlines()[-1])
    ref = res.get('reference', {})
    base = ref if 'hpsi_value' in ref else res['port']
    cores = base.get('processes', base.get('threads'))
    return {'value': base['hpsi_value'], 'unit': 'band*gridpts/s',
            'cores': cores, 'kind': base['kind'],
            'hpsi_plus_precond_value': base['hpsi_plus_precond_value'],
            'precond_value': base['precond_value'],
            'sample': '%d FP64 bands of the same 96^3 system, %d repeats '
                      'of H psi then of the multigrid preconditioner; %s'
                      % (base['bands'], base['reps'],
                         'the reference C, one process per core' if
                         base['kind'] == 'reference' else
                         'the C oracle, one OpenMP thread per band'),
            'cpu_model': res.get('cpu_model'), 'nproc': res.get('nproc'),
            'affinity': res.get('affinity'),
            'port': res['port'],
            'port_over_reference': res.get('port_over_reference')}


if __name__ == '__main__':
    main()
