"""Finite-difference multigrid Poisson solver on the device.

Drop-in for gpaw/poisson.py:47-315: `PoissonSolver(nn=3, relax='J',
eps=2e-10, maxiter=1000)` with `set_grid_descriptor(gd)`, `initialize()`,
`solve(phi, rho, charge=None, eps=None, maxcharge=1e-6,
zero_initial_phi=False)` returning the iteration count, and `iterate2`.
The operator is -1/(4 pi) times the nn-th order Laplacian on the fine grid
(or the Mehrstellen pair A phi = B rho for nn='M'), 7-point Laplacians on
the coarse grids, nn=1 transformers between levels, weighted Jacobi
smoothing (2 pre- / 1 post-sweeps at weight 2/3 on the fine grid, 4 / 4 at
weight 1 below, 8 / 8 on the coarsest) or, with relax='GS', Gauss-Seidel
sweeps in the reference's lexicographic order.  Every step runs in this
library's kernels: relax, stencil, restrict / interpolate, batched axpy and
dot.

A charged system with zero boundaries is solved as the reference does
(gpaw/poisson.py:240-298): the monopole is moved into a Gaussian
(gpaw/utilities/gauss.py:193-238, L = 0) whose potential is known in
closed form, the neutral rest goes through the multigrid solver, and the
Gaussian's potential is added back; `use_charge_center` places the
Gaussian at the centre of the majority charge.  The Gaussian is tabulated
on the host in FP64 once per grid and centre.

Not covered: the multipole removal (remove_moment) and the FFT /
dipole-layer solvers.
"""
import ctypes
from math import pi

import numpy as np

from gpawdft_amd._lib import check, lib
from gpawdft_amd.device import DeviceView, stream_ptr, torch
from gpawdft_amd.eigensolvers import axpy, dots
from gpawdft_amd.fd_operators import Laplace, LaplaceA, LaplaceB
from gpawdft_amd.transformers import Transformer


class PoissonConvergenceError(RuntimeError):
    pass


def create_poisson_solver(name='fd', **kwargs):
    if name == 'fd':
        return PoissonSolver(**kwargs)
    raise NotImplementedError('Poisson solver %r is not part of this build'
                              % name)


def PoissonSolver(dipolelayer=None, **kwargs):
    if dipolelayer is not None:
        raise NotImplementedError('dipole-layer correction is not part of '
                                  'this build')
    return FDPoissonSolver(**kwargs)


def grid_point_distance_vectors(gd, r_v):
    """r_vG: the grid points' displacement from r_v, as
    GridDescriptor.get_grid_point_distance_vectors (gpaw/grid_descriptor.py:
    638-657) for cells without periodic axes (no minimum-image shift)."""
    idx = np.meshgrid(*[np.arange(n) for n in gd.n_c], indexing='ij')
    s_c = np.linalg.solve(gd.cell_cv.T, np.asarray(r_v, float))
    s_cG = [(idx[c] + gd.beg_c[c]) / gd.N_c[c] - s_c[c] for c in range(3)]
    if gd.pbc_c.any():
        for c in range(3):
            if gd.pbc_c[c]:
                for _ in range(2):
                    s_cG[c] = s_cG[c] - (2 * s_cG[c]).astype(int)
    return np.array([sum(s_cG[c] * gd.cell_cv[c, v] for c in range(3))
                     for v in range(3)])


def gaussian_monopole(gd, a=19.0, center=None):
    """(rho_g, phi_g) of the generalized Gaussian L = 0 of
    gpaw/utilities/gauss.py:193-238: width set from the cell (a / r_min^2
    around `center`, or 4 a max|icell|^2 at the cell's centre),
    g = sqrt(4 a^3) / pi exp(-a r^2) and its potential
    2 sqrt(pi) erf(sqrt(a) r) / r (r^2 floored at 1e-12, as
    gpaw/utilities/tools.py:106-125)."""
    from scipy.special import erf
    origin = 0.5 * gd.cell_cv.sum(0) if center is None else center
    r_vG = grid_point_distance_vectors(gd, origin)
    r2 = np.sum(r_vG**2, axis=0)
    r2 = np.where(r2 < 1e-12, 1e-12, r2)
    r = np.sqrt(r2)
    if center is None:
        a = 4 * a * (gd.icell_cv**2).sum(1).max()
    else:
        cell_center = gd.cell_cv.sum(1) / 2
        r_min = (cell_center - np.abs(center - cell_center)).min()
        a = a / r_min**2
    rho_g = np.sqrt(a**3 * 4) / pi * np.exp(-a * r2)
    phi_g = 2.0 * 1.7724538509055159 * erf(np.sqrt(a) * r) / r
    return np.ascontiguousarray(rho_g), np.ascontiguousarray(phi_g)


def dipole_moment(gd, rho_g):
    """GridDescriptor.calculate_dipole_moment (gpaw/grid_descriptor.py:
    576-585) for one domain."""
    rho_01 = rho_g.sum(axis=2)
    rho_02 = rho_g.sum(axis=1)
    rho_cg = [rho_01.sum(axis=1), rho_01.sum(axis=0), rho_02.sum(axis=0)]
    rhog_c = [np.dot(np.arange(gd.beg_c[c], gd.end_c[c]), rho_cg[c])
              for c in range(3)]
    return -np.dot(rhog_c, gd.h_cv) * gd.dv


class FDPoissonSolver:
    def __init__(self, nn=3, relax='J', eps=2e-10, maxiter=1000,
                 remove_moment=None, use_charge_center=False):
        if relax not in ('J', 'GS'):
            raise NotImplementedError('Relaxation method %s' % relax)
        if remove_moment is not None:
            raise NotImplementedError('multipole removal is not part of '
                                      'this build')
        self.relax = relax
        self.relax_method = 1 if relax == 'GS' else 2
        self.nn = nn
        self.eps = eps
        self.maxiter = maxiter
        self.remove_moment = remove_moment
        self.use_charge_center = use_charge_center
        self.description = None

    def todict(self):
        return {'name': 'fd', 'nn': self.nn, 'relax': self.relax,
                'eps': self.eps, 'remove_moment': self.remove_moment}

    def get_stencil(self):
        return self.nn

    def set_grid_descriptor(self, gd):
        self.gd = gd
        scale = -0.25 / pi
        if self.nn == 'M':
            self.operators = [LaplaceA(gd, -scale)]
            self.B = LaplaceB(gd)
        else:
            self.operators = [Laplace(gd, scale, self.nn)]
            self.B = None
        self.interpolators = []
        self.restrictors = []
        self.presmooths = [2]
        self.postsmooths = [1]
        self.weights = [2.0 / 3.0]
        level = 0
        while level < 8:
            try:
                gd2 = gd.coarsen()
            except ValueError:
                break
            self.operators.append(Laplace(gd2, scale, 1))
            self.interpolators.append(Transformer(gd2, gd))
            self.restrictors.append(Transformer(gd, gd2))
            self.presmooths.append(4)
            self.postsmooths.append(4)
            self.weights.append(1.0)
            level += 1
            gd = gd2
        self.levels = level

    def get_description(self):
        coarsest = ' x '.join(str(N) for N in self.operators[-1].gd.N_c)
        return ('Jacobi solver with %d multi-grid levels\n'
                '    Coarsest grid: %s points\n    Stencil: %s\n'
                '    Tolerance: %e\n    Max iterations: %d'
                % (self.levels + 1, coarsest,
                   self.operators[0].description, self.eps, self.maxiter))

    def initialize(self, load_gauss=False, device='cuda'):
        gd = self.gd
        dt = torch.float64
        self.rhos = [gd.empty(device=device)]
        self.phis = [None]
        self.residuals = [gd.empty(device=device)]
        for level in range(self.levels):
            gd2 = gd.coarsen()
            self.phis.append(gd2.empty(device=device))
            self.rhos.append(gd2.empty(device=device))
            self.residuals.append(gd2.empty(device=device))
            gd = gd2
        self.step = 0.66666666 / self.operators[0].get_diagonal_element()
        self.presmooths[self.levels] = 8
        self.postsmooths[self.levels] = 8
        self._ones = torch.ones(tuple(int(n) for n in self.gd.n_c), dtype=dt,
                                device=device)
        # the V-cycle's axpy coefficient, resident on the device (a host
        # coefficient would be copied per call, waiting for the queue)
        self._minus_one = torch.full((1,), -1.0, dtype=dt, device=device)
        self._norm = torch.zeros(1, dtype=dt, device=device)
        self._vc = None
        if load_gauss:
            self.load_gauss()

    def load_gauss(self, center=None):
        """The L = 0 Gaussian charge and its potential on the grid
        (gpaw/poisson.py:195-199), on the device."""
        if not hasattr(self, 'rho_gauss') or center is not None:
            rho_g, phi_g = gaussian_monopole(self.gd, center=center)
            dev = self._ones.device
            self.rho_gauss = torch.from_numpy(rho_g).to(dev)
            self.phi_gauss = torch.from_numpy(phi_g).to(dev)

    def _sum(self, a):
        """sum of a grid (a batched dot with ones)."""
        return float(dots(a[None], self._ones[None])[0])

    def solve(self, phi, rho, charge=None, eps=None, maxcharge=1e-6,
              zero_initial_phi=False):
        """phi (in/out) and rho: FP64 device tensors or numpy arrays of the
        grid's shape.  Returns the number of V-cycles."""
        assert tuple(phi.shape) == tuple(self.gd.n_c)
        assert tuple(rho.shape) == tuple(self.gd.n_c)
        if eps is None:
            eps = self.eps
        vphi = DeviceView(phi)
        vrho = DeviceView(rho)
        actual_charge = self._sum(vrho.t) * self.gd.dv
        background = actual_charge / self.gd.dv / np.prod(self.gd.N_c)
        if charge is None:
            charge = actual_charge
        if abs(charge) > maxcharge and not self.gd.pbc_c.any():
            niter = self._solve_charged_zero_boundary(vphi.t, vrho.t,
                                                      actual_charge, eps,
                                                      zero_initial_phi)
            vphi.finish()
            return niter
        if abs(charge) > maxcharge and not self.gd.pbc_c.all():
            raise NotImplementedError('Charged systems with mixed '
                                      'periodic/zero boundary conditions')
        if abs(charge) > maxcharge and zero_initial_phi:
            vphi.t.zero_()
        neutral = vrho.t.clone()
        axpy(np.array([-background]), self._ones[None], neutral[None])
        niter = self.solve_neutral(vphi.t, neutral, eps=eps)
        vphi.finish()
        return niter

    def _solve_charged_zero_boundary(self, phi, rho, actual_charge, eps,
                                     zero_initial_phi):
        """gpaw/poisson.py:249-298: subtract a Gaussian carrying the
        monopole, solve for the neutral rest, add the Gaussian's
        potential."""
        if self.use_charge_center:
            rho_np = rho.cpu().numpy()
            sign = actual_charge / abs(actual_charge)
            rho_sign = rho_np * sign
            rho_sign[rho_sign < 0] = 0
            absolute_charge = float(rho_sign.sum()) * self.gd.dv
            center = -dipole_moment(self.gd, rho_sign) / absolute_charge
            border_offset = np.inner(self.gd.h_cv, np.array((7, 7, 7)))
            borders = np.inner(self.gd.h_cv, self.gd.N_c) - border_offset
            if np.any(center > borders) or np.any(center < border_offset):
                raise RuntimeError('Poisson solver: center of charge '
                                   'outside borders - please increase box')
            self.load_gauss(center=center)
        else:
            self.load_gauss()
        q = actual_charge / np.sqrt(4 * pi)
        neutral = rho.clone()
        axpy(np.array([-q]), self.rho_gauss[None], neutral[None])
        if zero_initial_phi:
            phi.zero_()
        else:
            axpy(np.array([-q]), self.phi_gauss[None], phi[None])
        niter = self.solve_neutral(phi, neutral, eps=eps)
        axpy(np.array([q]), self.phi_gauss[None], phi[None])
        return niter

    def solve_neutral(self, phi, rho, eps=2e-10):
        self.phis[0] = phi
        if self.B is None:
            self.rhos[0].copy_(rho)
        else:
            self.B.apply(rho, self.rhos[0])
        niter = 1
        while self.iterate2(self.step) > eps and niter < self.maxiter:
            niter += 1
        if niter == self.maxiter:
            raise PoissonConvergenceError(
                'Poisson solver did not converge in %d iterations!'
                % self.maxiter)
        # zero average potential on periodic grids
        if self.gd.pbc_c.all():
            ave = self._sum(phi) / np.prod(self.gd.N_c)
            axpy(np.array([-ave]), self._ones[None], phi[None])
        return niter

    def iterate2(self, step, level=0):
        """One V-cycle from `level` (gpaw/poisson.py:278-311); at level 0
        returns sum(residual^2) dv.  From level 0 the whole cycle is one
        library call (gpd_poisson_vcycle), which walks the levels with the
        differences formed in the stencils and the interpolations and the
        coarsest levels in one launch.  phi and the residual of level 0 and
        the norm are those of iterate2_calls bit for bit; the grids below
        are its scratch (some are not written at all)."""
        if level == 0:
            return self._vcycle()
        return self.iterate2_calls(step, level)

    def _vcycle(self):
        phi = self.phis[0]
        if (phi.dtype != torch.float64 or not phi.is_contiguous()
                or phi.device != self._norm.device):
            raise TypeError('phi must be a contiguous FP64 grid on the '
                            'solver\'s device')
        if self._vc is None:
            n = self.levels + 1
            vp = ctypes.c_void_p
            self._vc = {
                'ops': (vp * n)(*[op.handle for op in self.operators]),
                'res': (vp * max(1, n - 1))(*[t.handle
                                              for t in self.restrictors]),
                'int': (vp * max(1, n - 1))(*[t.handle
                                              for t in self.interpolators]),
                'phis': (vp * n)(*([0] + [p.data_ptr()
                                          for p in self.phis[1:]])),
                'rhos': (vp * n)(*[r.data_ptr() for r in self.rhos]),
                'resid': (vp * n)(*[r.data_ptr() for r in self.residuals]),
                'pre': (ctypes.c_int * n)(*self.presmooths[:n]),
                'post': (ctypes.c_int * n)(*self.postsmooths[:n]),
                'w': (ctypes.c_double * n)(*self.weights[:n])}
        t = self._vc
        t['phis'][0] = phi.data_ptr()
        check(lib().gpd_poisson_vcycle(
            self.levels, t['ops'], t['res'], t['int'], t['phis'], t['rhos'],
            t['resid'], t['pre'], t['post'], t['w'], self.relax_method,
            float(self.gd.dv), self._minus_one.data_ptr(),
            self._norm.data_ptr(), stream_ptr()), 'Poisson V-cycle')
        return float(self._norm.cpu()[0])

    def iterate2_calls(self, step, level=0):
        """iterate2 issued one operator call at a time, as the reference
        does (gpaw/poisson.py:278-311)."""
        residual = self.residuals[level]
        op = self.operators[level]
        if level < self.levels:
            op.relax(self.relax_method, self.phis[level], self.rhos[level],
                     self.presmooths[level], self.weights[level])
            op.apply(self.phis[level], residual)
            axpy(self._minus_one, self.rhos[level][None], residual[None])
            self.restrictors[level].apply(residual, self.rhos[level + 1])
            self.phis[level + 1].zero_()
            self.iterate2_calls(4.0 * step, level + 1)
            self.interpolators[level].apply(self.phis[level + 1], residual)
            axpy(self._minus_one, residual[None], self.phis[level][None])
        op.relax(self.relax_method, self.phis[level], self.rhos[level],
                 self.postsmooths[level], self.weights[level])
        if level == 0:
            op.apply(self.phis[level], residual)
            axpy(self._minus_one, self.rhos[level][None], residual[None])
            return float(dots(residual[None], residual[None],
                              self.gd.dv)[0])
