// One V-cycle of the finite-difference Poisson solver's multigrid
// (gpaw/poisson.py:278-311, PoissonSolver.iterate2 from level 0), issued
// from the host in one call.
//
// The reference recurses in Python, one operator call at a time; issuing
// the ~90 launches of a V-cycle one Python call each made the solve
// host-bound (about 19 us per call against 1.2 ms of kernels per cycle).
// Here the cycle's kernels run in the same order with the same rounding as
// the call-by-call sequence (relax, stencil, transformers, axpy, dot), bit
// for bit; the differences (op phi - rho and phi - the interpolated
// correction) are epilogues of the stencil and the interpolation, and the
// Jacobi sweeps alternate between phi and the level's residual array.  A
// cycle at 192^3 has 410 us of kernels (840 with the differences and the
// copies of an odd sweep as passes of their own, the norm's sum on 64
// workgroups and a launch for each sweep and each step of the coarsest
// levels), of which 80 are the 24 sweeps of the levels of 96^3 to 24^3.  Clearing
// the next level's phi is a small fill kernel (no hipMemsetAsync, so the call
// can be captured into a graph); nothing here allocates except what the dot and
// stencils off the axes allocate stream-ordered themselves.
#include "common.hpp"
#include "fd.hpp"
#include "transformer.hpp"

namespace gpd {

__global__ void fill_zero_f64_kernel(double* __restrict__ p, long n)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = 0.0;
}

// ------------------------------------------------------------------ //
// The levels that fit into the LDS of one workgroup together, in one launch:
// from phi = 0 on the finest of them to its phi, sweep for sweep the
// arithmetic of the stencil, restriction and interpolation kernels (three
// arrays a level: phi, a second one for the next sweep or the residual, rho).
// A sweep is the latency of its chain of sums and its division, one barrier,
// instead of a launch: 12^3, 6^3 and 3^3 with 24 sweeps take 40 us, in 36
// launches 180.

constexpr int kBottomLevels = 8;
constexpr int kBottomThreads = 1024;
constexpr size_t kBottomBytes = 150 * 1024;   // of the 160 KB of a CU

struct BottomLevel {
    int n[3];
    int pbc[3];
    int off;               // of its three arrays in LDS
    int pre, post;
    float inv1, inv2;      // 1 / n[1], 1 / n[2]
    double c0, c[3][2], w;
    TransformDims down, up;   // restriction from it, interpolation to it
};

struct BottomArgs {
    int count;
    BottomLevel l[kBottomLevels];
};

struct Point {
    int i0, i1, i2;
};

// q / n for 0 <= q < 2^16 from the reciprocal (an integer division is many
// instructions): (q + 0.5) / n is at least 0.5 / n from an integer, and its
// error below q / n * 2^-22
__device__ __forceinline__ int quotient(int q, float inv)
{
    return (int)(((float)q + 0.5f) * inv);
}

__device__ __forceinline__ Point point_of(const BottomLevel& l, int q)
{
    const int r = quotient(q, l.inv2), i0 = quotient(r, l.inv1);
    return {i0, r - i0 * l.n[1], q - r * l.n[2]};
}

// index at most n beyond the axis: inside, or -1 at a zero boundary
__device__ __forceinline__ int wrap_once(int i, int n, int pbc)
{
    const int j = i < 0 ? i + n : (i >= n ? i - n : i);
    return pbc || j == i ? j : -1;
}

__device__ __forceinline__ double at(const double* f, const BottomLevel& l, int i0, int i1, int i2)
{
    i0 = wrap_once(i0, l.n[0], l.pbc[0]);
    i1 = wrap_once(i1, l.n[1], l.pbc[1]);
    i2 = wrap_once(i2, l.n[2], l.pbc[2]);
    const bool in = i0 >= 0 && i1 >= 0 && i2 >= 0;
    const double v = f[in ? (i0 * l.n[1] + i1) * l.n[2] + i2 : 0];
    return in ? v : 0.0;
}

// s plus the neighbours' terms of point q: axis 2, 1, 0, each +1 then -1
__device__ __forceinline__ double neighbours(const BottomLevel& l, const double* f, int q,
                                             double s)
{
    const Point p = point_of(l, q);
    const int i[3] = {p.i0, p.i1, p.i2}, step[3] = {l.n[1] * l.n[2], l.n[2], 1};
    double v[6];
#pragma unroll
    for (int k = 0; k < 6; k++) {
        const int ax = 2 - k / 2, d = k % 2 ? -1 : 1;
        const int j = wrap_once(i[ax] + d, l.n[ax], l.pbc[ax]);
        const double x = f[q + (max(j, 0) - i[ax]) * step[ax]];
        v[k] = j >= 0 ? x : 0.0;
    }
#pragma unroll
    for (int k = 0; k < 6; k++) s = madd<double>(s, v[k], l.c[2 - k / 2][k % 2]);
    return s;
}

__global__ __launch_bounds__(kBottomThreads) void poisson_bottom_kernel(
    BottomArgs a, const double* __restrict__ rho, double* __restrict__ phi)
{
    extern __shared__ double lds[];
    unsigned second = 0;   // bit l: phi of level l is in its second array
    auto points = [&](int l) { return a.l[l].n[0] * a.l[l].n[1] * a.l[l].n[2]; };
    auto array = [&](int l, int which) { return lds + a.l[l].off + which * points(l); };
    auto sweeps = [&](int l, int count) {
        const BottomLevel& v = a.l[l];
        const double* r = array(l, 2);
        for (int it = 0; it < count; it++) {
            const double* f = array(l, second >> l & 1);
            double* o = array(l, ~second >> l & 1);
            for (int q = threadIdx.x; q < points(l); q += kBottomThreads) {
                const double s = neighbours(v, f, q, 0.0);
                const double t1 = (1.0 - v.w) * f[q];
                const double t2 = (v.w * (r[q] - s)) / v.c0;
                o[q] = t1 + t2;
            }
            second ^= 1u << l;
            __syncthreads();
        }
    };

    for (int q = threadIdx.x; q < points(0); q += kBottomThreads) array(0, 2)[q] = rho[q];
    for (int l = 0; l < a.count; l++) {
        const BottomLevel& v = a.l[l];
        for (int q = threadIdx.x; q < points(l); q += kBottomThreads) array(l, 0)[q] = 0.0;
        __syncthreads();
        if (l == a.count - 1) {
            sweeps(l, v.post);
            break;
        }
        sweeps(l, v.pre);
        const double* f = array(l, second >> l & 1);
        double* res = array(l, ~second >> l & 1);
        for (int q = threadIdx.x; q < points(l); q += kBottomThreads)
            res[q] = neighbours(v, f, q, madd<double>(0.0, f[q], v.c0)) -
                     array(l, 2)[q];
        __syncthreads();
        const AxisMap* m = v.down.ax;
        for (int q = threadIdx.x; q < points(l + 1); q += kBottomThreads) {
            const Point p = point_of(a.l[l + 1], q);
            const int j0 = 2 * p.i0 + m[0].shift, j1 = 2 * p.i1 + m[1].shift;
            const int j2 = 2 * p.i2 + m[2].shift;
            array(l + 1, 2)[q] = restrict_point<2, double>([&](int t0) {
                return restrict_point<2, double>([&](int t1) {
                    return restrict_point<2, double>([&](int t2) {
                        return at(res, v, j0 + t0, j1 + t1, j2 + t2);
                    });
                });
            });
        }
    }
    for (int l = a.count - 2; l >= 0; l--) {
        const BottomLevel& v = a.l[l];
        const BottomLevel& u = a.l[l + 1];
        const double* f = array(l + 1, second >> (l + 1) & 1);
        double* o = array(l, second >> l & 1);
        const AxisMap* m = v.up.ax;
        for (int q = threadIdx.x; q < points(l); q += kBottomThreads) {
            const Point p = point_of(v, q);
            const int u0 = p.i0 + m[0].skip0, u1 = p.i1 + m[1].skip0, u2 = p.i2 + m[2].skip0;
            const int j0 = u0 / 2 + m[0].shift, j1 = u1 / 2 + m[1].shift;
            const int j2 = u2 / 2 + m[2].shift;
            // a point of an axis, or between two, of what g gives there
            auto along = [](int odd, auto g) {
                return odd ? interp_point<2, double>(g) : g(0);
            };
            o[q] -= along(u0 & 1, [&](int t0) {
                return along(u1 & 1, [&](int t1) {
                    return along(u2 & 1, [&](int t2) {
                        return at(f, u, j0 + t0, j1 + t1, j2 + t2);
                    });
                });
            });
        }
        __syncthreads();
        sweeps(l, v.post);
    }
    const double* f = array(0, second & 1);
    for (int q = threadIdx.x; q < points(0); q += kBottomThreads) phi[q] = f[q];
}

// ------------------------------------------------------------------ //
// Several Jacobi sweeps in one launch for a second-order stencil along the
// axes: a workgroup takes 16^3 points, `sweeps` of them on each side a halo
// that its neighbours compute as well.  A lane holds kTileP points of an
// axis-0 column in registers with their rho; a sweep reads the in-plane
// neighbours and the column's ends from one LDS copy and leaves its values
// in the other, with one barrier.  After sweep s the s outermost layers are
// not those of the grid (the first ones read the guard planes and the next
// row's ends), so the inner points hold the sweeps' exact values, term for
// term those of the stencil with the relaxation epilogue.  Points past a
// zero boundary stay zero, periodic images are computed as such.
// Bound by what a launch and its loads cost (4.7 us), then about 1 us a
// sweep: four sweeps of 24^3 or 48^3 take 8.0 and 8.8 us, 20 to 24 in four
// launches; two of 96^3 12.4, 14.4 in two.  The neighbours along axis 2 by
// lane shifts, waves and planes left out once they lie in the halo, and 8
// points a lane changed nothing or cost 5 %.

constexpr int kTileE = 16;
constexpr int kTileP = 4;
constexpr int kTileThreads = kTileE * kTileE * kTileE / kTileP;
constexpr int kTileSweeps = 4;
// Tiles of a launch: two a CU (their LDS).  Above, a sweep of its own is
// bound by the traffic, which the halos would multiply.
constexpr long kTileLimit = 512;

struct TileDims {
    int n[3], pbc[3];
    int core, sweeps;
    double c0, c[3][2], w;
};

__global__ __launch_bounds__(kTileThreads) void jacobi_tile_kernel(
    const double* __restrict__ in,   // NULL: zeros
    const double* __restrict__ src, double* __restrict__ out, TileDims d)
{
    constexpr int E = kTileE, P = kTileP, E2 = E * E;
    constexpr int kPlanes = (E + 2) * E2;   // a guard plane on either side
    __shared__ double lds[2 * kPlanes];

    const int t1 = (d.n[1] + d.core - 1) / d.core, t2 = (d.n[2] + d.core - 1) / d.core;
    const int b2 = blockIdx.x % t2, b1 = blockIdx.x / t2 % t1, b0 = blockIdx.x / t2 / t1;
    const int p2 = threadIdx.x % E, p1 = threadIdx.x / E % E, p0 = threadIdx.x / E2 * P;
    const int g0 = b0 * d.core - d.sweeps + p0, g1 = b1 * d.core - d.sweeps + p1;
    const int g2 = b2 * d.core - d.sweeps + p2;
    // a halo can be wider than the grid
    auto wrap = [](int i, int n, int pbc) {
        if (!pbc) return i < n ? i : -1;
        while (i < 0) i += n;
        while (i >= n) i -= n;
        return i;
    };
    const int j1 = wrap(g1, d.n[1], d.pbc[1]), j2 = wrap(g2, d.n[2], d.pbc[2]);
    double f[P], r[P];
    bool ok[P];
#pragma unroll
    for (int k = 0; k < P; k++) {
        const int j0 = wrap(g0 + k, d.n[0], d.pbc[0]);
        ok[k] = j0 >= 0 && j1 >= 0 && j2 >= 0;
        const long q = ok[k] ? ((long)j0 * d.n[1] + j1) * d.n[2] + j2 : 0;
        f[k] = in ? in[q] : 0.0;
        r[k] = src[q];
    }
    const int own = (p0 + 1) * E2 + p1 * E + p2;
#pragma unroll
    for (int k = 0; k < P; k++) {
        if (!ok[k]) f[k] = 0.0;
        lds[own + k * E2] = f[k];
    }
    const double u = 1.0 - d.w;
    for (int s = 0; s < d.sweeps; s++) {
        __syncthreads();
        const double* l = lds + (s & 1) * kPlanes + own;
        double* o = lds + (~s & 1) * kPlanes + own;
        double before = l[-E2];
        const double after = l[P * E2];
#pragma unroll
        for (int k = 0; k < P; k++) {
            const double next = k + 1 < P ? f[k + 1 < P ? k + 1 : k] : after;
            // axis 2, 1, 0, each +1 then -1
            const double* m = l + k * E2;
            double a = madd<double>(0.0, m[1], d.c[2][0]);
            a = madd<double>(a, m[-1], d.c[2][1]);
            a = madd<double>(a, m[E], d.c[1][0]);
            a = madd<double>(a, m[-E], d.c[1][1]);
            a = madd<double>(a, next, d.c[0][0]);
            a = madd<double>(a, before, d.c[0][1]);
            before = f[k];
            const double x1 = u * f[k];
            const double x2 = (d.w * (r[k] - a)) / d.c0;
            f[k] = ok[k] ? x1 + x2 : 0.0;
        }
        if (s + 1 < d.sweeps) {
#pragma unroll
            for (int k = 0; k < P; k++) o[k * E2] = f[k];
        }
    }
    auto inner = [&](int p, int g, int n) {
        return p >= d.sweeps && p < d.sweeps + d.core && g < n;
    };
    if (!inner(p1, g1, d.n[1]) || !inner(p2, g2, d.n[2])) return;
#pragma unroll
    for (int k = 0; k < P; k++)
        if (inner(p0 + k, g0 + k, d.n[0]))
            out[((long)(g0 + k) * d.n[1] + g1) * d.n[2] + g2] = f[k];
}

struct VCycle {
    int levels;
    gpd_operator* const* ops;
    gpd_transformer* const* restrictors;
    gpd_transformer* const* interpolators;
    double* const* phis;
    double* const* rhos;
    double* const* residuals;
    const int* presmooths;
    const int* postsmooths;
    const double* weights;
    int relax_method;
    hipStream_t st;
    int bottom;                // first level of bottom_args, or levels + 1
    BottomArgs bottom_args;
};

static long grid_points(const gpd_operator* op)
{
    return (long)op->n[0] * op->n[1] * op->n[2];
}

// Second-order stencils along the axes, Jacobi
static bool short_stencil(const VCycle& v, int level)
{
    return v.relax_method == 2 && fd_epilogue_fused<double>(v.ops[level]) &&
           v.ops[level]->range == 1;
}

// The levels below the first that poisson_bottom_kernel can take: second-
// order stencils along the axes, their transfers, Jacobi.
static void find_bottom(VCycle& v)
{
    v.bottom = v.levels + 1;
    size_t bytes = 0;
    for (int l = v.levels; l >= 1 && v.levels - l < kBottomLevels; l--) {
        const gpd_operator* op = v.ops[l];
        bool ok = short_stencil(v, l) && v.presmooths[l] >= 0 && v.postsmooths[l] >= 0;
        for (int c = 0; c < 3 && l < v.levels; c++) {
            const gpd_transformer *r = v.restrictors[l], *i = v.interpolators[l];
            ok = ok && r->k == 2 && !r->interpolate && r->n_in[c] == op->n[c] &&
                 r->n_out[c] == v.ops[l + 1]->n[c] && r->pbc[c] == op->pbc[c];
            ok = ok && i->k == 2 && i->interpolate && i->n_out[c] == op->n[c] &&
                 i->n_in[c] == v.ops[l + 1]->n[c] && i->pbc[c] == v.ops[l + 1]->pbc[c];
        }
        bytes += 3 * sizeof(double) * grid_points(op);
        if (!ok || bytes > kBottomBytes) break;
        v.bottom = l;
    }
    v.bottom_args = {};
    int off = 0;
    for (int l = v.bottom; l <= v.levels; l++) {
        BottomLevel& b = v.bottom_args.l[v.bottom_args.count++];
        const gpd_operator* op = v.ops[l];
        for (int c = 0; c < 3; c++) {
            b.n[c] = op->n[c];
            b.pbc[c] = op->pbc[c];
            // canonical blocks come axis 2 first
            for (int j = 0; j < 2; j++) b.c[c][j] = op->canon_c[2 - c][j];
        }
        b.inv1 = 1.0f / op->n[1];
        b.inv2 = 1.0f / op->n[2];
        b.off = off;
        off += (int)(3 * grid_points(op));
        b.pre = v.presmooths[l];
        b.post = v.postsmooths[l];
        b.c0 = op->canon_c0;
        b.w = v.weights[l];
        if (l < v.levels) {
            b.down = make_dims(v.restrictors[l]);
            b.up = make_dims(v.interpolators[l]);
        }
    }
}

static int run_bottom(const VCycle& v)
{
    size_t bytes = 0;
    for (int l = v.bottom; l <= v.levels; l++) bytes += 3 * sizeof(double) * grid_points(v.ops[l]);
    // the process's attribute, always the same: another thread's call may come
    // between this and the launch
    hipError_t e = hipFuncSetAttribute((const void*)poisson_bottom_kernel,
                                       hipFuncAttributeMaxDynamicSharedMemorySize,
                                       (int)kBottomBytes);
    if (e != hipSuccess) {
        set_last_error(hipGetErrorString(e));
        return GPD_ERR_HIP;
    }
    hipLaunchKernelGGL(poisson_bottom_kernel, dim3(1), dim3(kBottomThreads), bytes, v.st,
                       v.bottom_args, v.rhos[v.bottom], v.phis[v.bottom]);
    return last_error_to_status(hipGetLastError());
}

// res = op phi - rho
static int residual(const VCycle& v, int level)
{
    FdEpilogue<double> ep = {};
    ep.aux = v.rhos[level];
    return fd_apply_typed<double>(v.ops[level], EPI_SUB, 1, v.phis[level], v.residuals[level], ep,
                                  v.st);
}

static long tiles(const gpd_operator* op, int sweeps)
{
    long t = 1;
    for (int c = 0; c < 3; c++) {
        const int core = kTileE - 2 * sweeps;
        t *= (op->n[c] + core - 1) / core;
    }
    return t;
}

// How many of the level's sweeps jacobi_tile_kernel takes in a launch; 0:
// none, one launch of the stencil kernel each.
static int sweeps_per_launch(const VCycle& v, int level)
{
    if (!short_stencil(v, level)) return 0;
    for (int k = kTileSweeps; k > 1; k--)
        if (tiles(v.ops[level], k) <= kTileLimit) return k;
    return 0;
}

static int launch_tiles(const VCycle& v, int level, int sweeps, const double* in, double* out)
{
    const gpd_operator* op = v.ops[level];
    TileDims d;
    for (int c = 0; c < 3; c++) {
        d.n[c] = op->n[c];
        d.pbc[c] = op->pbc[c];
        // canonical blocks come axis 2 first
        for (int j = 0; j < 2; j++) d.c[c][j] = op->canon_c[2 - c][j];
    }
    d.core = kTileE - 2 * sweeps;
    d.sweeps = sweeps;
    d.c0 = op->canon_c0;
    d.w = v.weights[level];
    hipLaunchKernelGGL(jacobi_tile_kernel, dim3((unsigned)tiles(op, sweeps)), dim3(kTileThreads),
                       0, v.st, in, v.rhos[level], out, d);
    return last_error_to_status(hipGetLastError());
}

// Relaxation by tiles from `from` (NULL: zeros; phi or res) in `launches`
// launches, the last of which writes phi.
static int relax_tiles(const VCycle& v, int level, int sweeps, int launches, const double* from)
{
    double *phi = v.phis[level], *res = v.residuals[level];
    int rc = GPD_OK;
    for (int k = launches; k > 0 && rc == GPD_OK; k--) {
        const int now = (sweeps + k - 1) / k;
        double* to = k % 2 ? phi : res;
        rc = launch_tiles(v, level, now, from, to);
        from = to;
        sweeps -= now;
    }
    return rc;
}

// The array that a level's sweeps may alternate with: its residual, which the
// coarsest level has no use for otherwise and a caller need not keep for it.
static double* second_array(const VCycle& v, int level)
{
    return level < v.levels || level == 0 ? v.residuals[level] : nullptr;
}

// Launches of `sweeps` Jacobi sweeps of the level, alternating between phi
// and its second array.
static int relax_launches(const VCycle& v, int level, int sweeps)
{
    const int m = sweeps_per_launch(v, level);
    return m ? (sweeps + m - 1) / m : sweeps;
}

// Relaxation from the array `from` (phi or the second array) to phi; an odd
// number of launches that starts in phi, or one without a second array, is
// left to gpd_operator_relax and its copy (as are the calls it refuses).
static int relax(const VCycle& v, int level, int sweeps, double* from)
{
    double *phi = v.phis[level], *other = second_array(v, level);
    if (other && sweeps > 0 && sweeps_per_launch(v, level)) {
        int launches = relax_launches(v, level, sweeps);
        if (from == phi && launches % 2) launches++;
        if (launches < sweeps) return relax_tiles(v, level, sweeps, launches, from);
    }
    const std::vector<int>& off = v.ops[level]->off;
    const bool centre_first = off[0] == 0 && off[1] == 0 && off[2] == 0;
    if (v.relax_method != 2 || sweeps < 0 || !centre_first ||
        (from == phi && (sweeps % 2 || !other)))
        return gpd_operator_relax(v.ops[level], GPD_F64, v.relax_method, 1, phi, v.rhos[level],
                                  sweeps, v.weights[level], v.st);
    return fd_jacobi_sweeps<double>(v.ops[level], 1, &from, from == phi ? other : phi,
                                    v.rhos[level], sweeps, v.weights[level], v.st);
}

// The first relaxation of a level below 0, where phi starts from zero
static int relax_zero(const VCycle& v, int level, int sweeps)
{
    if (sweeps > 0 && sweeps_per_launch(v, level)) {
        const int launches = relax_launches(v, level, sweeps);
        if (launches == 1 || second_array(v, level))
            return relax_tiles(v, level, sweeps, launches, nullptr);
    }
    const long n = grid_points(v.ops[level]);
    hipLaunchKernelGGL(fill_zero_f64_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, v.st,
                       v.phis[level], n);
    const int rc = last_error_to_status(hipGetLastError());
    return rc ? rc : relax(v, level, sweeps, v.phis[level]);
}

// gpaw/poisson.py:278-303 for `level`, whose phi is zero at the start below
// level 0; the level-0 residual and its norm are the caller's
static int vcycle_level(const VCycle& v, int level)
{
    double* phi = v.phis[level];
    double* res = v.residuals[level];
    const int post = v.postsmooths[level];
    const int first = level == v.levels ? post : v.presmooths[level];
    int rc = level ? relax_zero(v, level, first) : relax(v, level, first, phi);
    if (level == v.levels) return rc;
    if (!rc) rc = residual(v, level);
    if (!rc)
        rc = transformer_apply_typed<double>(v.restrictors[level], TEPI_PLAIN, false, 1, res,
                                             v.rhos[level + 1], nullptr, 0.0, v.st);
    if (rc) return rc;
    rc = level + 1 == v.bottom ? run_bottom(v) : vcycle_level(v, level + 1);
    if (rc) return rc;
    // phi -= interpolated correction; before an odd number of Jacobi launches
    // into res, so that the last one ends in phi
    double* to = v.relax_method == 2 && post > 0 && relax_launches(v, level, post) % 2 ? res : phi;
    rc = transformer_apply_typed<double>(v.interpolators[level], TEPI_SUBTRACT_FROM, false, 1,
                                         v.phis[level + 1], to, phi, 0.0, v.st);
    if (rc) return rc;
    return relax(v, level, post, to);
}

}  // namespace gpd

using namespace gpd;

extern "C" int gpd_poisson_vcycle(int levels, gpd_operator* const* ops,
                                  gpd_transformer* const* restrictors,
                                  gpd_transformer* const* interpolators, double* const* phis,
                                  double* const* rhos, double* const* residuals,
                                  const int* presmooths, const int* postsmooths,
                                  const double* weights, int relax_method, double dv,
                                  const double* d_minus_one, double* d_norm, void* stream)
{
    GPD_REQUIRE(levels >= 0 && levels <= 16, GPD_ERR_ARG, "bad number of levels");
    GPD_REQUIRE(ops && phis && rhos && residuals && presmooths && postsmooths && weights &&
                    d_minus_one && d_norm,
                GPD_ERR_ARG, "null argument");
    GPD_REQUIRE(levels == 0 || (restrictors && interpolators), GPD_ERR_ARG,
                "null transformer list");
    for (int l = 0; l <= levels; l++) {
        GPD_REQUIRE(ops[l] && phis[l] && rhos[l] && residuals[l], GPD_ERR_ARG,
                    "null operator or grid");
        GPD_REQUIRE(phis[l] != rhos[l], GPD_ERR_ARG, "phi and rho must be distinct");
        if (l < levels || l == 0)
            GPD_REQUIRE(residuals[l] != phis[l] && residuals[l] != rhos[l], GPD_ERR_ARG,
                        "phi, rho and residual must be distinct");
        if (l < levels) {
            GPD_REQUIRE(restrictors[l] && interpolators[l], GPD_ERR_ARG, "null transformer");
            GPD_REQUIRE(residuals[l] != rhos[l + 1] && phis[l + 1] != residuals[l] &&
                            phis[l + 1] != phis[l],
                        GPD_ERR_ARG, "the levels' grids must be distinct");
        }
    }
    VCycle v{levels,     ops,         restrictors, interpolators, phis,
             rhos,       residuals,   presmooths,  postsmooths,   weights,
             relax_method, (hipStream_t)stream, 0, {}};
    find_bottom(v);
    int rc = vcycle_level(v, 0);
    if (rc) return rc;
    // gpaw/poisson.py:304-311: the level-0 residual and dv * sum(r^2)
    rc = residual(v, 0);
    if (rc) return rc;
    const long nG = grid_points(ops[0]);
    return gpd_dots(GPD_F64, 1, nG, dv, residuals[0], residuals[0], d_norm, v.st);
}
