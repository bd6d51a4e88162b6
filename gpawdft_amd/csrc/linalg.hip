// Dense FP64 linear algebra of the subspace step, on the GPU (gfx950).
//
// inverse_cholesky (replaces c/lapack.c:324-370, dpotrf("U") + dtrtri on
// the C-ordered matrix): S = L L^T from the lower triangle of S, then
// S <- L^-1 (lower), upper triangle zeroed.  info = k > 0 when the leading
// minor of order k is not positive definite (S is then left partly
// factored, as LAPACK does).  Blocked by 64 x 64 tiles: each diagonal
// tile is factored and inverted in LDS by one workgroup, the panel and
// trailing updates and the tiles of the inverse run one workgroup per
// tile.
//
// diagonalize (replaces c/lapack.c:129-160, dsyev("V", "U") on the C view,
// i.e. the lower triangle; zheev for complex matrices): cyclic two-sided
// Jacobi.  Up to 64 rows one workgroup runs all sweeps in LDS.  Larger
// matrices are cut into blocks of 32; a round pairs the blocks as a
// tournament, one workgroup per pair annihilates the pair's elements in LDS
// and the matrix and the eigenvectors are updated by 64 x 64 products with
// the accumulated rotations.  Sweeps repeat until the off-diagonal norm is
// below 3e-15 sqrt(n) of the Frobenius norm.  Eigenvalues ascending in w,
// eigenvectors in the rows of A.
#include <cmath>
#include <vector>

#include "common.hpp"

namespace gpd {

// ------------------------------------------------------------------ //
// Element arithmetic of the dense kernels: FP64 real, or complex128
// (double2) with the conjugations of the Hermitian algorithms.
template <typename T> struct El;
template <> struct El<double> {
    __device__ static double zero() { return 0.0; }
    __device__ static double mul(double a, double b) { return a * b; }
    __device__ static double mulc(double a, double b) { return a * b; }   // a conj(b)
    __device__ static double add(double a, double b) { return a + b; }
    __device__ static double sub(double a, double b) { return a - b; }
    __device__ static double neg(double a) { return -a; }
    __device__ static double re(double a) { return a; }
    __device__ static double div(double a, double r) { return a / r; }
    __device__ static double real(double r) { return r; }
};
template <> struct El<double2> {
    __device__ static double2 zero() { return make_double2(0.0, 0.0); }
    __device__ static double2 mul(double2 a, double2 b)
    {
        return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
    }
    __device__ static double2 mulc(double2 a, double2 b)
    {
        return make_double2(a.x * b.x + a.y * b.y, a.y * b.x - a.x * b.y);
    }
    __device__ static double2 add(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
    __device__ static double2 sub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
    __device__ static double2 neg(double2 a) { return make_double2(-a.x, -a.y); }
    __device__ static double re(double2 a) { return a.x; }
    __device__ static double2 div(double2 a, double r) { return make_double2(a.x / r, a.y / r); }
    __device__ static double2 real(double r) { return make_double2(r, 0.0); }
};

// ------------------------------------------------------------------ //
// Cholesky + inverse, blocked by kCB x kCB tiles (right-looking), for
// S = L L^T (real) or S = L L^H (complex):
//   for each diagonal tile k: factor it in LDS and invert its factor
//   (chol_diag_kernel); L_ik = A_ik L_kk^-H for the tiles below it
//   (chol_panel_kernel); A_ij -= L_ik L_jk^H for the trailing tiles
//   (chol_update_kernel).  Then X = L^-1 tile row by tile row:
//   X_ij = -L_ii^-1 sum_{k=j}^{i-1} L_ik X_kj (chol_inverse_kernel).
// Every launch after a failed diagonal tile returns at once, so A keeps
// the partial factorisation and info the failing order.
constexpr int kCB = 64;

__device__ __forceinline__ int tile_rows(int n, int t) { return min(kCB, n - t * kCB); }

// broadcast of a lane's value (lane uniform)
__device__ __forceinline__ double lane_value(double v, int lane)
{
    return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), lane),
                            __builtin_amdgcn_readlane(__double2loint(v), lane));
}
__device__ __forceinline__ double2 lane_value(double2 v, int lane)
{
    return make_double2(lane_value(v.x, lane), lane_value(v.y, lane));
}

// Diagonal tile: the elimination of [S | 1] by panels of kCP columns.  One
// wave factors a panel with a row per lane in registers (the pivots pass by
// lane broadcast, no barrier between columns) while the other three apply
// the panel before it to the right-hand side; then all update the trailing
// columns, and one wave solves the panel's rows of the right-hand side,
// which ends as L^-1.  What is left is the chain of 64 square roots and
// divisions.  (Column by column with three barriers each, then a forward
// substitution by one thread a column: 184 us a tile, 35 now.)
constexpr int kCP = 8;

template <typename T>
__global__ __launch_bounds__(256) void chol_diag_kernel(T* __restrict__ A, int n, int kb,
                                                        T* __restrict__ Dinv,
                                                        int* __restrict__ info)
{
    typedef El<T> E;
    if (*info) return;
    __shared__ T L[kCB][kCB + 1];
    __shared__ T X[kCB][kCB + 1];
    __shared__ int fail;
    const int tid = threadIdx.x;
    const int wave = tid / 64, lane = tid % 64;
    const int k0 = kb * kCB, nb = tile_rows(n, kb);
    // Hermitian input: only the lower triangle is read; rows past the last
    // are those of the unit matrix
    for (int idx = tid; idx < kCB * kCB; idx += 256) {
        const int i = idx / kCB, j = idx % kCB;
        const bool in = i < nb && j <= i;
        const T v = A[in ? (long)(k0 + i) * n + k0 + j : (long)k0 * n + k0];
        L[i][j] = in ? v : (i == j ? E::real(1.0) : E::zero());
        X[i][j] = i == j ? E::real(1.0) : E::zero();
    }
    if (tid == 0) fail = 0;
    __syncthreads();
    // panel p of L: one wave, row `lane`
    auto factor = [&](int p) {
        const int c0 = p * kCP;
        T a[kCP];
#pragma unroll
        for (int k = 0; k < kCP; k++) a[k] = L[lane][c0 + k];
#pragma unroll
        for (int k = 0; k < kCP; k++) {
            const double d = E::re(lane_value(a[k], c0 + k));
            if (!(d > 0.0)) {                 // uniform
                if (lane == 0) fail = k0 + c0 + k + 1;
                break;
            }
            const double l = sqrt(d);
            if (lane == c0 + k) a[k] = E::real(l);
            if (lane > c0 + k) a[k] = E::div(a[k], l);
#pragma unroll
            for (int j = k + 1; j < kCP; j++) {
                const T ljk = lane_value(a[k], c0 + j);
                if (lane >= c0 + j) a[j] = E::sub(a[j], E::mulc(a[k], ljk));
            }
        }
        if (lane >= c0)
#pragma unroll
            for (int k = 0; k < kCP; k++)
                if (lane >= c0 + k) L[lane][c0 + k] = a[k];
    };
    // rows below panel p of X, columns up to it: X_i -= L_ip X_p (tid from 64)
    auto apply = [&](int p) {
        const int c0 = p * kCP, c1 = c0 + kCP, j = lane;
        T x[kCP];
#pragma unroll
        for (int k = 0; k < kCP; k++) x[k] = X[c0 + k][j];
        if (j < c1)
            for (int i = c1 + wave - 1; i < kCB; i += 3) {
                T v = X[i][j];
#pragma unroll
                for (int k = 0; k < kCP; k++) v = E::sub(v, E::mul(L[i][c0 + k], x[k]));
                X[i][j] = v;
            }
    };
    if (wave == 0) factor(0);
    __syncthreads();
    for (int p = 0; p < kCB / kCP && !fail; p++) {
        const int c0 = p * kCP, c1 = c0 + kCP;
        // rows of the panel in X: X_p <- L_pp^-1 X_p, a column per lane
        if (wave == 3) {
            T x[kCP];
#pragma unroll
            for (int k = 0; k < kCP; k++) {
                T v = X[c0 + k][lane];
#pragma unroll
                for (int m = 0; m < k; m++) v = E::sub(v, E::mul(L[c0 + k][c0 + m], x[m]));
                x[k] = E::div(v, E::re(L[c0 + k][c0 + k]));
                X[c0 + k][lane] = x[k];
            }
        }
        // trailing columns: L_ij -= L_ip L_jp^H, j >= c1
        const int tr = tid / 16, tc = tid % 16;
        for (int i = c1 + tr; i < kCB; i += 16) {
            T li[kCP];
#pragma unroll
            for (int k = 0; k < kCP; k++) li[k] = L[i][c0 + k];
            for (int j = c1 + tc; j <= i; j += 16) {
                T v = L[i][j];
#pragma unroll
                for (int k = 0; k < kCP; k++) v = E::sub(v, E::mulc(li[k], L[j][c0 + k]));
                L[i][j] = v;
            }
        }
        __syncthreads();
        if (wave == 0) {
            if (p + 1 < kCB / kCP) factor(p + 1);
        } else {
            apply(p);
        }
        __syncthreads();
    }
    T* D = Dinv + (long)kb * kCB * kCB;
    for (int idx = tid; idx < kCB * kCB; idx += 256) {
        const int i = idx / kCB, j = idx % kCB;
        if (!fail) D[idx] = (i < nb && j <= i) ? X[i][j] : E::zero();
        if (i < nb && j <= i) A[(long)(k0 + i) * n + k0 + j] = L[i][j];
    }
    if (fail && tid == 0) *info = fail;
}

// 64 x 64 product of two tiles in LDS, 4 x 4 elements a thread: rows of P
// against rows of Q conjugated (NT), or against columns of Q
template <typename T, bool NT>
__device__ __forceinline__ void tile_product(const T (&P)[kCB][kCB + 1], const T (&Q)[kCB][kCB + 1],
                                             int m, T (&acc)[4][4])
{
    typedef El<T> E;
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
    for (int k = 0; k < m; k++) {
        T a[4], b[4];
#pragma unroll
        for (int u = 0; u < 4; u++) {
            a[u] = P[tr + 16 * u][k];
            b[u] = NT ? Q[tc + 16 * u][k] : Q[k][tc + 16 * u];
        }
#pragma unroll
        for (int u = 0; u < 4; u++)
#pragma unroll
            for (int v = 0; v < 4; v++)
                acc[u][v] = E::add(acc[u][v], NT ? E::mulc(a[u], b[v]) : E::mul(a[u], b[v]));
    }
}

template <typename T> __device__ __forceinline__ void tile_zero(T (&acc)[4][4])
{
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) acc[u][v] = El<T>::zero();
}

// L_ik = A_ik L_kk^-H: one workgroup per tile below the diagonal tile kb
// (the inverse's upper triangle is zero)
template <typename T>
__global__ __launch_bounds__(256) void chol_panel_kernel(T* __restrict__ A, int n, int kb,
                                                         const T* __restrict__ Dinv,
                                                         const int* __restrict__ info)
{
    typedef El<T> E;
    if (*info) return;
    __shared__ T Ai[kCB][kCB + 1];
    __shared__ T Di[kCB][kCB + 1];
    const int ib = kb + 1 + blockIdx.x;
    const int i0 = ib * kCB, k0 = kb * kCB;
    const int ni = tile_rows(n, ib), nk = tile_rows(n, kb);
    const T* D = Dinv + (long)kb * kCB * kCB;
    for (int idx = threadIdx.x; idx < kCB * kCB; idx += blockDim.x) {
        const int r = idx / kCB, c = idx % kCB;
        Ai[r][c] = (r < ni && c < nk) ? A[(long)(i0 + r) * n + k0 + c] : E::zero();
        Di[r][c] = D[idx];
    }
    __syncthreads();
    T acc[4][4];
    tile_zero(acc);
    tile_product<T, true>(Ai, Di, nk, acc);
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = tr + 16 * u, c = tc + 16 * v;
            if (r < ni && c < nk) A[(long)(i0 + r) * n + k0 + c] = acc[u][v];
        }
}

// A_ij -= L_ik L_jk^H for the trailing tiles i >= j > kb (one workgroup per
// tile pair; 4 x 4 outputs per thread)
template <typename T>
__global__ __launch_bounds__(256) void chol_update_kernel(T* __restrict__ A, int n, int kb,
                                                          const int* __restrict__ info)
{
    typedef El<T> E;
    if (*info) return;
    __shared__ T Li[kCB][kCB + 1];
    __shared__ T Lj[kCB][kCB + 1];
    int t = blockIdx.x, ib = kb + 1;
    while (t >= ib - kb) {       // pairs (ib, jb), kb < jb <= ib, row by row
        t -= ib - kb;
        ib++;
    }
    const int jb = kb + 1 + t;
    const int i0 = ib * kCB, j0 = jb * kCB, k0 = kb * kCB;
    const int ni = tile_rows(n, ib), nj = tile_rows(n, jb), nk = tile_rows(n, kb);
    for (int idx = threadIdx.x; idx < kCB * kCB; idx += blockDim.x) {
        const int r = idx / kCB, c = idx % kCB;
        Li[r][c] = (r < ni && c < nk) ? A[(long)(i0 + r) * n + k0 + c] : E::zero();
        Lj[r][c] = (r < nj && c < nk) ? A[(long)(j0 + r) * n + k0 + c] : E::zero();
    }
    __syncthreads();
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
    T acc[4][4];
    tile_zero(acc);
    tile_product<T, true>(Li, Lj, nk, acc);
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = tr + 16 * u, c = tc + 16 * v;
            if (r < ni && c < nj) {
                T* e = &A[(long)(i0 + r) * n + j0 + c];
                *e = E::sub(*e, acc[u][v]);
            }
        }
}

// tile row ib of X = L^-1: X_ib,jb for jb < ib (one workgroup each) and the
// diagonal tile from Dinv; X rows above ib are final
template <typename T>
__global__ __launch_bounds__(256) void chol_inverse_kernel(const T* __restrict__ A, int n, int ib,
                                                           const T* __restrict__ Dinv,
                                                           T* __restrict__ X,
                                                           const int* __restrict__ info)
{
    typedef El<T> E;
    if (*info) return;
    __shared__ T Lt[kCB][kCB + 1];
    __shared__ T Xt[kCB][kCB + 1];
    const int jb = blockIdx.x;
    const int i0 = ib * kCB, j0 = jb * kCB;
    const int ni = tile_rows(n, ib), nj = tile_rows(n, jb);
    const T* D = Dinv + (long)ib * kCB * kCB;
    if (jb == ib) {
        for (int idx = threadIdx.x; idx < ni * nj; idx += blockDim.x) {
            const int r = idx / nj, c = idx % nj;
            X[(long)(i0 + r) * n + j0 + c] = D[r * kCB + c];
        }
        return;
    }
    const int tr = threadIdx.x / 16, tc = threadIdx.x % 16;
    T acc[4][4];
    tile_zero(acc);
    // T = sum_{kb=jb}^{ib-1} L_ib,kb X_kb,jb
    for (int kb = jb; kb < ib; kb++) {
        const int k0 = kb * kCB, nk = tile_rows(n, kb);
        __syncthreads();
        for (int idx = threadIdx.x; idx < kCB * kCB; idx += blockDim.x) {
            const int r = idx / kCB, c = idx % kCB;
            Lt[r][c] = (r < ni && c < nk) ? A[(long)(i0 + r) * n + k0 + c] : E::zero();
            Xt[r][c] = (r < nk && c < nj) ? X[(long)(k0 + r) * n + j0 + c] : E::zero();
        }
        __syncthreads();
        tile_product<T, false>(Lt, Xt, nk, acc);
    }
    // X_ib,jb = -Dinv_ib T
    __syncthreads();
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) Xt[tr + 16 * u][tc + 16 * v] = acc[u][v];
    for (int idx = threadIdx.x; idx < kCB * kCB; idx += blockDim.x)
        Lt[idx / kCB][idx % kCB] = D[idx];
    __syncthreads();
    tile_zero(acc);
    tile_product<T, false>(Lt, Xt, ni, acc);
#pragma unroll
    for (int u = 0; u < 4; u++)
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const int r = tr + 16 * u, c = tc + 16 * v;
            if (r < ni && c < nj) X[(long)(i0 + r) * n + j0 + c] = E::neg(acc[u][v]);
        }
}

__global__ void chol_init_kernel(int* __restrict__ info) { *info = 0; }

// A = X below and on the diagonal, 0 above
template <typename T>
__global__ void chol_finish_kernel(T* __restrict__ A, const T* __restrict__ X, int n,
                                   const int* __restrict__ info)
{
    if (*info) return;
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)n * n) return;
    const int i = (int)(idx / n), j = (int)(idx % n);
    A[idx] = j <= i ? X[idx] : El<T>::zero();
}

template <typename T>
static int inverse_cholesky_typed(int n, T* d_A, int* info, hipStream_t st)
{
    *info = 0;
    if (n == 0) return GPD_OK;
    const int nt = (n + kCB - 1) / kCB;
    // X (n x n), the inverted diagonal tiles, info
    const size_t nX = (size_t)n * n, nD = (size_t)nt * kCB * kCB;
    T* X = nullptr;
    GPD_CHECK_HIP(hipMallocAsync((void**)&X, sizeof(T) * (nX + nD) + 64, st));
    T* Dinv = X + nX;
    int* dinfo = (int*)(Dinv + nD);
    hipLaunchKernelGGL(chol_init_kernel, dim3(1), dim3(1), 0, st, dinfo);
    int rc = last_error_to_status(hipGetLastError());
    for (int kb = 0; kb < nt && !rc; kb++) {
        hipLaunchKernelGGL(chol_diag_kernel<T>, dim3(1), dim3(256), 0, st, d_A, n, kb, Dinv,
                           dinfo);
        const int below = nt - kb - 1;
        if (below > 0) {
            hipLaunchKernelGGL(chol_panel_kernel<T>, dim3(below), dim3(256), 0, st, d_A, n, kb,
                               (const T*)Dinv, (const int*)dinfo);
            hipLaunchKernelGGL(chol_update_kernel<T>, dim3(below * (below + 1) / 2), dim3(256),
                               0, st, d_A, n, kb, (const int*)dinfo);
        }
        rc = last_error_to_status(hipGetLastError());
    }
    for (int ib = 0; ib < nt && !rc; ib++) {
        hipLaunchKernelGGL(chol_inverse_kernel<T>, dim3(ib + 1), dim3(256), 0, st,
                           (const T*)d_A, n, ib, (const T*)Dinv, X, (const int*)dinfo);
        rc = last_error_to_status(hipGetLastError());
    }
    if (!rc) {
        const long nn = (long)n * n;
        hipLaunchKernelGGL(chol_finish_kernel<T>, dim3((nn + 255) / 256), dim3(256), 0, st, d_A,
                           (const T*)X, n, (const int*)dinfo);
        rc = last_error_to_status(hipGetLastError());
    }
    int hinfo = 0;
    if (!rc) {
        hipError_t e = hipMemcpyAsync(&hinfo, dinfo, sizeof(int), hipMemcpyDeviceToHost, st);
        if (e == hipSuccess) e = hipStreamSynchronize(st);
        if (e != hipSuccess) {
            set_last_error(hipGetErrorString(e));
            rc = GPD_ERR_HIP;
        }
    }
    (void)hipFreeAsync(X, st);
    *info = hinfo;
    return rc;
}

// ------------------------------------------------------------------ //
// Jacobi eigensolver

// round-robin pairing, rounds r = 0 .. n - 2: position 0 fixed, positions
// 1 .. n - 1 rotate
__device__ __forceinline__ int player(int pos, int r, int n)
{
    const int v = pos + r;
    return pos == 0 ? 0 : (v >= n ? v - (n - 1) : v);
}

// 1 / sqrt(x) for normal x: the hardware's estimate (about 2^-26), one
// third-order and one second-order Newton step
__device__ __forceinline__ double rsqrt_newton(double x)
{
    double y = __builtin_amdgcn_rsq(x);
    double e = __builtin_fma(-x * y, y, 1.0);
    y = __builtin_fma(y * e, __builtin_fma(0.375, e, 0.5), y);
    e = __builtin_fma(-x * y, y, 1.0);
    return __builtin_fma(0.5 * y, e, y);
}

// rotation (c, s) that zeroes A[p][q] of the symmetric 2 x 2 block: with
// d = a_qq - a_pp, h = 2 a_pq (scaled by their larger exponent) and
// u = |d| + sqrt(d^2 + h^2), t = +-h / u is the smaller root, so c = u q and
// s = +-h q with q = 1 / sqrt(u^2 + h^2): two reciprocal square roots in the
// chain every round waits for (three divisions and two square roots before)
__device__ __forceinline__ void jacobi_angle(double app, double aqq, double apq, double& c,
                                             double& s, bool& rot)
{
    rot = apq != 0.0 && fabs(apq) > 1e-300 &&
          fabs(apq) > 2.220446049250313e-16 * 1e-3 * __builtin_amdgcn_sqrt(fabs(app * aqq));
    double d = aqq - app, h = 2.0 * apq;
    const int ex = -__builtin_amdgcn_frexp_exp(fmax(fabs(d), fabs(h)));
    d = __builtin_ldexp(d, ex);
    h = __builtin_ldexp(h, ex);
    const double x = __builtin_fma(d, d, h * h);
    const double u = __builtin_fma(x, rsqrt_newton(x), fabs(d));
    const double q = rsqrt_newton(__builtin_fma(u, u, h * h));
    c = rot ? u * q : 1.0;
    s = rot ? (d < 0.0 ? -h : h) * q : 0.0;
}

// Rotation of a pair (p, q): J = diag(1, e) R with e = conj(a_pq) / |a_pq|
// (which makes the 2 x 2 block real; 1 for real matrices) and R the real
// rotation of [[a_pp, |a_pq|], [|a_pq|, a_qq]]: J = [[c, s], [-s e, c e]].
template <typename T> struct Rot;
template <> struct Rot<double> {
    double c, s;
    int rot;
    __device__ void set(double app, double aqq, double apq)
    {
        bool r;
        jacobi_angle(app, aqq, apq, c, s, r);
        rot = r;
    }
    // (x, y) <- (c x - s e y, s x + c e y): columns p, q times J
    __device__ void cols(double& x, double& y) const
    {
        const double u = c * x - s * y;
        y = s * x + c * y;
        x = u;
    }
    // rows p, q: J^H times the pair (real: the same numbers)
    __device__ void rows(double& x, double& y) const { cols(x, y); }
};
template <> struct Rot<double2> {
    double c, s;
    double2 e;
    int rot;
    __device__ void set(double app, double aqq, double2 apq)
    {
        const double m = hypot(apq.x, apq.y);
        bool r;
        jacobi_angle(app, aqq, m, c, s, r);
        rot = r;
        e = r ? make_double2(apq.x / m, -apq.y / m) : make_double2(1.0, 0.0);
    }
    __device__ static double2 lin(double u, double2 a, double w, double2 b)
    {
        return make_double2(u * a.x + w * b.x, u * a.y + w * b.y);
    }
    __device__ void cols(double2& x, double2& y) const
    {
        const double2 ey = El<double2>::mul(e, y);
        y = lin(s, x, c, ey);
        x = lin(c, x, -s, ey);
    }
    __device__ void rows(double2& x, double2& y) const
    {
        const double2 ey = El<double2>::mulc(y, e);      // conj(e) y
        y = lin(s, x, c, ey);
        x = lin(c, x, -s, ey);
    }
};
__device__ __forceinline__ double el_real_diag(double a) { return a; }
__device__ __forceinline__ double2 el_real_diag(double2 a) { return make_double2(a.x, 0.0); }
__device__ __forceinline__ double el_conj(double a) { return a; }
__device__ __forceinline__ double2 el_conj(double2 a) { return make_double2(a.x, -a.y); }
__device__ __forceinline__ double el_norm(double a) { return a * a; }
__device__ __forceinline__ double el_norm(double2 a) { return a.x * a.x + a.y * a.y; }

constexpr int kJB = 64;          // rows of a subproblem
constexpr int kJT = 1024;        // threads

template <typename T> struct JacobiLds {
    T B[kJB][kJB + 1];           // the matrix (and scratch of the updates)
    T U[kJB][kJB + 1];           // J^H accumulated: row i is conj(column i of J) (and scratch)
    Rot<T> rot[2][kJB / 2];
    double red[2][kJT / 64];
};

// element (i, j) of the matrix, of which LDS holds the upper triangle
__device__ __forceinline__ double conj_if(bool c, double a) { return a; }
__device__ __forceinline__ double2 conj_if(bool c, double2 a)
{
    return make_double2(a.x, c ? -a.y : a.y);
}
template <typename T> __device__ __forceinline__ T tri_get(const JacobiLds<T>& l, int i, int j)
{
    return conj_if(i > j, l.B[min(i, j)][max(i, j)]);
}
template <typename T> __device__ __forceinline__ void tri_set(JacobiLds<T>& l, int i, int j, T v)
{
    l.B[min(i, j)][max(i, j)] = conj_if(i > j, v);
}
// thread t's pair of pairs (a, b), a <= b < h (a = -1: none)
__device__ __forceinline__ void tri_item(int t, int h, int& a, int& b)
{
    const int i = t / (h + 1), j = t % (h + 1);
    if (i >= (h + 1) / 2) {
        a = b = -1;
    } else if (j < h - i) {
        a = i;
        b = i + j;
    } else {
        a = 2 * i == h - 1 ? -1 : h - 1 - i;
        b = a + j - (h - i);
    }
}

// One round of h disjoint pairs pq(k) -> (p, q) on the m x m matrix in LDS,
// rotations of round `it` in rot[it & 1]: wave 0 finds the angles while the
// other waves bring U up to the round before (U lags by one round:
// jacobi_flush), then thread (a, b) rotates the 2 x 2 block of pairs a and
// b.  Bound by latencies: the angle's two reciprocal square roots, the LDS
// reads behind each of the two barriers.
template <typename T, typename PQ, typename PQP>
__device__ __forceinline__ void jacobi_lds_round(JacobiLds<T>& l, int it, int h, int m, int a,
                                                 int b, bool lag, PQ pq, PQP pq_prev)
{
    const int t = threadIdx.x, lane = t % 64;
    const int wave = __builtin_amdgcn_readfirstlane(t / 64);
    if (wave == 0) {
        if (lane < h) {
            int p, q;
            pq(lane, p, q);
            Rot<T> r;
            r.set(El<T>::re(l.B[p][p]), El<T>::re(l.B[q][q]), tri_get(l, p, q));
            l.rot[it & 1][lane] = r;
        }
    } else if (lag) {
        for (int k = wave - 1; k < h; k += kJT / 64 - 1) {
            const Rot<T> r = l.rot[(it & 1) ^ 1][k];
            if (lane >= m) continue;
            int p, q;
            pq_prev(k, p, q);
            T x = l.U[p][lane], y = l.U[q][lane];
            r.rows(x, y);
            l.U[p][lane] = x;
            l.U[q][lane] = y;
        }
    }
    __syncthreads();
    if (a >= 0) {
        int pa, qa, pb, qb;
        pq(a, pa, qa);
        pq(b, pb, qb);
        const Rot<T> rb = l.rot[it & 1][b], ra = l.rot[it & 1][a];
        T b00 = tri_get(l, pa, pb), b01 = tri_get(l, pa, qb), b10 = tri_get(l, qa, pb),
          b11 = tri_get(l, qa, qb);
        rb.cols(b00, b01);
        rb.cols(b10, b11);
        ra.rows(b00, b10);
        ra.rows(b01, b11);
        if (a == b) {
            b00 = el_real_diag(b00);
            b11 = el_real_diag(b11);
            if (ra.rot) b01 = b10 = El<T>::zero();
        }
        tri_set(l, pa, pb, b00);
        tri_set(l, pa, qb, b01);
        if (a != b) tri_set(l, qa, pb, b10);
        tri_set(l, qa, qb, b11);
    }
    __syncthreads();
}

template <typename T, typename PQ>
__device__ __forceinline__ void jacobi_flush(JacobiLds<T>& l, int it, int h, int m, PQ pq)
{
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    for (int k = wave; k < h; k += kJT / 64) {
        const Rot<T> r = l.rot[it & 1][k];
        if (lane >= m) continue;
        int p, q;
        pq(k, p, q);
        T x = l.U[p][lane], y = l.U[q][lane];
        r.rows(x, y);
        l.U[p][lane] = x;
        l.U[q][lane] = y;
    }
    __syncthreads();
}

// sums of two values over the workgroup, in a fixed order
template <typename T>
__device__ __forceinline__ void jacobi_sum2(JacobiLds<T>& l, double& o, double& d)
{
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    for (int s = 32; s > 0; s >>= 1) {
        o += __shfl_down(o, s, 64);
        d += __shfl_down(d, s, 64);
    }
    if (lane == 0) {
        l.red[0][wave] = o;
        l.red[1][wave] = d;
    }
    __syncthreads();
    o = d = 0.0;
    for (int w = 0; w < kJT / 64; w++) {
        o += l.red[0][w];
        d += l.red[1][w];
    }
    __syncthreads();
}

constexpr double kJacobiStop = 1e-29;

__device__ __forceinline__ bool jacobi_converged(double off, double diag, int n)
{
    // the off-diagonal norm is at 3e-15 sqrt(n) of the Frobenius norm, a few
    // times the rounding floor (NaN: never)
    return off <= kJacobiStop * n * (off + diag);
}

// n <= 64: the whole eigenproblem in one workgroup (32 bands: 465 launches
// of 2.7 us before, 0.85 ms in all; 0.22 ms now, of 64 rows 1.84 -> 0.59)
template <typename T>
__global__ __launch_bounds__(kJT) void jacobi_small_kernel(T* __restrict__ A, int n,
                                                          double* __restrict__ w,
                                                          int* __restrict__ sweeps)
{
    typedef El<T> E;
    __shared__ JacobiLds<T> l;
    __shared__ double ev[kJB];
    const int t = threadIdx.x;
    const int m = n + (n & 1), h = m / 2;      // padding: an isolated zero eigenvalue
    for (int idx = t; idx < m * m; idx += kJT) {
        const int i = idx / m, j = idx % m;
        T v = E::zero();
        if (i < n && j < n) v = i >= j ? A[(long)i * n + j] : el_conj(A[(long)j * n + i]);
        if (i == j) v = el_real_diag(v);
        l.B[i][j] = v;
        l.U[i][j] = E::real(i == j ? 1.0 : 0.0);
    }
    __syncthreads();
    int ia, ib;
    tri_item(t, h, ia, ib);
    int sweep = 0, it = 0;
    for (; sweep < 40 && m > 1;) {
        for (int r = 0; r < m - 1; r++, it++) {
            auto pq = [&](int k, int& p, int& q) {
                p = player(k, r, m);
                q = player(m - 1 - k, r, m);
            };
            auto prev = [&](int k, int& p, int& q) {
                const int rp = r ? r - 1 : m - 2;
                p = player(k, rp, m);
                q = player(m - 1 - k, rp, m);
            };
            jacobi_lds_round(l, it, h, m, ia, ib, it > 0, pq, prev);
        }
        sweep++;
        double o = 0.0, d = 0.0;
        for (int idx = t; idx < m * m; idx += kJT) {
            const int i = idx / m, j = idx % m;
            const double v = el_norm(l.B[i][j]);
            if (i == j) d += v;
            else if (i < j) o += 2.0 * v;
        }
        jacobi_sum2(l, o, d);
        if (jacobi_converged(o, d, m)) break;
    }
    if (it > 0)
        jacobi_flush(l, it - 1, h, m, [&](int k, int& p, int& q) {
            p = player(k, m - 2, m);
            q = player(m - 1 - k, m - 2, m);
        });
    if (t < n) ev[t] = E::re(l.B[t][t]);
    __syncthreads();
    // ascending (ties by index); row `rank` of A is row i of J^H
    for (int i = t / 64; i < n; i += kJT / 64) {
        const int lane = t % 64;
        const double wi = ev[i];
        const bool before = lane < n && (ev[lane] < wi || (ev[lane] == wi && lane < i));
        const int rank = __popcll(__ballot(before));
        if (lane == 0) w[rank] = wi;
        if (lane < n) A[(long)rank * n + lane] = l.U[i][lane];
    }
    if (t == 0) *sweeps = sweep;
}

// 16 x 16 block (w / 4, w % 4) of a 64 x 64 product by wave w: P Q, or P^H Q
// (CT), on v_mfma_f64_16x16x4 (D: row 4 v + lane / 16, column lane % 16)
typedef double f64x4 __attribute__((ext_vector_type(4)));
template <bool CT>
__device__ __forceinline__ void wave_product(const double (&P)[kJB][kJB + 1],
                                             const double (&Q)[kJB][kJB + 1], double (&out)[4])
{
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, kk = lane / 16;
    const int i = 16 * (wave / 4) + r, j = 16 * (wave % 4) + r;
    f64x4 acc = {0.0, 0.0, 0.0, 0.0};
#pragma unroll 4
    for (int k = kk; k < kJB; k += 4)
        acc = __builtin_amdgcn_mfma_f64_16x16x4f64(CT ? P[k][i] : P[i][k], Q[k][j], acc, 0, 0, 0);
#pragma unroll
    for (int v = 0; v < 4; v++) out[v] = acc[v];
}
template <bool CT>
__device__ __forceinline__ void wave_product(const double2 (&P)[kJB][kJB + 1],
                                             const double2 (&Q)[kJB][kJB + 1], double2 (&out)[4])
{
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64, r = lane % 16, kk = lane / 16;
    const int i = 16 * (wave / 4) + r, j = 16 * (wave % 4) + r;
    f64x4 re = {0.0, 0.0, 0.0, 0.0}, im = re;
#pragma unroll 4
    for (int k = kk; k < kJB; k += 4) {
        double2 a = CT ? P[k][i] : P[i][k];
        const double2 b = Q[k][j];
        if (CT) a.y = -a.y;
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.x, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.x, b.y, im, 0, 0, 0);
        re = __builtin_amdgcn_mfma_f64_16x16x4f64(-a.y, b.y, re, 0, 0, 0);
        im = __builtin_amdgcn_mfma_f64_16x16x4f64(a.y, b.x, im, 0, 0, 0);
    }
#pragma unroll
    for (int v = 0; v < 4; v++) out[v] = make_double2(re[v], im[v]);
}

// element v of a wave's block -> row, column of the 64 x 64 product
__device__ __forceinline__ void wave_element(int v, int& i, int& j)
{
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
    i = 16 * (wave / 4) + 4 * v + lane / 16;
    j = 16 * (wave % 4) + lane % 16;
}

// the blocks of pair a in round r of the tournament of nblk blocks, and the
// pair and side of a block
__device__ __forceinline__ void pair_blocks(int a, int r, int nblk, int& I, int& J)
{
    I = player(a, r, nblk);
    J = player(nblk - 1 - a, r, nblk);
}
__device__ __forceinline__ void block_pair(int I, int r, int nblk, int& a, int& side)
{
    const int pos = I == 0 ? 0 : (I > r ? I - r : I - r + nblk - 1);
    side = pos < nblk / 2 ? 0 : 1;
    a = side ? nblk - 1 - pos : pos;
}

// One launch per round.  With S the matrix before the previous round's
// rotations U (of the pairing `rp`), Bd its rotated diagonal pairs and Vh
// the eigenvectors' conjugate transpose so far:
//  * workgroups [0, ninner): pair `w` of the launch's pairing: its 64 x 64
//    matrix (diagonal blocks from Bd, the cross block by two products), the
//    round's rotations in LDS, U and Bd out for the next launch;
//  * the others bring S and Vh up to the previous round meanwhile: Snew =
//    U_a^H S U_b for a < b (the mirror block conjugated), Bd on the
//    diagonal, Vh <- U_a^H Vh; with norms, each writes its share of the
//    squared off-diagonal and diagonal norms of Snew.
// 512 rows: a sweep is 15 launches of about 47 us (32 rounds in LDS each, 63
// in the first, which also takes the pairs within a block); one launch per
// scalar round was 511 of 6.4 us (30.5 ms in all, 6.7 now).
template <typename T>
__global__ __launch_bounds__(kJT) void jacobi_block_kernel(
    const T* __restrict__ S, T* __restrict__ Snew, T* __restrict__ Vh, int nblk, int r, int rp,
    int ninner, const T* __restrict__ Up, const T* __restrict__ Bp, T* __restrict__ Un,
    T* __restrict__ Bn, double* __restrict__ norms)
{
    typedef El<T> E;
    __shared__ JacobiLds<T> l;
    constexpr int HB = kJB / 2, NN = kJB * kJB;
    const int t = threadIdx.x;
    const int np = nblk / 2;
    const long ld = (long)nblk * HB;
    auto row_of = [&](int I, int J, int i) { return (long)(i < HB ? I : J) * HB + i % HB; };
    int w = blockIdx.x;
    if (w < ninner) {
        int I, J, a, sa, c, sc;
        pair_blocks(w, r, nblk, I, J);
        block_pair(I, rp, nblk, a, sa);
        block_pair(J, rp, nblk, c, sc);
        int aI, aJ, cI, cJ;
        pair_blocks(a, rp, nblk, aI, aJ);
        pair_blocks(c, rp, nblk, cI, cJ);
        // cross block: (U_a^H S U_c) at rows of I, columns of J
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            l.B[i][j] = S[row_of(aI, aJ, i) * ld + row_of(cI, cJ, j)];
            l.U[i][j] = Up[(long)c * NN + idx];
        }
        __syncthreads();
        T x[4];
        wave_product<false>(l.B, l.U, x);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++) {
            int i, j;
            wave_element(v, i, j);
            l.B[i][j] = x[v];
        }
        for (int idx = t; idx < NN; idx += kJT) l.U[idx / kJB][idx % kJB] = Up[(long)a * NN + idx];
        __syncthreads();
        wave_product<true>(l.U, l.B, x);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++) {
            int i, j;
            wave_element(v, i, j);
            if (i / HB == sa && j / HB == sc) {
                l.B[i % HB][HB + j % HB] = x[v];
                l.B[HB + j % HB][i % HB] = el_conj(x[v]);
            }
        }
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            l.U[i][j] = E::real(i == j ? 1.0 : 0.0);
            if (i < HB && j < HB)
                l.B[i][j] = Bp[(long)a * NN + (sa * HB + i) * kJB + sa * HB + j];
            else if (i >= HB && j >= HB)
                l.B[i][j] = Bp[(long)c * NN + (sc * HB + i - HB) * kJB + sc * HB + j - HB];
        }
        __syncthreads();
        int ia, ib;
        tri_item(t, HB, ia, ib);
        if (r == 0) {
            for (int k = 0; k < kJB - 1; k++) {
                auto pq = [&](int u, int& p, int& q) {
                    p = player(u, k, kJB);
                    q = player(kJB - 1 - u, k, kJB);
                };
                auto prev = [&](int u, int& p, int& q) {
                    p = player(u, k - 1, kJB);
                    q = player(kJB - 1 - u, k - 1, kJB);
                };
                jacobi_lds_round(l, k, HB, kJB, ia, ib, k > 0, pq, prev);
            }
            jacobi_flush(l, kJB - 2, HB, kJB, [&](int u, int& p, int& q) {
                p = player(u, kJB - 2, kJB);
                q = player(kJB - 1 - u, kJB - 2, kJB);
            });
        } else {
            for (int k = 0; k < HB; k++) {
                auto pq = [&](int u, int& p, int& q) {
                    p = u;
                    q = HB + (u + k >= HB ? u + k - HB : u + k);
                };
                auto prev = [&](int u, int& p, int& q) {
                    p = u;
                    q = HB + (u + k - 1 >= HB ? u + k - 1 - HB : u + k - 1);
                };
                jacobi_lds_round(l, k, HB, kJB, ia, ib, k > 0, pq, prev);
            }
            jacobi_flush(l, HB - 1, HB, kJB, [&](int u, int& p, int& q) {
                p = u;
                q = HB + (u + HB - 1) % HB;
            });
        }
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            Un[(long)w * NN + idx] = el_conj(l.U[j][i]);     // columns of J
            Bn[(long)w * NN + idx] = tri_get(l, i, j);
        }
        return;
    }
    w -= ninner;
    const int nupper = np * (np - 1) / 2;
    double o = 0.0, d = 0.0;
    if (w < nupper) {
        int a = 0, b = w;                      // pairs (a, b), a < b
        while (b >= np - 1 - a) {
            b -= np - 1 - a;
            a++;
        }
        b += a + 1;
        int aI, aJ, bI, bJ;
        pair_blocks(a, rp, nblk, aI, aJ);
        pair_blocks(b, rp, nblk, bI, bJ);
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            l.B[i][j] = S[row_of(aI, aJ, i) * ld + row_of(bI, bJ, j)];
            l.U[i][j] = Up[(long)b * NN + idx];
        }
        __syncthreads();
        T x[4];
        wave_product<false>(l.B, l.U, x);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++) {
            int i, j;
            wave_element(v, i, j);
            l.B[i][j] = x[v];
        }
        for (int idx = t; idx < NN; idx += kJT) l.U[idx / kJB][idx % kJB] = Up[(long)a * NN + idx];
        __syncthreads();
        wave_product<true>(l.U, l.B, x);
        __syncthreads();
#pragma unroll
        for (int v = 0; v < 4; v++) {
            int i, j;
            wave_element(v, i, j);
            l.B[i][j] = x[v];
            o += 2.0 * el_norm(x[v]);
        }
        __syncthreads();
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            Snew[row_of(aI, aJ, i) * ld + row_of(bI, bJ, j)] = l.B[i][j];
            Snew[row_of(bI, bJ, i) * ld + row_of(aI, aJ, j)] = el_conj(l.B[j][i]);
        }
    } else if (w < nupper + np) {
        const int a = w - nupper;
        int aI, aJ;
        pair_blocks(a, rp, nblk, aI, aJ);
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            const T v = Bp[(long)a * NN + idx];
            Snew[row_of(aI, aJ, i) * ld + row_of(aI, aJ, j)] = v;
            if (i == j) d += el_norm(v);
            else o += el_norm(v);
        }
    } else {
        const int v0 = w - nupper - np, a = v0 % np;
        const long c0 = (long)(v0 / np) * kJB;
        int aI, aJ;
        pair_blocks(a, rp, nblk, aI, aJ);
        for (int idx = t; idx < NN; idx += kJT) {
            const int i = idx / kJB, j = idx % kJB;
            l.B[i][j] = Vh[row_of(aI, aJ, i) * ld + c0 + j];
            l.U[i][j] = Up[(long)a * NN + idx];
        }
        __syncthreads();
        T x[4];
        wave_product<true>(l.U, l.B, x);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            int i, j;
            wave_element(v, i, j);
            Vh[row_of(aI, aJ, i) * ld + c0 + j] = x[v];
        }
        return;
    }
    if (norms) {
        jacobi_sum2(l, o, d);
        if (t == 0) {
            norms[2 * w] = o;
            norms[2 * w + 1] = d;
        }
    }
}

// S and Vh = 1 padded to nblk blocks (padding: isolated zero eigenvalues),
// U = 1 and Bd for the pairing rp
template <typename T>
__global__ void jacobi_init_kernel(const T* __restrict__ A, int n, int nblk, int rp,
                                   T* __restrict__ S, T* __restrict__ Vh, T* __restrict__ U,
                                   T* __restrict__ Bd)
{
    typedef El<T> E;
    const int ld = nblk * (kJB / 2);
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)ld * ld) return;
    const int i = (int)(idx / ld), j = (int)(idx % ld);
    T v = E::zero();
    if (i < n && j < n) v = i >= j ? A[(long)i * n + j] : el_conj(A[(long)j * n + i]);
    if (i == j) v = el_real_diag(v);
    S[idx] = v;
    const T one = E::real(i == j ? 1.0 : 0.0);
    Vh[idx] = one;
    int a, sa, b, sb;
    block_pair(i / (kJB / 2), rp, nblk, a, sa);
    block_pair(j / (kJB / 2), rp, nblk, b, sb);
    if (a == b) {
        const long e = (long)a * kJB * kJB + (sa * (kJB / 2) + i % (kJB / 2)) * kJB +
                       sb * (kJB / 2) + j % (kJB / 2);
        Bd[e] = v;
        U[e] = one;
    }
}

__global__ __launch_bounds__(64) void jacobi_norms_kernel(const double* __restrict__ part, int n,
                                                         double* __restrict__ out)
{
    double o = 0.0, d = 0.0;
    for (int k = threadIdx.x; k < n; k += 64) {
        o += part[2 * k];
        d += part[2 * k + 1];
    }
    for (int s = 32; s > 0; s >>= 1) {
        o += __shfl_down(o, s, 64);
        d += __shfl_down(d, s, 64);
    }
    if (threadIdx.x == 0) {
        out[0] = o;
        out[1] = d;
    }
}

// eigenvalues ascending (ties by index), eigenvectors into rows: one
// workgroup per eigenvalue
template <typename T>
__global__ __launch_bounds__(256) void jacobi_finish_kernel(const T* __restrict__ S,
                                                           const T* __restrict__ Vh, int n,
                                                           int ld, double* __restrict__ w,
                                                           T* __restrict__ A)
{
    __shared__ int before;
    const int i = blockIdx.x;
    if (threadIdx.x == 0) before = 0;
    __syncthreads();
    const double wi = El<T>::re(S[(long)i * ld + i]);
    int rank = 0;
    for (int j = threadIdx.x; j < n; j += 256) {
        const double wj = El<T>::re(S[(long)j * ld + j]);
        if (wj < wi || (wj == wi && j < i)) rank++;
    }
    if (rank) atomicAdd(&before, rank);
    __syncthreads();
    rank = before;
    if (threadIdx.x == 0) w[rank] = wi;
    for (int j = threadIdx.x; j < n; j += 256) A[(long)rank * n + j] = Vh[(long)i * ld + j];
}

static int read_back(void* dst, const void* src, size_t bytes, hipStream_t st)
{
    hipError_t e = hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, st);
    if (e == hipSuccess) e = hipStreamSynchronize(st);
    if (e == hipSuccess) return GPD_OK;
    set_last_error(hipGetErrorString(e));
    return GPD_ERR_HIP;
}

template <typename T>
static int diagonalize_typed(int n, T* d_A, double* d_w, int* sweeps, hipStream_t st)
{
    if (sweeps) *sweeps = 0;
    if (n == 0) return GPD_OK;
    int sweep = 0, rc = GPD_OK;
    if (n <= kJB) {
        int* dsw = nullptr;
        GPD_CHECK_HIP(hipMallocAsync((void**)&dsw, sizeof(int), st));
        hipLaunchKernelGGL(jacobi_small_kernel<T>, dim3(1), dim3(kJT), 0, st, d_A, n, d_w, dsw);
        rc = last_error_to_status(hipGetLastError());
        if (!rc) rc = read_back(&sweep, dsw, sizeof(int), st);
        (void)hipFreeAsync(dsw, st);
        if (sweeps) *sweeps = sweep;
        return rc;
    }
    const int nblk = ((n + kJB - 1) / kJB) * 2, np = nblk / 2;     // blocks of 32, in pairs
    const long ld = (long)nblk * (kJB / 2), NN = ld * ld;
    const long NP = (long)np * kJB * kJB;
    const int nshare = np * (np - 1) / 2 + np, napply = nshare + np * np;
    const size_t bytes = sizeof(T) * (3 * NN + 4 * NP) + sizeof(double) * (2 * nshare + 2);
    T* buf = nullptr;
    GPD_CHECK_HIP(hipMallocAsync((void**)&buf, bytes, st));
    T *S = buf, *Sn = buf + NN, *Vh = buf + 2 * NN;
    T *U = buf + 3 * NN, *Un = U + NP, *B = U + 2 * NP, *Bn = U + 3 * NP;
    double* part = (double*)(U + 4 * NP);
    double* norms = part + 2 * nshare;
    int rp = nblk - 2;
    hipLaunchKernelGGL(jacobi_init_kernel<T>, dim3((NN + 255) / 256), dim3(256), 0, st, d_A, n,
                       nblk, rp, S, Vh, U, B);
    rc = last_error_to_status(hipGetLastError());
    // The launch of a sweep's first round brings S to the end of the sweep
    // before and gives its norms; once those have converged the rotations
    // that launch found are dropped.
    for (; !rc; sweep++) {
        for (int r = 0; r < nblk - 1 && !rc; r++) {
            const bool check = r == 0 && sweep > 0;
            hipLaunchKernelGGL(jacobi_block_kernel<T>, dim3(np + napply), dim3(kJT), 0, st,
                               (const T*)S, Sn, Vh, nblk, r, rp, np, (const T*)U, (const T*)B, Un,
                               Bn, check ? part : nullptr);
            rc = last_error_to_status(hipGetLastError());
            std::swap(S, Sn);
            std::swap(U, Un);
            std::swap(B, Bn);
            rp = r;
            if (check && !rc) {
                double hn[2] = {0, 0};
                hipLaunchKernelGGL(jacobi_norms_kernel, dim3(1), dim3(64), 0, st,
                                   (const double*)part, nshare, norms);
                rc = last_error_to_status(hipGetLastError());
                if (!rc) rc = read_back(hn, norms, sizeof(hn), st);
                if (rc || hn[0] <= kJacobiStop * ld * (hn[0] + hn[1]) || sweep >= 40) goto done;
            }
        }
    }
done:
    if (!rc) {
        hipLaunchKernelGGL(jacobi_finish_kernel<T>, dim3(n), dim3(256), 0, st, (const T*)S,
                           (const T*)Vh, n, (int)ld, d_w, d_A);
        rc = last_error_to_status(hipGetLastError());
    }
    (void)hipFreeAsync(buf, st);
    if (sweeps) *sweeps = sweep;
    return rc;
}

}  // namespace gpd

using namespace gpd;

extern "C" int gpd_inverse_cholesky(int n, double* d_A, int* info, void* stream)
{
    GPD_REQUIRE(n >= 0 && d_A && info, GPD_ERR_ARG, "bad arguments");
    return inverse_cholesky_typed<double>(n, d_A, info, (hipStream_t)stream);
}

extern "C" int gpd_inverse_cholesky_z(int n, double* d_A, int* info, void* stream)
{
    GPD_REQUIRE(n >= 0 && d_A && info, GPD_ERR_ARG, "bad arguments");
    return inverse_cholesky_typed<double2>(n, (double2*)d_A, info, (hipStream_t)stream);
}

extern "C" int gpd_diagonalize(int n, double* d_A, double* d_w, int* sweeps, void* stream)
{
    GPD_REQUIRE(n >= 0 && d_A && d_w, GPD_ERR_ARG, "bad arguments");
    return diagonalize_typed<double>(n, d_A, d_w, sweeps, (hipStream_t)stream);
}

extern "C" int gpd_diagonalize_z(int n, double* d_A, double* d_w, int* sweeps, void* stream)
{
    GPD_REQUIRE(n >= 0 && d_A && d_w, GPD_ERR_ARG, "bad arguments");
    return diagonalize_typed<double2>(n, (double2*)d_A, d_w, sweeps, (hipStream_t)stream);
}
