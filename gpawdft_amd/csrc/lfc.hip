// Localized functions (PAW projectors) on the grid: integrate and add
// (gfx950).
//
// Behaviour follows _gpaw.LFC (c/lfc.c:106-186, 361-425, 724-783) for real
// functions.  The reference sweeps a G-sorted list of boundary events and
// keeps the set of "active" volumes in between (c/lfc.h:38-87).  Here that
// sweep runs once, on the host, when the object is created, and is turned
// into flat device tables:
//  * per covered grid point, the list of (A row, M, nm) in the sweep's
//    active-volume order -- add() walks it point by point, so FP64 sums
//    round exactly as the reference's a_G[G] += A * c loop;
//  * per function block M, the (G, A row) sequence in the sweep's order --
//    the FP64 integrate() walks it sequentially per (band, block), so
//    c_M += (a_G * dv) * A rounds as the reference;
//  * the same sequences grouped by identical point lists with the A values
//    laid out densely -- the FP32 integrate() reads each point once for all
//    functions of an atom and a block of bands, and reduces in LDS.
#include <algorithm>
#include <cstring>
#include <map>
#include <new>
#include <vector>

#include "common.hpp"
#include "lfc.hpp"

namespace gpd {

template <> const double* lfc_values<double>(const gpd_lfc* l) { return l->A64; }
template <> const float* lfc_values<float>(const gpd_lfc* l) { return l->A32; }

constexpr int kNF = 16;   // functions per group held in registers
constexpr int kDepth = 1;  // FP32 integrate: chunks of staged values in flight (1 measured
                           // fastest at 96^3 x 256: 3 cost more in registers than it hid)

// ------------------------------------------------------------------ //
// kernels

// FP32 integrate on MFMA: one workgroup per (group, block of 32 bands).
// Per group, P[b][f] += dv * sum_p x[b][p] A[p][f] is the product of a
// [32 bands x K points] and a [K points x 32 functions] matrix (nf <= 16
// of the 32 columns used).  Chunks of 64 points are staged in LDS as in
// the exact kernel below (kDepth chunks in flight); each
// wave runs v_mfma_f32_32x32x2_f32 over 16 of a chunk's points and flushes
// its accumulator into FP64 registers after every chunk.  The four waves'
// partial products are summed through LDS at the end.
//
// With nseg > 1 a group's point list is split into nseg segments of whole
// chunks, one workgroup each (a sphere is hundreds of chunks, and one
// workgroup per group and band block leaves about one workgroup per CU to
// hide the latency of each chunk's loads).  Each segment then writes its
// dv-scaled sums to part[g][s][band][function] and
// lfc_integrate_segments_kernel adds the segments to c in a fixed order.
__global__ __launch_bounds__(256) void lfc_integrate_mfma_kernel(
    const float* __restrict__ a, float* __restrict__ c, long nG, int Mmax, long nx, double dv,
    int ngroups, int nfmax, const long* __restrict__ grp_off, const int* __restrict__ grp_nf,
    const int* __restrict__ grp_fM, const int* __restrict__ grp_G,
    const float* __restrict__ grp_A, int nseg, float* __restrict__ part)
{
    constexpr int NT = 256, NBB = 32, CH = 64;
    constexpr int LR = NT / CH;            // band rows per load pass
    constexpr int NXL = NBB / LR;          // staged values per thread per chunk
    constexpr int NAL = CH * kNF / NT;     // A values per thread per chunk
    __shared__ float xs[2][CH][NBB + 1];
    __shared__ float As[2][CH * kNF];
    __shared__ float red[4][32][33];

    const long nbb = (nx + NBB - 1) / NBB;
    const long w = xcd_work_index(blockIdx.x, nbb * ngroups * nseg);
    if (w < 0) return;
    const int sg = (int)(w % nseg);          // a group's segments are neighbours
    const int g = (int)((w / nseg) % ngroups);
    const long b0 = (w / nseg / ngroups) * NBB;
    const int nf = grp_nf[g];
    // this workgroup's points: whole chunks of segment sg of the group
    const long ga = grp_off[g], gb = grp_off[g + 1];
    const long nch = (gb - ga + CH - 1) / CH, cps = (nch + nseg - 1) / nseg;
    const long j0 = min(gb, ga + sg * cps * CH), j1 = min(gb, j0 + cps * CH);
    const int t = threadIdx.x;
    const int wave = t / 64, lane = t % 64, l32 = lane % 32, half = lane / 32;

    const int lp = t % CH, lr = t / CH;
    constexpr int D = kDepth;
    float xr[D][NXL], ar[D][NAL];
    int Gs[D];
    auto index = [&](long jc) { return (jc + lp < j1) ? grp_G[jc + lp] : -1; };
    auto load = [&](float* xv, float* av, long jc, int G) {
#pragma unroll
        for (int q = 0; q < NXL; q++) {
            const long b = b0 + lr + LR * q;
            if (G >= 0 && b < nx) xv[q] = a[b * nG + G];
        }
        const long left = j1 - jc;
        const long na = (left < CH ? left : CH) * nfmax;
        const float* Ac = grp_A + jc * nfmax;
#pragma unroll
        for (int q = 0; q < NAL; q++)
            if (t + NT * q < na) av[q] = Ac[t + NT * q];
    };
#pragma unroll
    for (int s = 0; s < D; s++) {
        Gs[s] = index(j0 + s * CH);
        load(xr[s], ar[s], j0 + s * CH, Gs[s]);
    }
    int Gn = index(j0 + D * CH);

    f32x16 acc = {};
    double acc64[16];
#pragma unroll
    for (int v = 0; v < 16; v++) acc64[v] = 0.0;
    int it = 0;
    for (long jb = j0; jb < j1; jb += D * CH) {
#pragma unroll
        for (int s = 0; s < D; s++) {
            const long jc = jb + s * CH;
            if (jc >= j1) break;
            const int buf = it & 1;
            it++;
            const long left = j1 - jc;
            const int np = (int)(left < CH ? left : CH);
#pragma unroll
            for (int q = 0; q < NXL; q++) {
                const long b = b0 + lr + LR * q;
                xs[buf][lp][lr + LR * q] = (Gs[s] >= 0 && b < nx) ? xr[s][q] : 0.f;
            }
#pragma unroll
            for (int q = 0; q < NAL; q++)
                if (t + NT * q < np * nfmax) As[buf][t + NT * q] = ar[s][q];
            lds_barrier();
            if (jc + D * CH < j1) {
                Gs[s] = Gn;
                load(xr[s], ar[s], jc + D * CH, Gn);
                Gn = index(jc + (D + 1) * CH);
            }
            // A operand: lane -> (band l32, point half); B: (point half,
            // function l32)
#pragma unroll
            for (int k2 = 0; k2 < 8; k2++) {
                const int p = 16 * wave + 2 * k2 + half;
                const float av = xs[buf][p][l32];
                const float bv = (p < np && l32 < nf) ? As[buf][p * nfmax + l32] : 0.f;
                acc = __builtin_amdgcn_mfma_f32_32x32x2f32(av, bv, acc, 0, 0, 0);
            }
#pragma unroll
            for (int v = 0; v < 16; v++) {
                acc64[v] += (double)acc[v];
                acc[v] = 0.f;
            }
        }
    }
    // output register v: band row 8 (v / 4) + 4 half + v % 4, function l32
#pragma unroll
    for (int v = 0; v < 16; v++)
        red[wave][8 * (v / 4) + 4 * half + (v % 4)][l32] = (float)(acc64[v] * dv);
    __syncthreads();
    for (int idx = t; idx < 32 * 32; idx += NT) {
        const int row = idx / 32, col = idx % 32;
        const long band = b0 + row;
        if (col < nf && band < nx) {
            const float s = (red[0][row][col] + red[1][row][col]) +
                            (red[2][row][col] + red[3][row][col]);
            if (nseg > 1) {
                part[(((long)g * nseg + sg) * nx + band) * nfmax + col] = s;
            } else {
                float* cp = c + band * Mmax + grp_fM[(long)g * nfmax + col];
                *cp = *cp + s;
            }
        }
    }
}

// c[band][M] += the segments' sums of its group, in segment order (FP64)
__global__ void lfc_integrate_segments_kernel(const float* __restrict__ part,
                                              float* __restrict__ c, int Mmax, long nx,
                                              int ngroups, int nfmax, int nseg,
                                              const int* __restrict__ grp_nf,
                                              const int* __restrict__ grp_fM)
{
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= (long)ngroups * nx * nfmax) return;
    const int col = (int)(idx % nfmax);
    const long band = (idx / nfmax) % nx;
    const int g = (int)(idx / nfmax / nx);
    if (col >= grp_nf[g]) return;
    double s = 0.0;
    for (int sg = 0; sg < nseg; sg++) s += (double)part[(((long)g * nseg + sg) * nx + band) * nfmax + col];
    float* cp = c + band * Mmax + grp_fM[(long)g * nfmax + col];
    *cp = *cp + (float)s;
}

// Grouped add (FP32): one thread per point of a group, NB bands per
// workgroup; all functions of the group are summed, then added once.
// Groups of one launch ("colour") cover disjoint points, so the
// read-modify-writes do not race.  The NB x nf coefficients of the
// workgroup are staged in LDS once; each thread issues its NB loads
// together, then the sums, then the NB stores.
template <int NB, int NF>
__global__ __launch_bounds__(256) void lfc_add_grp_kernel(
    const float* __restrict__ c, float* __restrict__ a, long nG, int Mmax, long nx, int nfmax,
    int nitems, const int* __restrict__ item_g, const long* __restrict__ item_j0,
    const long* __restrict__ grp_off, const int* __restrict__ grp_nf,
    const int* __restrict__ grp_fM, const int* __restrict__ grp_G,
    const float* __restrict__ grp_A)
{
    static_assert(NB * NF <= 256, "one coefficient per thread");
    __shared__ float cs[NB][NF];
    const long nbblk = (nx + NB - 1) / NB;
    const long w = xcd_work_index(blockIdx.x, (long)nitems * nbblk);
    if (w < 0) return;
    const int item = (int)(w % nitems);
    const long b0 = (w / nitems) * NB;
    const int g = item_g[item];
    const int nf = grp_nf[g];
    const int* fM = grp_fM + (long)g * nfmax;
    if ((int)threadIdx.x < NB * NF) {
        const int bb = threadIdx.x / NF, f = threadIdx.x % NF;
        const long b = b0 + bb;
        cs[bb][f] = (f < nf && b < nx) ? c[b * Mmax + fM[f]] : 0.f;
    }
    __syncthreads();
    const long j = item_j0[item] + threadIdx.x;
    if (j >= grp_off[g + 1]) return;
    const long G = grp_G[j];
    const float* Ar = grp_A + j * nfmax;
    float cur[NB];
#pragma unroll
    for (int bb = 0; bb < NB; bb++) {
        const long b = b0 + bb;
        cur[bb] = b < nx ? a[b * nG + G] : 0.f;
    }
    float av[NF];
#pragma unroll
    for (int f = 0; f < NF; f++) av[f] = f < nf ? Ar[f] : 0.f;
#pragma unroll
    for (int bb = 0; bb < NB; bb++) {
        float s = 0.f;
#pragma unroll
        for (int f = 0; f < NF; f++) s = __builtin_fmaf(av[f], cs[bb][f], s);
        cur[bb] = cur[bb] + s;
    }
#pragma unroll
    for (int bb = 0; bb < NB; bb++) {
        const long b = b0 + bb;
        if (b < nx) a[b * nG + G] = cur[bb];
    }
}

// add: one thread per (covered point, NBT bands), entries in sweep order.
// Each A value is loaded once for the NBT bands; every band's sum keeps
// the reference's order.
template <typename T, int NBT>
__global__ void lfc_add_kernel(const T* __restrict__ c, T* __restrict__ a, long nG, int Mmax,
                               long nx, long ncov, const T* __restrict__ A,
                               const int* __restrict__ cov_G, const int* __restrict__ cov_ptr,
                               const int2* __restrict__ ent)
{
    const long nbblk = (nx + NBT - 1) / NBT;
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nbblk * ncov) return;
    const long i = idx % ncov;
    const long b0 = (idx / ncov) * NBT;
    const long G = cov_G[i];
    T v[NBT];
#pragma unroll
    for (int bb = 0; bb < NBT; bb++) v[bb] = b0 + bb < nx ? a[(b0 + bb) * nG + G] : T(0);
    const int e1 = cov_ptr[i + 1];
    for (int e = cov_ptr[i]; e < e1; e++) {
        const int2 en = ent[e];
        const int nm = en.y & 15;
        const T* Ar = A + en.x;
        const int M = en.y >> 4;
        for (int m = 0; m < nm; m++) {
            const T Am = Ar[m];
#pragma unroll
            for (int bb = 0; bb < NBT; bb++) {
                const long b = b0 + bb < nx ? b0 + bb : b0;
                v[bb] = madd<T>(v[bb], Am, c[b * Mmax + M + m]);
            }
        }
    }
#pragma unroll
    for (int bb = 0; bb < NBT; bb++)
        if (b0 + bb < nx) a[(b0 + bb) * nG + G] = v[bb];
}

// add by chunks of consecutive covered points: one workgroup per (chunk,
// block of NB bands), one thread per point.  The coefficients of the
// chunk's functions (at most kAddFuns, the distinct function blocks of its
// points) for the NB bands are staged in LDS once; each thread loads its A
// rows once for the NB bands and walks its entries in the sweep's volume
// order, so in FP64 every band's a_G += A * c chain rounds as the
// reference's (c/lfc.c:743-752).
constexpr int kAddChunk = 256;   // points per chunk (at most)
constexpr int kAddFuns = 256;    // staged functions per chunk (at most)

template <typename T, int NB>
__global__ __launch_bounds__(256) void lfc_add_chunk_kernel(
    const T* __restrict__ c, T* __restrict__ a, long nG, int Mmax, long nx, long nchunks,
    const int* __restrict__ ch_i0, const int* __restrict__ ch_foff,
    const int* __restrict__ ch_col, const T* __restrict__ A, const int* __restrict__ cov_G,
    const int* __restrict__ cov_ptr, const int2* __restrict__ ent,
    const unsigned char* __restrict__ ent_f)
{
    __shared__ T cs[kAddFuns][NB];
    const long nbb = (nx + NB - 1) / NB;
    const long w = xcd_work_index(blockIdx.x, nchunks * nbb);
    if (w < 0) return;
    const long ch = w / nbb;              // a chunk's band blocks share its A rows in L2
    const long b0 = (w % nbb) * NB;
    const int f0 = ch_foff[ch], nf = ch_foff[ch + 1] - f0;
    for (int idx = threadIdx.x; idx < nf * NB; idx += blockDim.x) {
        const int f = idx % nf, b = idx / nf;
        const long band = b0 + b;
        cs[f][b] = band < nx ? c[band * Mmax + ch_col[f0 + f]] : T(0);
    }
    __syncthreads();
    const long i = ch_i0[ch] + threadIdx.x;
    if (i >= ch_i0[ch + 1]) return;
    const long G = cov_G[i];
    T v[NB];
#pragma unroll
    for (int b = 0; b < NB; b++) v[b] = b0 + b < nx ? a[(b0 + b) * nG + G] : T(0);
    // per entry, all of its A values are loaded before the sums (one load
    // latency per entry, not per function); the next entry's table entry
    // is fetched meanwhile
    const int e0 = cov_ptr[i], e1 = cov_ptr[i + 1];
    int2 en = ent[e0];
    int fs = ent_f[e0];
    for (int e = e0; e < e1; e++) {
        const int nm = en.y & 15, cur_fs = fs;
        const T* Ar = A + en.x;
        T Av[kNF - 1];
#pragma unroll
        for (int m = 0; m < kNF - 1; m++)
            if (m < nm) Av[m] = Ar[m];
        if (e + 1 < e1) {
            en = ent[e + 1];
            fs = ent_f[e + 1];
        }
#pragma unroll
        for (int m = 0; m < kNF - 1; m++) {
            if (m >= nm) break;
#pragma unroll
            for (int b = 0; b < NB; b++) v[b] = madd<T>(v[b], Av[m], cs[cur_fs + m][b]);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
        if (b0 + b < nx) a[(b0 + b) * nG + G] = v[b];
}

// ------------------------------------------------------------------ //
// complex (Bloch) functions, exact order (c/lfc.c:400-423, 758-781): a
// volume's values are multiplied by its phase for this k-point.

// add by chunks of covered points (complex): the chunk's coefficient
// blocks for NB bands staged in LDS once, as lfc_add_chunk_kernel; per
// (point, band, entry) the arithmetic of lfc_add_z_kernel, so the result
// is bit-identical to it.
template <int NB>
__global__ __launch_bounds__(256) void lfc_add_chunk_z_kernel(
    const double2* __restrict__ c, double2* __restrict__ a, long nG, int Mmax, long nx,
    long nchunks, const int* __restrict__ ch_i0, const int* __restrict__ ch_foff,
    const int* __restrict__ ch_col, const double* __restrict__ A,
    const int* __restrict__ cov_G, const int* __restrict__ cov_ptr,
    const int2* __restrict__ ent, const unsigned char* __restrict__ ent_f,
    const int* __restrict__ ent_W, const double2* __restrict__ phase_W)
{
    __shared__ double2 cs[kAddFuns][NB];
    const long nbb = (nx + NB - 1) / NB;
    const long w = xcd_work_index(blockIdx.x, nchunks * nbb);
    if (w < 0) return;
    const long ch = w / nbb;
    const long b0 = (w % nbb) * NB;
    const int f0 = ch_foff[ch], nf = ch_foff[ch + 1] - f0;
    for (int idx = threadIdx.x; idx < nf * NB; idx += blockDim.x) {
        const int f = idx % nf, b = idx / nf;
        const long band = b0 + b;
        cs[f][b] = band < nx ? c[band * Mmax + ch_col[f0 + f]] : make_double2(0.0, 0.0);
    }
    __syncthreads();
    const long i = ch_i0[ch] + threadIdx.x;
    if (i >= ch_i0[ch + 1]) return;
    const long G = cov_G[i];
    double2 v[NB];
#pragma unroll
    for (int b = 0; b < NB; b++)
        v[b] = b0 + b < nx ? a[(b0 + b) * nG + G] : make_double2(0.0, 0.0);
    const int e0 = cov_ptr[i], e1 = cov_ptr[i + 1];
    for (int e = e0; e < e1; e++) {
        const int2 en = ent[e];
        const int nm = en.y & 15, fs = ent_f[e];
        const double* Ar = A + en.x;
        double Av[kNF - 1];
#pragma unroll
        for (int m = 0; m < kNF - 1; m++)
            if (m < nm) Av[m] = Ar[m];
        const double2 ph = phase_W[ent_W[e]];
        double tr[NB], ti[NB];
#pragma unroll
        for (int b = 0; b < NB; b++) tr[b] = ti[b] = 0.0;
#pragma unroll
        for (int m = 0; m < kNF - 1; m++) {
            if (m < nm) {
#pragma unroll
                for (int b = 0; b < NB; b++) {
                    const double2 cm = cs[fs + m][b];
                    tr[b] = madd<double>(tr[b], Av[m], cm.x);
                    ti[b] = madd<double>(ti[b], Av[m], cm.y);
                }
            }
        }
        const double pr = ph.x, pim = -ph.y;
#pragma unroll
        for (int b = 0; b < NB; b++) {
            const double r1 = tr[b] * pr, r2 = ti[b] * pim;
            const double i1 = tr[b] * pim, i2 = ti[b] * pr;
            v[b].x = v[b].x + (r1 - r2);
            v[b].y = v[b].y + (i1 + i2);
        }
    }
#pragma unroll
    for (int b = 0; b < NB; b++)
        if (b0 + b < nx) a[(b0 + b) * nG + G] = v[b];
}

// ------------------------------------------------------------------ //
// Exact integrate (FP64 and complex128) by groups of keys with identical
// point lists.
//
// Per (point, band) the value the reference multiplies into every function
// of the volume -- a_G * dv for real functions, a_G * (phase * dv) for
// Bloch functions (c/lfc.c:382, 408-410) -- is rounded once, as there; the
// chain of a function is then c_M += value * A point by point in the key's
// own order, two roundings per step, i.e. exactly the reference's
// c_M1[m] += av * A_gm[gm] sequence.
//
// A chain cannot be split, so a launch is bound by how fast one chain steps
// (one product and one addition per point) and, when the chip is full, by
// what the steps read from LDS.  A workgroup is one staging wave and Q
// summing waves.  The staging wave keeps D chunks of 64 points of loads in
// flight and writes the values and the group's A rows to LDS, points
// contiguous, so a summing wave reads two points per 16-byte read.  Lane
// (band, function) of a summing wave carries one chain, NBL = 64 / NFT bands
// side by side, and issues nothing but LDS reads, products and additions:
// 19 clocks a point measured, 90 us for the 11,300 points of a sphere of
// 2.5 Angstrom at a spacing of 0.18 (one wave doing both: 126 us; staged by
// all lanes of a workgroup in step: 256 to 680 us).
// LDS holds three chunks: one being summed, the next (whose first batches
// are already read), and the one being written; one barrier per chunk.
// Nothing is allocated.
template <typename V> struct ExactStage;
template <> struct ExactStage<double> {
    __device__ static double value(double x, double dv, double2) { return x * dv; }
    __device__ static void add(double& acc, double av, double A) { acc = acc + av * A; }
};
template <> struct ExactStage<double2> {
    __device__ static double2 value(double2 x, double dv, double2 ph)
    {
        const double vr = ph.x * dv, vi = ph.y * dv;
        const double r1 = x.x * vr, r2 = x.y * vi;
        const double i1 = x.x * vi, i2 = x.y * vr;
        return make_double2(r1 - r2, i1 + i2);
    }
    __device__ static void add(double2& acc, double2 av, double A)
    {
        acc.x = acc.x + av.x * A;
        acc.y = acc.y + av.y * A;
    }
};

//
// KEYED: every key is a group of its own, with its A rows where key_row
// points (Bloch functions whose volumes do not share their image's phase:
// cells smaller than the spheres).
//
// P staging waves share the rows; the shapes (Q, P) and the rule between
// them are at lfc_integrate_exact below.
template <typename V, int NFT, int Q, int P, int D, bool KEYED>
__global__ __launch_bounds__(64 * (P + Q)) void lfc_integrate_exact_kernel(
    const V* __restrict__ a, V* __restrict__ c, long nG, int Mmax, long nx, double dv,
    int ngroups, int nfmax, const long* __restrict__ grp_off, const int* __restrict__ grp_nf,
    const int* __restrict__ grp_fM, const int* __restrict__ grp_G,
    const double* __restrict__ grp_A, const int* __restrict__ key_row,
    const int* __restrict__ grp_W, const double2* __restrict__ phase_W)
{
    constexpr bool kZ = std::is_same<V, double2>::value;
    constexpr int CH = 64;                     // points per chunk: one per lane
    constexpr int CHP = CH + 2;                // padded row: 16 rows on distinct banks
    constexpr int NBL = 64 / NFT;              // bands side by side
    constexpr int NB = NBL * Q;                // bands per workgroup
    constexpr int NP = kZ ? 2 : 1;             // parts of a value
    constexpr int BT = 8;                      // points per batch of LDS reads
    __shared__ __attribute__((aligned(16))) double xs[3][NP][NB][CHP];
    __shared__ __attribute__((aligned(16))) double As[3][NFT][CHP];

    // the band blocks of one group are neighbours: they share its A rows
    // and point list in their XCD's L2
    const long nbb = (nx + NB - 1) / NB;
    const long w = xcd_work_index(blockIdx.x, nbb * ngroups);
    if (w < 0) return;
    const int g = (int)(w / nbb);
    const long b0 = (w % nbb) * NB;
    const int nf = grp_nf[g];
    const long j0 = grp_off[g], j1 = grp_off[g + 1];
    const long npts = j1 - j0;
    if (npts == 0) return;                     // (the clamped loads need a point)
    const int nfull = (int)(npts / CH);        // whole chunks; both roles pass nfull + 1 barriers
    const double* Ag = KEYED ? grp_A : grp_A + j0 * nfmax;   // function f: npts values at f * npts
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int lane = threadIdx.x % 64;

    if (wave < P) {
        // Every lane loads from clamped in-range addresses (a load under a
        // condition makes the compiler wait, at the join, for the loads
        // issued after the one it needs); points past the group are staged
        // and never summed.  Slot s holds the chunks n = s mod D: their
        // values, and the point index of the chunk D later, so no value
        // load waits for its own index.
        constexpr int NX = (NB + P - 1) / P, NA = (NFT + P - 1) / P;   // rows of a wave
        V xr[D][NX];
        double ar[D][NA];
        double2 ph[D];
        int Gi[D], Wi[D], Ri[D];
        auto index = [&](int s, int n) {
            const long j = min(j0 + (long)n * CH + lane, j1 - 1);
            Gi[s] = grp_G[j];
            Wi[s] = kZ ? grp_W[j] : 0;
            Ri[s] = KEYED ? key_row[j] : 0;
        };
        auto load = [&](int s, int n) {
#pragma unroll
            for (int q = 0; q < NX; q++)
                xr[s][q] = a[min(b0 + min(wave + P * q, NB - 1), nx - 1) * nG + Gi[s]];
            const long jl = min((long)n * CH + lane, npts - 1);
#pragma unroll
            for (int q = 0; q < NA; q++) {
                const int fq = min(wave + P * q, nf - 1);
                ar[s][q] = KEYED ? Ag[Ri[s] + fq] : Ag[fq * npts + jl];
            }
            if (kZ) ph[s] = phase_W[Wi[s]];
            index(s, n + D);
            // issue order kept: the waits count the loads after the slot
            __builtin_amdgcn_sched_barrier(0);
        };
        auto stage = [&](int s, int buf) {
#pragma unroll
            for (int q = 0; q < NX; q++) {
                const V v = ExactStage<V>::value(xr[s][q], dv, ph[s]);
                const int row = min(wave + P * q, NB - 1);   // past the last: the same value again
                if constexpr (kZ) {
                    xs[buf][0][row][lane] = v.x;
                    xs[buf][1][row][lane] = v.y;
                } else {
                    xs[buf][0][row][lane] = v;
                }
            }
#pragma unroll
            for (int q = 0; q < NA; q++) {
                const int row = min(wave + P * q, NFT - 1);
                As[buf][row][lane] = ar[s][q];
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int s = 0; s < D; s++) index(s, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < D; s++) load(s, s);
        // iteration n stages chunk n + 2; chunks 0 and 1 before the first
        // barrier (n = -2, -1)
        int buf = 0;
        for (int n = -2;; n += D) {
#pragma unroll
            for (int s = 0; s < D; s++) {
                if (n + s >= nfull) return;
                stage(s, buf);
                load(s, n + s + 2 + D);
                buf = buf == 2 ? 0 : buf + 1;
                if (n + s >= -1) lds_barrier();
            }
        }
    }

    const int f = lane % NFT, bl = lane / NFT;
    const int wb = (wave - P) * NBL;           // this wave's bands in the block
    const long band = b0 + wb + bl;
    const bool ok = bl < NBL && f < nf && band < nx;
    const int M = KEYED ? grp_fM[g] + f : grp_fM[(long)g * nfmax + (f < nf ? f : 0)];
    V* cp = c + band * Mmax + M;
    V acc = V();
    if (ok) acc = *cp;
    // idle lanes read a row of the block and are not stored
    const int fr = f < nf ? f : 0;
    const int xrow = wb + (bl < NBL ? bl : 0);

    // Batches of BT points in the pipeline: one being read from LDS, the
    // products of the next formed between the additions of the present one
    // (an addition waits for the one before it, not for its product).
    double2 xb[2][NP][BT / 2], ab[2][BT / 2];
    double pr[2][NP][BT];
    auto fetch = [&](int r, int buf, int p) {
#pragma unroll
        for (int u = 0; u < BT / 2; u++) {
            ab[r][u] = *(const double2*)&As[buf][fr][p + 2 * u];
#pragma unroll
            for (int k = 0; k < NP; k++)
                xb[r][k][u] = *(const double2*)&xs[buf][k][xrow][p + 2 * u];
        }
    };
    auto products = [&](int r, int u) {
        const double2 A = ab[r][u / 2];
#pragma unroll
        for (int k = 0; k < NP; k++) {
            const double2 x = xb[r][k][u / 2];
            pr[r][k][u] = (u & 1) ? x.y * A.y : x.x * A.x;
        }
    };
    auto add = [&](int r, int u) {
        if constexpr (kZ) {
            acc.x = acc.x + pr[r][0][u];
            acc.y = acc.y + pr[r][1][u];
        } else {
            acc = acc + pr[r][0][u];
        }
    };

    lds_barrier();                             // chunks 0 and 1 are in LDS
    fetch(0, 0, 0);
    fetch(1, 0, BT);
#pragma unroll
    for (int u = 0; u < BT; u++) products(0, u);
    int buf = 0;
    for (int n = 0; n < nfull; n++) {
        const int next = buf == 2 ? 0 : buf + 1;
#pragma unroll
        for (int m = 0; m < CH / BT; m++) {
            const int r = m & 1;
            __builtin_amdgcn_sched_barrier(0);
            if (m + 2 < CH / BT) fetch(r, buf, (m + 2) * BT);
            else fetch(r, next, (m + 2 - CH / BT) * BT);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < BT; u++) {
                add(r, u);
                products(r ^ 1, u);
            }
        }
        // every read of this chunk has been used above (the scheduling
        // barrier keeps it so); the reads in flight are of the next chunk,
        // which this barrier does not release for writing
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        buf = next;
    }
    const int np = (int)(npts - (long)nfull * CH);
    for (int p = 0; p < np; p++) {
        const double A = As[buf][fr][p];
        if constexpr (kZ)
            ExactStage<V>::add(acc, make_double2(xs[buf][0][xrow][p], xs[buf][1][xrow][p]), A);
        else
            ExactStage<V>::add(acc, xs[buf][0][xrow][p], A);
    }
    if (ok) *cp = acc;
}

// The same chains where workgroups are few.  The summing wave above is bound
// by what its lanes read from LDS, 16 bytes a point, so here a workgroup has
// few chains (18 for groups of nine functions: two bands, or the parts of one
// complex band, each part a chain of its own), a lane reads finished products
// only, and its wave issues nothing but those reads and the additions: P waves
// of lanes that are points load the values and A rows, form every chain's
// product and write it to LDS (chains by points).  An addition that waits for
// the one before it takes 8.6 clocks, with its share of a read 9.7; 11 measured
// here.  The sphere of 11,300 points: 4 bands of 24^3 and 2 atoms 57 us (19
// clocks a point and 93 us above), 32 bands and 10 atoms 64 (96); 4 complex
// bands and 2 atoms 65 (143), 64 and 8 atoms 90 (146).  With all 64 lanes in use
// 124 us: 128 bytes of LDS a clock are not to be had.
// LDS holds the products of three chunks as above.
template <typename V, int NFT, int NB, int P, int D, bool KEYED>
__global__ __launch_bounds__(64 * (P + 1)) void lfc_integrate_products_kernel(
    const V* __restrict__ a, V* __restrict__ c, long nG, int Mmax, long nx, double dv,
    int ngroups, int nfmax, const long* __restrict__ grp_off, const int* __restrict__ grp_nf,
    const int* __restrict__ grp_fM, const int* __restrict__ grp_G,
    const double* __restrict__ grp_A, const int* __restrict__ key_row,
    const int* __restrict__ grp_W, const double2* __restrict__ phase_W)
{
    constexpr bool kZ = std::is_same<V, double2>::value;
    constexpr int CH = 64;                     // points per chunk: one per lane
    constexpr int CHP = CH + 2;                // padded row: 16 rows on distinct banks
    constexpr int NP = kZ ? 2 : 1;             // parts of a value
    static_assert(NB * NP * NFT <= 64, "a lane a chain");
    constexpr int BT = 8;                      // points per batch of LDS reads
    constexpr int RB = 4;                      // batches of reads in registers
    __shared__ __attribute__((aligned(16))) double ps[3][NB * NP * NFT][CHP];

    const long nbb = (nx + NB - 1) / NB;
    const long w = xcd_work_index(blockIdx.x, nbb * ngroups);
    if (w < 0) return;
    const int g = (int)(w / nbb);
    const long b0 = (w % nbb) * NB;
    const int nf = grp_nf[g];
    const long j0 = grp_off[g], j1 = grp_off[g + 1];
    const long npts = j1 - j0;
    if (npts == 0) return;                     // (the clamped loads need a point)
    const int nfull = (int)(npts / CH);        // whole chunks; both roles pass nfull + 1 barriers
    const double* Ag = KEYED ? grp_A : grp_A + j0 * nfmax;   // function f: npts values at f * npts
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
    const int lane = threadIdx.x % 64;

    if (wave < P) {
        // loads as in lfc_integrate_exact_kernel: clamped addresses, slot s
        // the chunks n = s mod D
        constexpr int NX = (NB * NP + P - 1) / P;   // rows (band, part) of a wave
        V xr[D][NX];
        double ar[D][NFT];
        double2 ph[D];
        int Gi[D], Wi[D], Ri[D];
        auto index = [&](int s, int n) {
            const long j = min(j0 + (long)n * CH + lane, j1 - 1);
            Gi[s] = grp_G[j];
            Wi[s] = kZ ? grp_W[j] : 0;
            Ri[s] = KEYED ? key_row[j] : 0;
        };
        auto load = [&](int s, int n) {
#pragma unroll
            for (int q = 0; q < NX; q++)
                xr[s][q] = a[min(b0 + min((wave + P * q) / NP, NB - 1), nx - 1) * nG + Gi[s]];
            const long jl = min((long)n * CH + lane, npts - 1);
#pragma unroll
            for (int f = 0; f < NFT; f++) {
                const int fq = min(f, nf - 1);
                ar[s][f] = KEYED ? Ag[Ri[s] + fq] : Ag[fq * npts + jl];
            }
            if (kZ) ph[s] = phase_W[Wi[s]];
            index(s, n + D);
            // issue order kept: the waits count the loads after the slot
            __builtin_amdgcn_sched_barrier(0);
        };
        auto stage = [&](int s, int buf) {
#pragma unroll
            for (int q = 0; q < NX; q++) {
                const int row = wave + P * q;
                if (row >= NB * NP) break;
                const V v = ExactStage<V>::value(xr[s][q], dv, ph[s]);
#pragma unroll
                for (int f = 0; f < NFT; f++) {
                    if (f >= nf) break;
                    double x;
                    if constexpr (kZ) x = row % 2 ? v.y : v.x;
                    else x = v;
                    ps[buf][row * NFT + f][lane] = x * ar[s][f];
                }
            }
            __builtin_amdgcn_sched_barrier(0);
        };
#pragma unroll
        for (int s = 0; s < D; s++) index(s, s);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int s = 0; s < D; s++) load(s, s);
        // iteration n stages chunk n + 2; chunks 0 and 1 before the first
        // barrier (n = -2, -1)
        int buf = 0;
        for (int n = -2;; n += D) {
#pragma unroll
            for (int s = 0; s < D; s++) {
                if (n + s >= nfull) return;
                stage(s, buf);
                load(s, n + s + 2 + D);
                buf = buf == 2 ? 0 : buf + 1;
                if (n + s >= -1) lds_barrier();
            }
        }
    }

    const int f = lane % NFT, row = lane / NFT;   // row: band (and part)
    const int part = kZ ? row % 2 : 0;
    const long band = b0 + row / NP;
    const bool ok = row < NB * NP && f < nf && band < nx;
    const int M = KEYED ? grp_fM[g] + f : grp_fM[(long)g * nfmax + (f < nf ? f : 0)];
    double* cp = (double*)(c + band * Mmax + M) + part;
    if (!ok) return;                           // idle lanes would cost LDS bandwidth
    double acc = *cp;

    // RB batches of BT points: the one being added, the others in flight
    double2 pr[RB][BT / 2];
    auto fetch = [&](int r, int buf, int p) {
#pragma unroll
        for (int u = 0; u < BT / 2; u++) pr[r][u] = *(const double2*)&ps[buf][lane][p + 2 * u];
    };
    lds_barrier();                             // chunks 0 and 1 are in LDS
#pragma unroll
    for (int r = 0; r < RB - 1; r++) fetch(r, 0, r * BT);
    int buf = 0;
    for (int n = 0; n < nfull; n++) {
        const int next = buf == 2 ? 0 : buf + 1;
#pragma unroll
        for (int m = 0; m < CH / BT; m++) {
            constexpr int NM = CH / BT;
            const int ahead = m + RB - 1;
            __builtin_amdgcn_sched_barrier(0);
            if (ahead < NM) fetch(ahead % RB, buf, ahead * BT);
            else fetch(ahead % RB, next, (ahead - NM) * BT);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int u = 0; u < BT / 2; u++) {
                acc = acc + pr[m % RB][u].x;
                acc = acc + pr[m % RB][u].y;
            }
        }
        // every read of this chunk has been used above (the scheduling
        // barrier keeps it so); the reads in flight are of the next chunk,
        // which this barrier does not release for writing
        __builtin_amdgcn_sched_barrier(0);
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
        buf = next;
    }
    const int np = (int)(npts - (long)nfull * CH);
    for (int p = 0; p < np; p++) acc = acc + ps[buf][lane][p];
    *cp = acc;
}

// add: one thread per (covered point, NBT bands); per entry in the sweep's
// volume order t = sum_m A c (from 0), then a += t * conj(phase).  Each A
// value is loaded once for the NBT bands.
template <int NBT>
__global__ void lfc_add_z_kernel(const double2* __restrict__ c, double2* __restrict__ a,
                                 long nG, int Mmax, long nx, long ncov,
                                 const double* __restrict__ A, const int* __restrict__ cov_G,
                                 const int* __restrict__ cov_ptr, const int2* __restrict__ ent,
                                 const int* __restrict__ ent_W,
                                 const double2* __restrict__ phase_W)
{
    const long nbblk = (nx + NBT - 1) / NBT;
    const long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nbblk * ncov) return;
    const long i = idx % ncov;
    const long b0 = (idx / ncov) * NBT;
    const long G = cov_G[i];
    double2 v[NBT];
#pragma unroll
    for (int bb = 0; bb < NBT; bb++)
        v[bb] = b0 + bb < nx ? a[(b0 + bb) * nG + G] : make_double2(0.0, 0.0);
    const int e1 = cov_ptr[i + 1];
    for (int e = cov_ptr[i]; e < e1; e++) {
        const int2 en = ent[e];
        const int nm = en.y & 15;
        const double* Ar = A + en.x;
        const int M = en.y >> 4;
        double tr[NBT], ti[NBT];
#pragma unroll
        for (int bb = 0; bb < NBT; bb++) tr[bb] = ti[bb] = 0.0;
        for (int m = 0; m < nm; m++) {
            const double Am = Ar[m];
#pragma unroll
            for (int bb = 0; bb < NBT; bb++) {
                const long b = b0 + bb < nx ? b0 + bb : b0;
                const double2 cm = c[b * Mmax + M + m];
                tr[bb] = madd<double>(tr[bb], Am, cm.x);
                ti[bb] = madd<double>(ti[bb], Am, cm.y);
            }
        }
        const double2 ph = phase_W[ent_W[e]];
        const double pr = ph.x, pim = -ph.y;
#pragma unroll
        for (int bb = 0; bb < NBT; bb++) {
            const double r1 = tr[bb] * pr, r2 = ti[bb] * pim;
            const double i1 = tr[bb] * pim, i2 = ti[bb] * pr;
            v[bb].x = v[bb].x + (r1 - r2);
            v[bb].y = v[bb].y + (i1 + i2);
        }
    }
#pragma unroll
    for (int bb = 0; bb < NBT; bb++)
        if (b0 + bb < nx) a[(b0 + bb) * nG + G] = v[bb];
}

// ------------------------------------------------------------------ //
// host-side sweep

struct HostTables {
    std::vector<int> ptr;            // nG + 1
    std::vector<int2> ent;
    std::vector<int> ent_W;          // volume of each entry
    std::vector<int> cov_G, cov_ptr;
    std::map<int, int> key_of_M;     // M -> key
    std::vector<int> key_M, key_nm;
    std::vector<std::vector<int>> key_G, key_row, key_W;
};

static bool run_sweep(int nW, const long* A_off, const int* ng_W, const int* nm_W,
                      const int* M_W, int nB, const int* G_B, const int* W_B, long nG,
                      HostTables& h)
{
    struct Vol {
        long row;    // rows consumed
        int W;
    };
    std::vector<Vol> vol_i;
    std::vector<long> row_W(nW, 0);
    std::vector<int> i_W(nW, -1);
    h.ptr.assign(nG + 1, 0);
    std::vector<int> count(nG, 0);
    // first pass: count entries per point
    {
        long Ga = 0;
        int ni = 0;
        for (int B = 0; B < nB; B++) {
            long Gb = G_B[B];
            if (Gb < Ga || Gb > nG) return false;
            if (Gb > Ga && ni > 0)
                for (long G = Ga; G < Gb; G++) count[G] += ni;
            if (W_B[B] >= 0) ni++;
            else ni--;
            if (ni < 0) return false;
            Ga = Gb;
        }
        if (ni != 0) return false;
    }
    for (long G = 0; G < nG; G++) h.ptr[G + 1] = h.ptr[G] + count[G];
    h.ent.resize(h.ptr[nG]);
    h.ent_W.resize(h.ptr[nG]);
    std::vector<int> fill(h.ptr.begin(), h.ptr.end() - 1);
    for (int W = 0; W < nW; W++) {
        auto it = h.key_of_M.find(M_W[W]);
        if (it == h.key_of_M.end()) {
            int k = (int)h.key_M.size();
            h.key_of_M[M_W[W]] = k;
            h.key_M.push_back(M_W[W]);
            h.key_nm.push_back(nm_W[W]);
        } else if (h.key_nm[it->second] != nm_W[W]) {
            return false;
        }
    }
    h.key_G.assign(h.key_M.size(), {});
    h.key_row.assign(h.key_M.size(), {});
    h.key_W.assign(h.key_M.size(), {});

    long Ga = 0;
    for (int B = 0; B < nB; B++) {
        long Gb = G_B[B];
        long nGs = Gb - Ga;
        if (nGs > 0) {
            for (const Vol& v : vol_i)
                if (v.row + nGs > ng_W[v.W]) return false;
            for (long G = Ga; G < Gb; G++)
                for (const Vol& v : vol_i) {
                    int nm = nm_W[v.W];
                    long rowoff = A_off[v.W] + (v.row + (G - Ga)) * nm;
                    if (rowoff > 0x7fffffffL) return false;
                    h.ent_W[fill[G]] = v.W;
                    h.ent[fill[G]++] = make_int2((int)rowoff, (M_W[v.W] << 4) | nm);
                }
            for (const Vol& v : vol_i) {
                int k = h.key_of_M[M_W[v.W]];
                int nm = nm_W[v.W];
                for (long G = Ga; G < Gb; G++) {
                    h.key_G[k].push_back((int)G);
                    h.key_row[k].push_back((int)(A_off[v.W] + (v.row + (G - Ga)) * nm));
                    h.key_W[k].push_back(v.W);
                }
            }
            for (Vol& v : vol_i) v.row += nGs;
        }
        int Wn = W_B[B];
        if (Wn >= 0) {
            if (Wn >= nW || i_W[Wn] >= 0) return false;
            i_W[Wn] = (int)vol_i.size();
            vol_i.push_back({row_W[Wn], Wn});
        } else {
            int Wold = -1 - Wn;
            if (Wold >= nW || i_W[Wold] < 0) return false;
            int iold = i_W[Wold];
            row_W[Wold] = vol_i[iold].row;
            vol_i[iold] = vol_i.back();
            vol_i.pop_back();
            if (iold < (int)vol_i.size()) i_W[vol_i[iold].W] = iold;
            i_W[Wold] = -1;
        }
        Ga = Gb;
    }
    // every volume must have consumed exactly its rows
    if (!vol_i.empty()) return false;
    for (int W = 0; W < nW; W++)
        if (row_W[W] != ng_W[W]) return false;
    for (long G = 0; G < nG; G++)
        if (h.ptr[G + 1] > h.ptr[G]) {
            h.cov_G.push_back((int)G);
            h.cov_ptr.push_back(h.ptr[G]);
        }
    h.cov_ptr.push_back(h.ptr[nG]);
    return true;
}

template <typename V>
static hipError_t upload(V** dst, const V* src, size_t n)
{
    *dst = nullptr;
    // keep a valid pointer for empty tables
    hipError_t e = hipMalloc((void**)dst, sizeof(V) * (n ? n : 1));
    if (e != hipSuccess) return e;
    if (src && n) return hipMemcpy(*dst, src, sizeof(V) * n, hipMemcpyHostToDevice);
    return hipMemset(*dst, 0, sizeof(V) * (n ? n : 1));
}

template <typename T, int NB>
static int lfc_add_chunk_launch(const gpd_lfc* l, long nx, const T* c, T* a, hipStream_t st)
{
    const long nwork = l->nchunks * ((nx + NB - 1) / NB);
    hipLaunchKernelGGL((lfc_add_chunk_kernel<T, NB>), dim3(xcd_grid_size(nwork)), dim3(256), 0,
                       st, c, a, l->nG, l->Mmax, nx, l->nchunks, l->ch_i0, l->ch_foff,
                       l->ch_col, lfc_values<T>(l), l->cov_G, l->cov_ptr, l->ent, l->ent_f);
    return last_error_to_status(hipGetLastError());
}

int lfc_add_f32(const gpd_lfc* l, long nx, const float* c, float* a, hipStream_t st)
{
    if (nx == 0 || l->ncov == 0) return GPD_OK;
    if (l->nchunks > 0) return lfc_add_chunk_launch<float, 16>(l, nx, c, a, st);
    return lfc_add_grouped_f32(l, nx, c, a, st);
}

int lfc_add_exact_f64(const gpd_lfc* l, long nx, const double* c, double* a, hipStream_t st)
{
    if (nx == 0 || l->ncov == 0) return GPD_OK;
    if (l->nchunks > 0) return lfc_add_chunk_launch<double, 16>(l, nx, c, a, st);
    constexpr int NBT = 8;
    const long n = ((nx + NBT - 1) / NBT) * l->ncov;
    hipLaunchKernelGGL((lfc_add_kernel<double, NBT>), dim3((n + 255) / 256), dim3(256), 0, st, c,
                       a, l->nG, l->Mmax, nx, l->ncov, l->A64, l->cov_G, l->cov_ptr, l->ent);
    return last_error_to_status(hipGetLastError());
}

template <int NB, int NF>
static int lfc_add_grouped_launch(const gpd_lfc* l, long nx, const float* c, float* a,
                                  hipStream_t st)
{
    const long nbblk = (nx + NB - 1) / NB;
    const LfcGroups& gs = l->ga;
    for (int col = 0; col < gs.ncolours; col++) {
        const int i0 = gs.colour_items[col], i1 = gs.colour_items[col + 1];
        if (i1 == i0) continue;
        const long nwork = (long)(i1 - i0) * nbblk;
        hipLaunchKernelGGL((lfc_add_grp_kernel<NB, NF>), dim3(xcd_grid_size(nwork)), dim3(256), 0,
                           st, c, a, l->nG, l->Mmax, nx, gs.nfmax, i1 - i0, gs.item_g + i0,
                           gs.item_j0 + i0, gs.grp_off, gs.grp_nf, gs.grp_fM, gs.grp_G,
                           gs.grp_A32);
        int rc = last_error_to_status(hipGetLastError());
        if (rc) return rc;
    }
    return GPD_OK;
}

template <typename V, int NFT, int Q, int P, int D>
static int lfc_integrate_exact_launch(const gpd_lfc* l, long nx, const V* a, V* c,
                                      hipStream_t st)
{
    constexpr int NB = 64 / NFT * Q;
    const long nbb = (nx + NB - 1) / NB;
    if constexpr (std::is_same<V, double2>::value) {
        if (!l->grp_phase_shared) {
            hipLaunchKernelGGL((lfc_integrate_exact_kernel<V, NFT, Q, P, D, true>),
                               dim3(xcd_grid_size(nbb * l->nkeys)), dim3(64 * (P + Q)), 0, st, a,
                               c, l->nG, l->Mmax, nx, l->dv, l->nkeys, 0, l->key_off, l->key_nm,
                               l->key_M, l->key_G, l->A64, l->key_row, l->key_W, l->phase_W);
            return last_error_to_status(hipGetLastError());
        }
    }
    const LfcGroups& gs = l->gi;
    hipLaunchKernelGGL((lfc_integrate_exact_kernel<V, NFT, Q, P, D, false>),
                       dim3(xcd_grid_size(nbb * gs.ngroups)), dim3(64 * (P + Q)), 0, st, a, c,
                       l->nG, l->Mmax, nx, l->dv, gs.ngroups, gs.nfmax, gs.grp_off, gs.grp_nf,
                       gs.grp_fM, gs.grp_G, gs.grp_A64, nullptr, gs.grp_W, l->phase_W);
    return last_error_to_status(hipGetLastError());
}

template <typename V, int NFT, int NB, int P, int D>
static int lfc_integrate_products_launch(const gpd_lfc* l, long nx, const V* a, V* c,
                                         hipStream_t st)
{
    const long nbb = (nx + NB - 1) / NB;
    if constexpr (std::is_same<V, double2>::value) {
        if (!l->grp_phase_shared) {
            hipLaunchKernelGGL((lfc_integrate_products_kernel<V, NFT, NB, P, D, true>),
                               dim3(xcd_grid_size(nbb * l->nkeys)), dim3(64 * (P + 1)), 0, st, a,
                               c, l->nG, l->Mmax, nx, l->dv, l->nkeys, 0, l->key_off, l->key_nm,
                               l->key_M, l->key_G, l->A64, l->key_row, l->key_W, l->phase_W);
            return last_error_to_status(hipGetLastError());
        }
    }
    const LfcGroups& gs = l->gi;
    hipLaunchKernelGGL((lfc_integrate_products_kernel<V, NFT, NB, P, D, false>),
                       dim3(xcd_grid_size(nbb * gs.ngroups)), dim3(64 * (P + 1)), 0, st, a, c,
                       l->nG, l->Mmax, nx, l->dv, gs.ngroups, gs.nfmax, gs.grp_off, gs.grp_nf,
                       gs.grp_fM, gs.grp_G, gs.grp_A64, nullptr, gs.grp_W, l->phase_W);
    return last_error_to_status(hipGetLastError());
}

// Shapes of the exact integrate.  Few chains a workgroup and finished products
// while that gives at most two workgroups a CU (real bands, 64 of 64^3 and 10
// atoms, 320 workgroups: 78 us, 96 with the next shape; 128 bands, 640: 102 and
// 97), complex bands up to four (64 of 64^3, 12 atoms, 768: 108 and 147 us).
// Loads for six chunks ahead while workgroups leave half of the CUs free; with
// more of them fewer waves or registers, as H psi runs its stencil beside them
// (H psi of 64 complex bands of 48^3 and 8 atoms, 512 workgroups: 247 us with one
// product wave and four chunks, 304 with two and six; 64 real bands, 256: 164
// with two and three, 180 with two and six).  Then (summing waves, staging
// waves) = (1, 1), (2, 2) or, real bands, (3, 1): the first while its
// workgroups fit the 256 CUs (64^3 x 128, 10 atoms: 97 us, 104 and 131 with the
// others); then fewer workgroups that share the staged A rows (96^3 x 64, 32
// atoms, 320 workgroups: 131, 112 and 142 us; 96^3 x 256, 1184 workgroups: 305,
// 283 and 267 us).  gpd_lfc_set_launch picks one of these three by hand.
constexpr int kProductLanes = 20;   // chains of a workgroup of products, at most

template <typename V, int NFT>
static int lfc_integrate_exact_shape(const gpd_lfc* l, long nx, const V* a, V* c, hipStream_t st)
{
    constexpr bool kZ = std::is_same<V, double2>::value;
    constexpr int NBL = 64 / NFT;
    constexpr int NF = kProductLanes / (NFT * (kZ ? 2 : 1));
    constexpr int NB = NF > 0 ? NF : 1;
    const long groups = kZ && !l->grp_phase_shared ? l->nkeys : l->gi.ngroups;
    const long few = groups * ((nx + NB - 1) / NB);
    if (!l->exact_nbb && few <= 128)
        return lfc_integrate_products_launch<V, NFT, NB, 2, 6>(l, nx, a, c, st);
    if (!l->exact_nbb && few <= (kZ ? 1024 : 512))
        return lfc_integrate_products_launch<V, NFT, NB, kZ ? 1 : 2, kZ ? 4 : 3>(l, nx, a, c, st);
    const long wgs = groups * ((nx + NBL - 1) / NBL);
    const int shape = l->exact_nbb ? l->exact_nbb : (wgs <= 256 ? 16 : (wgs <= 1024 ? 32 : 64));
    if (shape == 16)
        return lfc_integrate_exact_launch<V, NFT, 1, 1, kZ ? 2 : 4>(l, nx, a, c, st);
    if constexpr (!kZ)
        if (shape == 64) return lfc_integrate_exact_launch<V, NFT, 3, 1, 3>(l, nx, a, c, st);
    return lfc_integrate_exact_launch<V, NFT, 2, 2, kZ ? 2 : 3>(l, nx, a, c, st);
}

template <typename V>
static int lfc_integrate_exact(const gpd_lfc* l, long nx, const V* a, V* c, hipStream_t st)
{
    // lanes per band: the functions of the largest group
    const int nf = l->gi.nfmax;
    if (l->gi.ngroups == 0) return GPD_OK;
    if (nf <= 4) return lfc_integrate_exact_shape<V, 4>(l, nx, a, c, st);
    if (nf <= 9) return lfc_integrate_exact_shape<V, 9>(l, nx, a, c, st);
    return lfc_integrate_exact_shape<V, kNF>(l, nx, a, c, st);
}

int lfc_add_grouped_f32(const gpd_lfc* l, long nx, const float* c, float* a, hipStream_t st)
{
    // 16 bands per workgroup share each point's A row when groups hold at
    // most 9 functions (one atom with l = 0..2)
    if (l->ga.nfmax <= 9) return lfc_add_grouped_launch<16, 9>(l, nx, c, a, st);
    return lfc_add_grouped_launch<8, kNF>(l, nx, c, a, st);
}



// Groups of keys with identical point lists (<= kNF functions each, keys
// taken in M order), their FP32 A tables and a greedy colouring into sets
// of groups with disjoint points; uploads everything into gs.
static hipError_t build_groups(const std::vector<int>& key_M, const std::vector<int>& key_nm,
                               const std::vector<std::vector<int>>& key_G,
                               const std::vector<std::vector<int>>& key_row,
                               const std::vector<std::vector<int>>* key_W, const double* A,
                               long nG, LfcGroups& gs)
{
    const int nkeys = (int)key_M.size();
    std::vector<int> order(nkeys);
    for (int k = 0; k < nkeys; k++) order[k] = k;
    std::stable_sort(order.begin(), order.end(),
                     [&](int x, int y) { return key_M[x] < key_M[y]; });
    std::vector<std::vector<int>> groups;
    std::vector<int> group_nf;
    for (int k : order) {
        int found = -1;
        for (int g = (int)groups.size() - 1; g >= 0 && g >= (int)groups.size() - 8; g--) {
            int k0 = groups[g][0];
            if (group_nf[g] + key_nm[k] <= kNF && key_G[k0] == key_G[k]) {
                found = g;
                break;
            }
        }
        if (found < 0) {
            groups.push_back({k});
            group_nf.push_back(key_nm[k]);
        } else {
            groups[found].push_back(k);
            group_nf[found] += key_nm[k];
        }
    }
    gs.ngroups = (int)groups.size();
    int nfmax = 1;
    for (int nf : group_nf) nfmax = std::max(nfmax, nf);
    gs.nfmax = nfmax;
    std::vector<long> grp_off(gs.ngroups + 1, 0);
    for (int g = 0; g < gs.ngroups; g++)
        grp_off[g + 1] = grp_off[g] + (long)key_G[groups[g][0]].size();
    gs.npts_total = grp_off[gs.ngroups];
    std::vector<int> gG(gs.npts_total), gfM((size_t)gs.ngroups * nfmax, 0);
    std::vector<float> gA((size_t)gs.npts_total * nfmax, 0.f);
    // the exact (FP64, complex) integrate also needs the FP64 values and the
    // volume (phase) of each point
    std::vector<double> gA64(key_W ? (size_t)gs.npts_total * nfmax : 0, 0.0);
    std::vector<int> gW(key_W ? gs.npts_total : 0, 0);
    std::vector<std::pair<int, int>> pairs;
    for (int g = 0; g < gs.ngroups; g++) {
        const std::vector<int>& pts = key_G[groups[g][0]];
        std::copy(pts.begin(), pts.end(), gG.begin() + grp_off[g]);
        int f = 0;
        for (int k : groups[g]) {
            for (int m = 0; m < key_nm[k]; m++, f++) {
                gfM[(size_t)g * nfmax + f] = key_M[k] + m;
                for (size_t j = 0; j < pts.size(); j++) {
                    gA[(grp_off[g] + j) * nfmax + f] = (float)A[key_row[k][j] + m];
                    if (key_W)
                        gA64[grp_off[g] * nfmax + f * pts.size() + j] = A[key_row[k][j] + m];
                }
            }
            if (key_W) {
                const std::vector<int>& W0 = (*key_W)[groups[g][0]];
                const std::vector<int>& Wk = (*key_W)[k];
                for (size_t j = 0; j < pts.size(); j++) {
                    gW[grp_off[g] + j] = W0[j];
                    if (Wk[j] != W0[j]) pairs.emplace_back(W0[j], Wk[j]);
                }
            }
        }
    }
    std::sort(pairs.begin(), pairs.end());
    pairs.erase(std::unique(pairs.begin(), pairs.end()), pairs.end());
    gs.phase_pairs = pairs;

    std::vector<int> colour_of(gs.ngroups, -1);
    std::vector<std::vector<char>> used;
    for (int g = 0; g < gs.ngroups; g++) {
        const std::vector<int>& pts = key_G[groups[g][0]];
        int col = 0;
        for (;; col++) {
            if (col == (int)used.size()) used.emplace_back(nG, 0);
            bool clash = false;
            for (int G : pts)
                if (used[col][G]) {
                    clash = true;
                    break;
                }
            if (!clash) break;
        }
        for (int G : pts) used[col][G] = 1;
        colour_of[g] = col;
    }
    gs.ncolours = (int)used.size();
    std::vector<int> item_g;
    std::vector<long> item_j0;
    gs.colour_items.assign(gs.ncolours + 1, 0);
    for (int col = 0; col < gs.ncolours; col++) {
        gs.colour_items[col] = (int)item_g.size();
        for (int g = 0; g < gs.ngroups; g++)
            if (colour_of[g] == col)
                for (long j = grp_off[g]; j < grp_off[g + 1]; j += 256) {
                    item_g.push_back(g);
                    item_j0.push_back(j);
                }
    }
    gs.colour_items[gs.ncolours] = (int)item_g.size();

    hipError_t e = hipSuccess;
    if (e == hipSuccess) e = upload(&gs.grp_off, grp_off.data(), grp_off.size());
    if (e == hipSuccess) e = upload(&gs.grp_nf, group_nf.data(), group_nf.size());
    if (e == hipSuccess) e = upload(&gs.grp_fM, gfM.data(), gfM.size());
    if (e == hipSuccess) e = upload(&gs.grp_G, gG.data(), gG.size());
    if (e == hipSuccess) e = upload(&gs.grp_A32, gA.data(), gA.size());
    if (key_W && e == hipSuccess) e = upload(&gs.grp_A64, gA64.data(), gA64.size());
    if (key_W && e == hipSuccess) e = upload(&gs.grp_W, gW.data(), gW.size());
    if (e == hipSuccess) e = upload(&gs.item_g, item_g.data(), item_g.size());
    if (e == hipSuccess) e = upload(&gs.item_j0, item_j0.data(), item_j0.size());
    return e;
}

static void free_groups(LfcGroups& gs)
{
    void* ptrs[] = {gs.grp_off, gs.grp_nf, gs.grp_fM, gs.grp_G, gs.grp_A32, gs.grp_A64,
                    gs.grp_W,   gs.item_g, gs.item_j0};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    gs = LfcGroups();
}

}  // namespace gpd

using namespace gpd;

extern "C" int gpd_lfc_destroy(gpd_lfc* l)
{
    if (!l) return GPD_OK;
    void* ptrs[] = {l->A64, l->A32, l->ptr, l->ent, l->cov_G, l->cov_ptr, l->key_M, l->key_nm,
                    l->key_off, l->key_G, l->key_row, l->ent_W, l->key_W,
                    l->phase_W, l->ch_i0, l->ch_foff, l->ch_col, l->ent_f};
    for (void* p : ptrs)
        if (p) (void)hipFree(p);
    if (l->seg_part) (void)hipFree(l->seg_part);
    free_groups(l->gi);
    if (!l->add_shares_groups) free_groups(l->ga);
    delete l;
    return GPD_OK;
}

extern "C" int gpd_lfc_create(int nW, const double* A, const int* ng_W, const int* nm_W,
                              const int* M_W, int nB, const int* G_B, const int* W_B, double dv,
                              long nG, int Mmax, gpd_lfc** out)
{
    GPD_REQUIRE(out, GPD_ERR_ARG, "null output");
    *out = nullptr;
    GPD_REQUIRE(nW >= 0 && nB >= 0 && nG > 0 && Mmax >= 0, GPD_ERR_ARG, "bad sizes");
    GPD_REQUIRE(nW == 0 || (A && ng_W && nm_W && M_W), GPD_ERR_ARG, "null volume arrays");
    GPD_REQUIRE(nB == 0 || (G_B && W_B), GPD_ERR_ARG, "null boundary arrays");
    std::vector<long> A_off(nW + 1, 0);
    for (int W = 0; W < nW; W++) {
        GPD_REQUIRE(nm_W[W] >= 1 && nm_W[W] <= kNF - 1 && ng_W[W] >= 0, GPD_ERR_ARG,
                    "volume with unsupported function count");
        GPD_REQUIRE(M_W[W] >= 0 && M_W[W] + nm_W[W] <= Mmax, GPD_ERR_ARG, "M index out of range");
        A_off[W + 1] = A_off[W] + (long)ng_W[W] * nm_W[W];
    }
    HostTables h;
    GPD_REQUIRE(run_sweep(nW, A_off.data(), ng_W, nm_W, M_W, nB, G_B, W_B, nG, h), GPD_ERR_ARG,
                "boundary list inconsistent with the volumes");

    gpd_lfc* l = new (std::nothrow) gpd_lfc();
    GPD_REQUIRE(l, GPD_ERR_NOMEM, "out of host memory");
    l->nG = nG;
    l->Mmax = Mmax;
    l->dv = dv;
    l->nvalues = A_off[nW];
    l->ncov = (long)h.cov_G.size();
    l->nent = (long)h.ent.size();
    l->nkeys = (int)h.key_M.size();

    // per-key flat arrays
    std::vector<long> key_off(l->nkeys + 1, 0);
    for (int k = 0; k < l->nkeys; k++) key_off[k + 1] = key_off[k] + (long)h.key_G[k].size();
    std::vector<int> kG, kR, kW;
    kG.reserve(key_off[l->nkeys]);
    kR.reserve(key_off[l->nkeys]);
    kW.reserve(key_off[l->nkeys]);
    for (int k = 0; k < l->nkeys; k++) {
        kG.insert(kG.end(), h.key_G[k].begin(), h.key_G[k].end());
        kR.insert(kR.end(), h.key_row[k].begin(), h.key_row[k].end());
        kW.insert(kW.end(), h.key_W[k].begin(), h.key_W[k].end());
    }
    l->nW = nW;
    std::vector<double2> ones(std::max(nW, 1), make_double2(1.0, 0.0));
    hipError_t e = build_groups(h.key_M, h.key_nm, h.key_G, h.key_row, &h.key_W, A, nG, l->gi);
    // sub-keys for the grouped add: the j-th visit of a point in a key's
    // list goes to sub-key j, so no sub-key repeats a point
    std::vector<int> sk_M, sk_nm;
    std::vector<std::vector<int>> sk_G, sk_row;
    bool repeats = false;
    {
        std::vector<int> seen(nG, 0);
        for (int k = 0; k < l->nkeys; k++) {
            std::vector<int> sub_of;   // occurrence -> sub-key index
            for (size_t j = 0; j < h.key_G[k].size(); j++) {
                const int G = h.key_G[k][j];
                const int occ = seen[G]++;
                if (occ > 0) repeats = true;
                if (occ == (int)sub_of.size()) {
                    sub_of.push_back((int)sk_M.size());
                    sk_M.push_back(h.key_M[k]);
                    sk_nm.push_back(h.key_nm[k]);
                    sk_G.emplace_back();
                    sk_row.emplace_back();
                }
                sk_G[sub_of[occ]].push_back(G);
                sk_row[sub_of[occ]].push_back(h.key_row[k][j]);
            }
            for (int G : h.key_G[k]) seen[G] = 0;
        }
    }
    if (!repeats) {
        l->ga = l->gi;
        l->add_shares_groups = true;
    } else {
        l->add_shares_groups = false;
        if (e == hipSuccess) e = build_groups(sk_M, sk_nm, sk_G, sk_row, nullptr, A, nG, l->ga);
    }
    std::vector<float> A32(A, A + l->nvalues);

    // chunks of the add: consecutive covered points, at most kAddChunk of
    // them and kAddFuns functions of distinct blocks; each entry's first
    // function in its chunk
    std::vector<int> ch_i0{0}, ch_foff{0}, ch_col;
    std::vector<unsigned char> ent_f(h.ent.size(), 0);
    bool chunks_ok = true;
    {
        const long ncov = (long)h.cov_G.size();
        std::vector<int> cur, cur_f;   // the chunk's blocks (Mnm) and their first function
        std::vector<int> add;
        int nfun = 0;
        long i = 0;
        while (i < ncov && chunks_ok) {
            cur.clear();
            cur_f.clear();
            nfun = 0;
            const long start = i;
            while (i < ncov && i - start < kAddChunk) {
                add.clear();
                int add_f = 0;
                for (int e = h.cov_ptr[i]; e < h.cov_ptr[i + 1]; e++) {
                    const int Mnm = h.ent[e].y;
                    if (std::find(cur.begin(), cur.end(), Mnm) == cur.end() &&
                        std::find(add.begin(), add.end(), Mnm) == add.end()) {
                        add.push_back(Mnm);
                        add_f += Mnm & 15;
                    }
                }
                if (nfun + add_f > kAddFuns) {
                    if (i == start) chunks_ok = false;
                    break;
                }
                for (int Mnm : add) {
                    cur.push_back(Mnm);
                    cur_f.push_back(nfun);
                    for (int m = 0; m < (Mnm & 15); m++) ch_col.push_back((Mnm >> 4) + m);
                    nfun += Mnm & 15;
                }
                for (int e = h.cov_ptr[i]; e < h.cov_ptr[i + 1]; e++)
                    ent_f[e] = (unsigned char)cur_f[std::find(cur.begin(), cur.end(), h.ent[e].y) -
                                                    cur.begin()];
                i++;
            }
            ch_i0.push_back((int)i);
            ch_foff.push_back((int)ch_col.size());
        }
    }
    l->nchunks = chunks_ok ? (long)ch_i0.size() - 1 : 0;

#define UP(dst, src, n) \
    if (e == hipSuccess) e = upload(&l->dst, src, n)
    UP(A64, A, l->nvalues);
    UP(A32, A32.data(), l->nvalues);
    UP(ptr, h.ptr.data(), h.ptr.size());
    UP(ent, h.ent.data(), h.ent.size());
    UP(cov_G, h.cov_G.data(), h.cov_G.size());
    UP(cov_ptr, h.cov_ptr.data(), h.cov_ptr.size());
    UP(key_M, h.key_M.data(), h.key_M.size());
    UP(key_nm, h.key_nm.data(), h.key_nm.size());
    UP(key_off, key_off.data(), key_off.size());
    UP(key_G, kG.data(), kG.size());
    UP(key_row, kR.data(), kR.size());
    UP(ent_W, h.ent_W.data(), h.ent_W.size());
    UP(key_W, kW.data(), kW.size());
    UP(phase_W, ones.data(), ones.size());
    UP(ch_i0, ch_i0.data(), ch_i0.size());
    UP(ch_foff, ch_foff.data(), ch_foff.size());
    UP(ch_col, ch_col.data(), ch_col.size());
    UP(ent_f, ent_f.data(), ent_f.size());
#undef UP
    if (e != hipSuccess) {
        set_last_error(hipGetErrorString(e));
        gpd_lfc_destroy(l);
        return GPD_ERR_HIP;
    }
    *out = l;
    return GPD_OK;
}

extern "C" int gpd_lfc_integrate(gpd_lfc* l, int dtype, long nx, const void* d_a_xG,
                                 void* d_c_xM, void* stream)
{
    GPD_REQUIRE(l, GPD_ERR_ARG, "null lfc");
    GPD_REQUIRE(nx >= 0, GPD_ERR_ARG, "negative batch");
    if (nx == 0 || l->nkeys == 0) return GPD_OK;
    GPD_REQUIRE(d_a_xG && d_c_xM, GPD_ERR_ARG, "null array");
    hipStream_t st = (hipStream_t)stream;
    if (dtype == GPD_F64)
        return lfc_integrate_exact<double>(l, nx, (const double*)d_a_xG, (double*)d_c_xM, st);
    if (dtype == GPD_C128)
        return lfc_integrate_exact<double2>(l, nx, (const double2*)d_a_xG, (double2*)d_c_xM, st);
    if (dtype == GPD_F32) {
        const LfcGroups& gs = l->gi;
        if (gs.ngroups == 0) return GPD_OK;
        const long nbb = (nx + 31) / 32;
        // segments per group: about kSegTarget workgroups in all, each at
        // least a few chunks of 64 points
        constexpr long kSegTarget = 4096, kMinChunks = 8;
        const long chunks = (gs.npts_total + 63) / 64;
        long nseg = (kSegTarget + nbb * gs.ngroups - 1) / (nbb * gs.ngroups);
        nseg = std::max(1L, std::min(nseg, chunks / (kMinChunks * gs.ngroups)));
        if (nseg > 1) {
            const size_t need = (size_t)gs.ngroups * nseg * nx * gs.nfmax;
            if (need > l->seg_part_n) {
                // grown outside any graph capture: a batch size's first call
                if (l->seg_part) (void)hipFree(l->seg_part);
                l->seg_part = nullptr;
                l->seg_part_n = 0;
                GPD_CHECK_HIP(hipMalloc((void**)&l->seg_part, need * sizeof(float)));
                l->seg_part_n = need;
            }
        }
        const long nwork = nbb * gs.ngroups * nseg;
        hipLaunchKernelGGL(lfc_integrate_mfma_kernel, dim3(xcd_grid_size(nwork)), dim3(256), 0,
                           st, (const float*)d_a_xG, (float*)d_c_xM, l->nG, l->Mmax, nx, l->dv,
                           gs.ngroups, gs.nfmax, gs.grp_off, gs.grp_nf, gs.grp_fM, gs.grp_G,
                           gs.grp_A32, (int)nseg, l->seg_part);
        int rc = last_error_to_status(hipGetLastError());
        if (rc || nseg == 1) return rc;
        const long n = (long)gs.ngroups * nx * gs.nfmax;
        hipLaunchKernelGGL(lfc_integrate_segments_kernel, dim3((unsigned)((n + 255) / 256)),
                           dim3(256), 0, st, l->seg_part, (float*)d_c_xM, l->Mmax, nx,
                           gs.ngroups, gs.nfmax, (int)nseg, gs.grp_nf, gs.grp_fM);
        return last_error_to_status(hipGetLastError());
    }
    GPD_REQUIRE(false, GPD_ERR_ARG, "unknown dtype");
}

extern "C" int gpd_lfc_set_phases(gpd_lfc* l, const double* phase_W)
{
    GPD_REQUIRE(l, GPD_ERR_ARG, "null lfc");
    if (l->nW == 0) return GPD_OK;
    std::vector<double2> ph(l->nW);
    for (int W = 0; W < l->nW; W++)
        ph[W] = phase_W ? make_double2(phase_W[2 * W], phase_W[2 * W + 1])
                        : make_double2(1.0, 0.0);
    // the grouped exact integrate takes one phase per group point: all the
    // keys of a group must see equal phases there (they do when the keys
    // are one atom's functions, whose volumes share the image displacement)
    bool shared = true;
    for (const auto& pr : l->gi.phase_pairs) {
        const double2 x = ph[pr.first], y = ph[pr.second];
        if (memcmp(&x, &y, sizeof(double2)) != 0) {
            shared = false;
            break;
        }
    }
    // kernels still running on any stream may read the current phases:
    // let them finish before the table is replaced
    hipError_t e = hipDeviceSynchronize();
    if (e == hipSuccess)
        e = hipMemcpy(l->phase_W, ph.data(), sizeof(double2) * l->nW, hipMemcpyHostToDevice);
    if (e != hipSuccess) {
        set_last_error(hipGetErrorString(e));
        return GPD_ERR_HIP;
    }
    l->grp_phase_shared = shared;
    return GPD_OK;
}

extern "C" int gpd_lfc_set_launch(gpd_lfc* l, int exact_bands)
{
    GPD_REQUIRE(l, GPD_ERR_ARG, "null lfc");
    GPD_REQUIRE(exact_bands == 0 || exact_bands == 16 || exact_bands == 32 || exact_bands == 64,
                GPD_ERR_ARG, "the launch shape must be 0 (automatic), 16, 32 or 64");
    l->exact_nbb = exact_bands;
    return GPD_OK;
}

extern "C" int gpd_lfc_add(gpd_lfc* l, int dtype, long nx, const void* d_c_xM, void* d_a_xG,
                           void* stream)
{
    GPD_REQUIRE(l, GPD_ERR_ARG, "null lfc");
    GPD_REQUIRE(nx >= 0, GPD_ERR_ARG, "negative batch");
    if (nx == 0 || l->ncov == 0) return GPD_OK;
    GPD_REQUIRE(d_a_xG && d_c_xM, GPD_ERR_ARG, "null array");
    hipStream_t st = (hipStream_t)stream;
    if (dtype == GPD_F64) return lfc_add_exact_f64(l, nx, (const double*)d_c_xM, (double*)d_a_xG, st);
    if (dtype == GPD_F32) return lfc_add_f32(l, nx, (const float*)d_c_xM, (float*)d_a_xG, st);
    if (dtype == GPD_C128 && l->nchunks > 0) {
        constexpr int NB = 8;
        const long nwork = l->nchunks * ((nx + NB - 1) / NB);
        hipLaunchKernelGGL((lfc_add_chunk_z_kernel<NB>), dim3(xcd_grid_size(nwork)), dim3(256), 0,
                           st, (const double2*)d_c_xM, (double2*)d_a_xG, l->nG, l->Mmax, nx,
                           l->nchunks, l->ch_i0, l->ch_foff, l->ch_col, l->A64, l->cov_G,
                           l->cov_ptr, l->ent, l->ent_f, l->ent_W, l->phase_W);
        return last_error_to_status(hipGetLastError());
    }
    if (dtype == GPD_C128) {
        constexpr int NBT = 4;
        const long n = ((nx + NBT - 1) / NBT) * l->ncov;
        hipLaunchKernelGGL((lfc_add_z_kernel<NBT>), dim3((n + 255) / 256), dim3(256), 0, st,
                           (const double2*)d_c_xM, (double2*)d_a_xG, l->nG, l->Mmax, nx, l->ncov,
                           l->A64, l->cov_G, l->cov_ptr, l->ent, l->ent_W, l->phase_W);
        return last_error_to_status(hipGetLastError());
    }
    GPD_REQUIRE(false, GPD_ERR_ARG, "unknown dtype");
}
