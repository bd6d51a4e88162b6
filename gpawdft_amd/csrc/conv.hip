// 3-D convolution kernels of the learned preconditioner (gfx950).
//
// Periodic 3x3x3 convolutions on grids (B, C, D, H, W), C-contiguous, the
// layout of a batch of band grids with a channel axis.  No counterpart in
// the reference: these serve the learned correction that stands beside the
// multigrid preconditioner.
//
//   forward:        y[b,o,p] = bias[o] + sum_{i,t} W[o,i,t] x[b,i,p+d_t]
//   backward data:  gx[b,i,p] = sum_{o,t} W[o,i,t] gy[b,o,p-d_t]
//   backward weight gW[o,i,t] = sum_{b,p} gy[b,o,p] x[b,i,p+d_t]
//   backward bias   gb[o]     = sum_{b,p} gy[b,o,p]
// with d_t = (t/9 - 1, (t/3)%3 - 1, t%3 - 1) and periodic wrap.  Weights are
// FP32 (o, i, 27).  An output of the data kernels is one chain of FMAs over
// channels and, within them, taps.  The weight kernel sums chunks of the points,
// each as 256 chains of FMAs, then the chunks, in a fixed order without atomics.
// All FP32 with FMA.
#include <algorithm>

#include "common.hpp"

namespace gpd {

struct ConvDims {
    int B, Cin, Cout, D, H, W;
};

__device__ __forceinline__ int wrapp(int i, int n) { return i < 0 ? i + n : (i >= n ? i - n : i); }

// What becomes of a result: added to the array (accumulate), a leaky ReLU
// (forward: slope for results <= 0, 1 for none), or the ReLU's derivative
// (backward data: slope where act, the layer's input, is <= 0; null for none).
struct ConvEpi {
    int accumulate;
    float slope;
    const float* act;
};

template <int MODE>
__device__ __forceinline__ void finish(const ConvEpi& ep, float v, long p, float* __restrict__ y)
{
    if (MODE == 0) v = v > 0.f ? v : ep.slope * v;
    else if (ep.act) v = ep.act[p] > 0.f ? v : ep.slope * v;
    y[p] = ep.accumulate ? y[p] + v : v;
}

// wrap any index of a tile that overhangs a periodic axis
__device__ __forceinline__ int wrapm(int i, int n)
{
    if (i < 0) return i + n;
    if (i >= n) i -= n;
    if (i >= n) i %= n;   // grids smaller than the overhang
    return i;
}

// ------------------------------------------------------------------ //
// Data kernels.  mode 0: forward (weight index o*Cin*27 + i*27 + t); mode 1:
// backward data (roles of o and i swapped, taps mirrored).
//
// Implicit GEMM on v_mfma_f32_16x16x4_f32: A = weights (16 output channels
// x 4 terms), B = inputs (4 terms x 16 points of 8 x 2); a term is one tap of
// one input channel, channels outermost.  The instruction is a chain of four
// FMAs in the order of its terms (equal to it bit for bit, denormals and
// signed zeros included), so an output is one chain over channels and taps.
// A workgroup takes 8 x 8 x TZ points (x, y, z) and MO blocks of 16 output
// channels, a wave TZ blocks of 16 points.  kXC input channels at a time are
// in LDS, points with their halo and the channels' weights; the next ones'
// loads are in flight meanwhile.  Four channels are 27 steps, whose offsets a
// lane keeps in registers.
// Bound by the matrix unit (an MFMA takes 32 clocks and needs 1 / MO + 1 / TZ
// reads of 4 B a lane), with little else in the way once the points fill
// the chip.  Batch 8, 32^3, 16 -> 32 channels 93 us (78 TFLOP/s) and its
// gradient 85; 16^3, 32 -> 64 50, 64 -> 32 51 us.  A point and 16 outputs a
// thread on the vector units took 225, 220, 156 and 304 us.

constexpr int kXC = 8;              // input channels in LDS
constexpr int kHX = 10, kHY = 10;   // tile with halo along axes 2 and 1

template <int MODE, int TZ, int MO>
__global__ __launch_bounds__(256) void conv3d_kernel(const float* __restrict__ x,
                                                    const float* __restrict__ Wt,
                                                    const float* __restrict__ bias,
                                                    float* __restrict__ y, ConvDims d,
                                                     ConvEpi ep)
{
    constexpr int NPT = kHX * kHY * (TZ + 2);
    constexpr int PPT = (NPT + 255) / 256;
    // weights in memory: runs of an output's kXC channels and taps (mode 0),
    // of an input channel's outputs and taps (mode 1); in LDS the terms of
    // an output, at a pitch that keeps 16 outputs on different banks
    constexpr int WRUNS = MODE == 0 ? 16 * MO : kXC;
    constexpr int WRUN = 27 * (MODE == 0 ? kXC : 16 * MO);
    constexpr int WPR = (WRUN + 255) / 256;
    constexpr int WP = 27 * kXC + 1;
    __shared__ float xs[kXC * NPT];
    __shared__ float ws[16 * MO * WP];

    const int P = d.D * d.H * d.W;
    // channels seen by this kernel: nin inputs, nout outputs
    const int nin = MODE == 0 ? d.Cin : d.Cout;
    const int nout = MODE == 0 ? d.Cout : d.Cin;
    const int ntx = (d.W + 7) / 8, nty = (d.H + 7) / 8, ntz = (d.D + TZ - 1) / TZ;
    const int nob = (nout + 16 * MO - 1) / (16 * MO);
    const long nwork = (long)ntz * nty * ntx * nob;
    const long w = xcd_work_index(blockIdx.x, nwork);
    if (w < 0) return;
    const int o0 = (int)(w % nob) * 16 * MO;
    long r = w / nob;
    const int x0 = (int)(r % ntx) * 8;
    r /= ntx;
    const int y0 = (int)(r % nty) * 8;
    r /= nty;
    const int z0 = (int)r * TZ;
    const int b = blockIdx.z;
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;

    // this thread's points of the tile with halo
    const float* xb = x + (long)b * nin * P;
    unsigned off[PPT];
#pragma unroll
    for (int e = 0; e < PPT; e++) {
        const int s = min(tid + 256 * e, NPT - 1);
        const int gx = wrapm(x0 - 1 + s % kHX, d.W);
        const int gy = wrapm(y0 - 1 + s / kHX % kHY, d.H);
        const int gz = wrapm(z0 - 1 + s / (kHX * kHY), d.D);
        off[e] = (gz * d.H + gy) * d.W + gx;
    }
    float xr[kXC][PPT], wr[WRUNS][WPR];
    auto load = [&](int c0) {
#pragma unroll
        for (int c = 0; c < kXC; c++) {
            const float* p = xb + (long)min(c0 + c, nin - 1) * P;
#pragma unroll
            for (int e = 0; e < PPT; e++) xr[c][e] = p[off[e]];
        }
        // outputs and channels past the last take the address of the last
#pragma unroll
        for (int q = 0; q < WRUNS; q++) {
            const float* p = MODE == 0 ? Wt + ((long)min(o0 + q, nout - 1) * d.Cin + c0) * 27
                                       : Wt + ((long)min(c0 + q, nin - 1) * d.Cin + o0) * 27;
            const int last = 27 * (MODE == 0 ? nin - c0 : nout - o0) - 1;
#pragma unroll
            for (int e = 0; e < WPR; e++)
                wr[q][e] = p[(unsigned)min(min(tid + 256 * e, WRUN - 1), last)];
        }
    };

    // this lane's column (point) and k (term) in the MFMA operands: its
    // block of points j lies j pairs of rows further
    const int k = lane / 16, px = lane % 8, py = lane / 8 % 2;
    const int z = wave * TZ / 4, yy = wave * TZ % 4 * 2 + py;
    const float* xl[27];
#pragma unroll
    for (int st = 0; st < 27; st++) {
        const int q = 4 * st + k, t = MODE == 0 ? q % 27 : 26 - q % 27;
        xl[st] = xs + q / 27 * NPT + ((z + t / 9) * kHY + yy + t / 3 % 3) * kHX + px + t % 3;
    }
    const float* wl = ws + lane % 16 * WP + k;

    f32x4 acc[MO][TZ];
#pragma unroll
    for (int m = 0; m < MO; m++)
#pragma unroll
        for (int j = 0; j < TZ; j++) acc[m][j] = f32x4{0.f, 0.f, 0.f, 0.f};

    load(0);
    for (int c0 = 0; c0 < nin; c0 += kXC) {
        lds_barrier();
#pragma unroll
        for (int c = 0; c < kXC; c++)
#pragma unroll
            for (int e = 0; e < PPT; e++) {
                const int s = tid + 256 * e;
                if (s < NPT) xs[c * NPT + s] = c0 + c < nin ? xr[c][e] : 0.f;
            }
#pragma unroll
        for (int q = 0; q < WRUNS; q++)
#pragma unroll
            for (int e = 0; e < WPR; e++) {
                const int s = tid + 256 * e;
                const bool ok = MODE == 0 ? o0 + q < nout && s < 27 * (nin - c0)
                                          : c0 + q < nin && s < 27 * (nout - o0);
                const int at = MODE == 0 ? q * WP + s : s / 27 * WP + q * 27 + s % 27;
                if (s < WRUN) ws[at] = ok ? wr[q][e] : 0.f;
            }
        if (c0 + kXC < nin) load(c0 + kXC);
        lds_barrier();
#pragma unroll
        for (int g = 0; g < kXC / 4; g++) {
            if (c0 + 4 * g >= nin) break;
#pragma unroll
            for (int st = 0; st < 27; st++) {
                float wv[MO], xv[TZ];
#pragma unroll
                for (int m = 0; m < MO; m++) wv[m] = wl[16 * m * WP + 108 * g + 4 * st];
#pragma unroll
                for (int j = 0; j < TZ; j++) xv[j] = xl[st][4 * g * NPT + 2 * j * kHX];
#pragma unroll
                for (int m = 0; m < MO; m++)
#pragma unroll
                    for (int j = 0; j < TZ; j++)
                        acc[m][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[m], xv[j], acc[m][j],
                                                                         0, 0, 0);
            }
        }
    }
    // D: column = point lane % 16, row = output channel 4 (lane / 16) + v
    float* yb = y + (long)b * nout * P;
#pragma unroll
    for (int j = 0; j < TZ; j++) {
        const int gz = z0 + z, gy = y0 + yy + 2 * j, gx = x0 + px;
        if (gz >= d.D || gy >= d.H || gx >= d.W) continue;
        float* dst = yb + ((long)gz * d.H + gy) * d.W + gx;
#pragma unroll
        for (int m = 0; m < MO; m++)
#pragma unroll
            for (int v = 0; v < 4; v++) {
                const int o = o0 + 16 * m + 4 * k + v;
                if (o >= nout) continue;
                const float val = acc[m][j][v] + ((MODE == 0 && bias) ? bias[o] : 0.f);
                finish<MODE>(ep, val, dst - y + (long)o * P, y);
            }
    }
}

// One or two output channels: a matrix block would be mostly idle, so the
// products are FMAs.  A workgroup takes 16 x 8 x 8 points, a thread four
// neighbours along x of all NO channels, and one input channel is in LDS at
// a time (the next one's loads in flight): nine runs of six values feed
// 108 NO FMAs, each output the chain of the kernel above.  16 -> 1 channels,
// batch 8 of 64^3: 69 us (166 with a point a thread and every tap from
// memory; 134 MB read).

template <int MODE, int NO>
__global__ __launch_bounds__(256) void conv3d_few_kernel(const float* __restrict__ x,
                                                        const float* __restrict__ Wt,
                                                        const float* __restrict__ bias,
                                                        float* __restrict__ y, ConvDims d,
                                                         ConvEpi ep)
{
    constexpr int HX = 18, PX = 20, HY = 10, HZ = 10;
    constexpr int NPT = HX * HY * HZ;
    constexpr int PPT = (NPT + 255) / 256;
    __shared__ __attribute__((aligned(16))) float xs[PX * HY * HZ];

    const int P = d.D * d.H * d.W;
    const int nin = MODE == 0 ? d.Cin : d.Cout;
    const int ntx = (d.W + 15) / 16, nty = (d.H + 7) / 8, ntz = (d.D + 7) / 8;
    const long nwork = (long)ntz * nty * ntx;
    const long w = xcd_work_index(blockIdx.x, nwork);
    if (w < 0) return;
    const int x0 = (int)(w % ntx) * 16;
    long r = w / ntx;
    const int y0 = (int)(r % nty) * 8;
    r /= nty;
    const int z0 = (int)r * 8;
    const int b = blockIdx.z;
    const int tid = threadIdx.x;

    const float* xb = x + (long)b * nin * P;
    int off[PPT], slot[PPT];
#pragma unroll
    for (int e = 0; e < PPT; e++) {
        const int s = min(tid + 256 * e, NPT - 1);
        const int gx = wrapm(x0 - 1 + s % HX, d.W);
        const int gy = wrapm(y0 - 1 + s / HX % HY, d.H);
        const int gz = wrapm(z0 - 1 + s / (HX * HY), d.D);
        off[e] = (gz * d.H + gy) * d.W + gx;
        slot[e] = s / HX * PX + s % HX;
    }
    float xr[PPT];
    auto load = [&](int c) {
#pragma unroll
        for (int e = 0; e < PPT; e++) xr[e] = xb[(long)c * P + off[e]];
    };
    const int tx = tid % 4 * 4, ty = tid / 4 % 8, tz = tid / 32;
    const float* xl = xs + (tz * HY + ty) * PX + tx;
    float acc[NO][4];
#pragma unroll
    for (int o = 0; o < NO; o++)
#pragma unroll
        for (int j = 0; j < 4; j++) acc[o][j] = 0.f;
    load(0);
    for (int c = 0; c < nin; c++) {
        lds_barrier();
#pragma unroll
        for (int e = 0; e < PPT; e++) xs[slot[e]] = xr[e];
        if (c + 1 < nin) load(c + 1);
        lds_barrier();
#pragma unroll
        for (int q = 0; q < 9; q++) {
            // taps 3 q .. 3 q + 2: run of the points x - 1 .. x + 4 of a row
            const int row = MODE == 0 ? q : 8 - q;
            const float* f = xl + (row / 3 * HY + row % 3) * PX;
            const float4 lo = *(const float4*)f;
            const float2 hi = *(const float2*)(f + 4);
            const float v[6] = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y};
#pragma unroll
            for (int o = 0; o < NO; o++) {
                const float* wr = MODE == 0 ? Wt + ((long)o * d.Cin + c) * 27
                                            : Wt + ((long)c * d.Cin + o) * 27;
#pragma unroll
                for (int dx = 0; dx < 3; dx++) {
                    const float wv = wr[3 * q + dx];
#pragma unroll
                    for (int j = 0; j < 4; j++)
                        acc[o][j] = __builtin_fmaf(wv, v[j + (MODE == 0 ? dx : 2 - dx)],
                                                   acc[o][j]);
                }
            }
        }
    }
    const int gz = z0 + tz, gy = y0 + ty;
    if (gz >= d.D || gy >= d.H) return;
    float* yb = y + (long)b * NO * P + ((long)gz * d.H + gy) * d.W + x0 + tx;
#pragma unroll
    for (int o = 0; o < NO; o++) {
        const float bo = (MODE == 0 && bias) ? bias[o] : 0.f;
#pragma unroll
        for (int j = 0; j < 4; j++) {
            if (x0 + tx + j >= d.W) continue;
            finish<MODE>(ep, acc[o][j] + bo, yb - y + (long)o * P + j, y);
        }
    }
}

// One or two input channels: all 27 NI terms at once, in the order of the
// kernel above.  A workgroup takes 16 x 8 x 8 points, a wave two z-planes, and the weights
// of a block of 16 output channels stay in registers.  A lane reads the
// values of its taps at fixed offsets from its point.  Bound by the stores:
// 2 -> 16 channels, batch 8 of 64^3, 134 MB written: 60 us (127 with a point a
// thread); 1 -> 16 channels 37 us (65).

template <int MODE, int NI>
__global__ __launch_bounds__(256) void conv3d_in_kernel(const float* __restrict__ x,
                                                       const float* __restrict__ Wt,
                                                       const float* __restrict__ bias,
                                                       float* __restrict__ y, ConvDims d,
                                                        ConvEpi ep)
{
    constexpr int HX = 18, HY = 10, HZ = 10;
    constexpr int NPT = HX * HY * HZ;
    constexpr int PPT = (NPT + 255) / 256;
    constexpr int NK = (27 * NI + 3) / 4;
    __shared__ float xs[NI * NPT + 1];   // and a zero for the terms past the last

    const int P = d.D * d.H * d.W;
    const int nout = MODE == 0 ? d.Cout : d.Cin;
    const int ntx = (d.W + 15) / 16, nty = (d.H + 7) / 8, ntz = (d.D + 7) / 8;
    const long nwork = (long)ntz * nty * ntx;
    const long w = xcd_work_index(blockIdx.x, nwork);
    if (w < 0) return;
    const int x0 = (int)(w % ntx) * 16;
    long r = w / ntx;
    const int y0 = (int)(r % nty) * 8;
    r /= nty;
    const int z0 = (int)r * 8;
    const int b = blockIdx.z;
    const int tid = threadIdx.x, wave = tid / 64, lane = tid % 64;
    const int k = lane / 16, px = lane % 16;

    const float* xb = x + (long)b * NI * P;
    float xr[NI][PPT];
#pragma unroll
    for (int e = 0; e < PPT; e++) {
        const int s = min(tid + 256 * e, NPT - 1);
        const int gx = wrapm(x0 - 1 + s % HX, d.W);
        const int gy = wrapm(y0 - 1 + s / HX % HY, d.H);
        const int gz = wrapm(z0 - 1 + s / (HX * HY), d.D);
#pragma unroll
        for (int c = 0; c < NI; c++) xr[c][e] = xb[(long)c * P + (gz * d.H + gy) * d.W + gx];
    }
    // tap of this lane in each step: its offset in the tile
    int toff[NK];
#pragma unroll
    for (int s = 0; s < NK; s++) {
        const int q = 4 * s + k, t = MODE == 0 ? q % 27 : 26 - q % 27;
        toff[s] = q < 27 * NI ? q / 27 * NPT + (t / 9 * HY + t / 3 % 3) * HX + t % 3 + px : -1;
    }
    if (tid == 0) xs[NI * NPT] = 0.f;
#pragma unroll
    for (int e = 0; e < PPT; e++) {
        const int s = tid + 256 * e;
#pragma unroll
        for (int c = 0; c < NI; c++)
            if (s < NPT) xs[c * NPT + s] = xr[c][e];
    }
    __syncthreads();
    float* yb = y + (long)b * nout * P;
    for (int o0 = 0; o0 < nout; o0 += 16) {
        float wv[NK];
        const int o = min(o0 + px, nout - 1);
#pragma unroll
        for (int s = 0; s < NK; s++) {
            const int q = min(4 * s + k, 27 * NI - 1);
            const float v = MODE == 0 ? Wt[((long)o * NI + q / 27) * 27 + q % 27]
                                      : Wt[((long)(q / 27) * d.Cin + o) * 27 + q % 27];
            wv[s] = 4 * s + k < 27 * NI ? v : 0.f;
        }
        float bo[4];
#pragma unroll
        for (int v = 0; v < 4; v++)
            bo[v] = (MODE == 0 && bias) ? bias[min(o0 + 4 * k + v, nout - 1)] : 0.f;
        // four rows of 16 points at a time
#pragma unroll 1
        for (int h = 0; h < 4; h++) {
            const int lz = 2 * wave + h / 2, ly = h % 2 * 4;
            f32x4 acc[4];
#pragma unroll
            for (int j = 0; j < 4; j++) acc[j] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int s = 0; s < NK; s++) {
                const bool term = 4 * s + 3 < 27 * NI || toff[s] >= 0;
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const int at = toff[s] + (lz * HY + ly + j) * HX;
                    acc[j] = __builtin_amdgcn_mfma_f32_16x16x4f32(
                        wv[s], xs[term ? at : NI * NPT], acc[j], 0, 0, 0);
                }
            }
            const int gz = z0 + lz, gx = x0 + px;
            if (gz >= d.D || gx >= d.W) continue;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const int gy = y0 + ly + j;
                if (gy >= d.H) continue;
                float* dst = yb + ((long)gz * d.H + gy) * d.W + gx;
#pragma unroll
                for (int v = 0; v < 4; v++) {
                    const int oo = o0 + 4 * k + v;
                    if (oo >= nout) continue;
                    finish<MODE>(ep, acc[j][v] + bo[v], dst - y + (long)oo * P, y);
                }
            }
        }
    }
}

// The few-channel kernel up to two outputs.  Otherwise 8 x 8 x 4 points and
// up to 32 output channels a workgroup (fewer bytes staged for each product)
// if that gives 1024 workgroups (batch 8 of 32^3, 32 outputs of 16 channels:
// forward 92 us, the gradient's 78; 102 and 99 with the small tiles), else 8 x 8
// x 2 points and 16 channels (batch 8 of 16^3, 64 -> 32: 51 us; 59 with four
// planes, 84 with 32 channels too).
template <int MODE>
static int launch_conv(const ConvDims& d, const float* x, const float* w, const float* bias,
                       float* y, const ConvEpi& ep, hipStream_t st)
{
    const int nout = MODE == 0 ? d.Cout : d.Cin;
    const auto tiles = [&](int tx, int ty, int tz) {
        return (long)((d.D + tz - 1) / tz) * ((d.H + ty - 1) / ty) * ((d.W + tx - 1) / tx);
    };
    const auto launch = [&](auto kernel, long nwork) {
        hipLaunchKernelGGL(kernel, dim3(xcd_grid_size(nwork), 1, d.B), dim3(256), 0, st, x, w,
                           bias, y, d, ep);
    };
    const int nin = MODE == 0 ? d.Cin : d.Cout;
    if (nin == 1) launch(conv3d_in_kernel<MODE, 1>, tiles(16, 8, 8));
    else if (nin == 2) launch(conv3d_in_kernel<MODE, 2>, tiles(16, 8, 8));
    else if (nout == 1) launch(conv3d_few_kernel<MODE, 1>, tiles(16, 8, 8));
    else if (nout == 2) launch(conv3d_few_kernel<MODE, 2>, tiles(16, 8, 8));
    else if (nout > 16 && d.B * tiles(8, 8, 4) * ((nout + 31) / 32) >= 1024)
        launch(conv3d_kernel<MODE, 4, 2>, tiles(8, 8, 4) * ((nout + 31) / 32));
    else if (nout <= 16 && d.B * tiles(8, 8, 4) >= 1024)
        launch(conv3d_kernel<MODE, 4, 1>, tiles(8, 8, 4));
    else
        launch(conv3d_kernel<MODE, 2, 1>, tiles(8, 8, 2) * ((nout + 15) / 16));
    return last_error_to_status(hipGetLastError());
}

// ------------------------------------------------------------------ //
// Weight gradient.  The B P points are cut into chunks, and a chunk's sum is
// 256 chains of FMAs, chain r over the points r, r + 256, .. of the chunk, then
// summed by halves (r and r + 128, r + 64, ..); the chunks are summed in order.
// This order is kept for its bits: an optimiser step takes the weights from
// them, and the next pass's results follow the weights.
//
// A thread carries a chain (workgroup: a chunk) of 9 taps, one dz, of OB outputs
// and IB inputs: 72 chains in registers (OB = 8) fed by 9 IB + OB loads, of which
// the next point's are in flight.  A channel's base is uniform, so that a point
// costs 33 instructions of index arithmetic for its 72 FMAs.  Bound by the
// vector units and the loads' way through the L1 in about equal parts, three
// workgroups a CU (two with 16 outputs a thread: no gain).  Batch 8: 64^3 2 ->
// 16 128 us and 16 -> 1 178, 32^3 16 -> 32 217, 32 -> 16 212, 16^3 32 -> 64 and
// 64 -> 32 119.  A workgroup a pair of channels took 609, 333, 1134, 1127, 637
// and 633; products on the matrix units, in another order, 126, 85, 106, 108, 69
// and 65.

constexpr int kWThreads = 256;

struct WgradDims {
    int B, Cin, Cout, D, H, W;
    int nchunk;
    long chunk;          // points of a chunk
    int sz, sy, sx;      // 256 points further along the grid
};

// I: byte offsets within an array, 32 bits where they fit
template <int OB, int IB, typename I>
__global__ __launch_bounds__(kWThreads, 3) void wgrad_kernel(const float* __restrict__ x,
                                                             const float* __restrict__ gy,
                                                             float* __restrict__ part,
                                                             float* __restrict__ partb,
                                                             WgradDims d)
{
    constexpr int NV = 9 * OB * IB;          // chains, and those of the bias
    __shared__ float red[2][NV + OB][64];
    const int nob = (d.Cout + OB - 1) / OB, nib = (d.Cin + IB - 1) / IB;
    const long w = xcd_work_index(blockIdx.x, (long)d.nchunk * 3 * nib * nob);
    if (w < 0) return;
    const int o0 = (int)(w % nob) * OB;
    long r = w / nob;
    const int i0 = (int)(r % nib) * IB;
    r /= nib;
    const int dz = (int)(r % 3), chunk = (int)(r / 3);
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid / 64), lane = tid % 64;
    const long P = (long)d.D * d.H * d.W;
    const long q0 = chunk * d.chunk, q1 = min((long)d.B * P, q0 + d.chunk);
    // of the chains past the chunk: the last point, not used
    const long q = min(q0 + tid, q1 - 1);
    int left = q0 + tid < q1 ? (int)((q1 - q0 - tid + kWThreads - 1) / kWThreads) : 0;
    int b = (int)(q / P), px, py, pz;
    {
        const int p = (int)(q % P);
        px = p % d.W;
        py = p / d.W % d.H;
        pz = p / d.W / d.H;
    }
    auto at = [](const float* base, I byte) { return *(const float*)((const char*)base + byte); };
    float xn[IB][9], gn[OB];
    auto load = [&]() {
        const I xb = (I)b * (I)(4 * P) * (I)d.Cin, gb = (I)b * (I)(4 * P) * (I)d.Cout;
        const int z = wrapp(pz + dz - 1, d.D);
        const int ry[3] = {wrapp(py - 1, d.H), py, wrapp(py + 1, d.H)};
        const int cx[3] = {wrapp(px - 1, d.W), px, wrapp(px + 1, d.W)};
#pragma unroll
        for (int t = 0; t < 9; t++) {
            const I off = xb + 4 * (I)((z * d.H + ry[t / 3]) * d.W + cx[t % 3]);
#pragma unroll
            for (int i = 0; i < IB; i++) xn[i][t] = at(x + min(i0 + i, d.Cin - 1) * P, off);
        }
        const I off = gb + 4 * (I)((pz * d.H + py) * d.W + px);
#pragma unroll
        for (int o = 0; o < OB; o++) gn[o] = at(gy + min(o0 + o, d.Cout - 1) * P, off);
    };
    auto advance = [&]() {
        px += d.sx;
        if (px >= d.W) px -= d.W, py++;
        py += d.sy;
        if (py >= d.H) py -= d.H, pz++;
        pz += d.sz;
        while (pz >= d.D) pz -= d.D, b++;
    };
    float acc[NV + OB];
#pragma unroll
    for (int v = 0; v < NV + OB; v++) acc[v] = 0.f;
    // the bias sums are those of one block of inputs and one dz
    const bool bias = i0 == 0 && dz == 1;
    load();
    while (left > 0) {
        float xv[IB][9], g[OB];
#pragma unroll
        for (int i = 0; i < IB; i++)
#pragma unroll
            for (int t = 0; t < 9; t++) xv[i][t] = xn[i][t];
#pragma unroll
        for (int o = 0; o < OB; o++) g[o] = gn[o];
        left--;
        if (left > 0) advance();
        load();                              // (past the last: the last again)
#pragma unroll
        for (int i = 0; i < IB; i++)
#pragma unroll
            for (int t = 0; t < 9; t++)
#pragma unroll
                for (int o = 0; o < OB; o++) {
                    float& s = acc[(o * IB + i) * 9 + t];
                    s = __builtin_fmaf(g[o], xv[i][t], s);
                }
        if (bias)
#pragma unroll
            for (int o = 0; o < OB; o++) acc[NV + o] += g[o];
    }
    // chains r and r + 128, then r + 64, by waves; the rest by a thread a sum,
    // which reads a row turned by its number so that no two share a bank
    if (wave >= 2)
#pragma unroll
        for (int v = 0; v < NV + OB; v++) red[wave - 2][v][lane] = acc[v];
    __syncthreads();
    if (wave < 2)
#pragma unroll
        for (int v = 0; v < NV + OB; v++) {
            acc[v] += red[wave][v][lane];
            if (wave == 1) red[1][v][lane] = acc[v];
        }
    __syncthreads();
    if (wave == 0)
#pragma unroll
        for (int v = 0; v < NV + OB; v++) red[0][v][(lane + v) % 64] = acc[v] + red[1][v][lane];
    __syncthreads();
    if (tid >= NV + OB) return;
    float sum[64];
#pragma unroll
    for (int k = 0; k < 64; k++) sum[k] = red[0][tid][(k + tid) % 64];
#pragma unroll
    for (int s = 32; s > 0; s >>= 1)
#pragma unroll
        for (int k = 0; k < s; k++) sum[k] += sum[k + s];
    if (tid < NV) {
        const int o = o0 + tid / (9 * IB), i = i0 + tid / 9 % IB;
        if (o < d.Cout && i < d.Cin)
            part[(((long)chunk * d.Cout + o) * d.Cin + i) * 27 + 9 * dz + tid % 9] = sum[0];
    } else if (bias && o0 + tid - NV < d.Cout) {
        partb[(long)chunk * d.Cout + o0 + tid - NV] = sum[0];
    }
}

// gW and gb = sums over the chunks, in order
__global__ __launch_bounds__(64) void wgrad_reduce_kernel(const float* __restrict__ part,
                                                          const float* __restrict__ partb,
                                                          float* __restrict__ gW,
                                                          float* __restrict__ gb, long n, int Cout,
                                                          int nchunk)
{
    const long k = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (k >= n + (gb ? Cout : 0)) return;
    const float* p = k < n ? part + k : partb + (k - n);
    const long step = k < n ? n : Cout;
    float s = 0.f;
#pragma unroll 16
    for (int c = 0; c < nchunk; c++) s += p[c * step];
    if (k < n) gW[k] = s;
    else gb[k - n] = s;
}

// A block of outputs by one input; for one or two outputs one of them by four
// inputs (by eight, 64^3 16 -> 1 took 169 us, but one sample of 16^3, with six
// workgroups, 36 with its launches, 24 now).
static int launch_wgrad(const ConvDims& c, const float* x, const float* gy, float* gw, float* gb,
                        hipStream_t st)
{
    // chunks of at least 4096 points, and so that a pair of channels and a
    // chunk are about 2048 items
    const long P = (long)c.D * c.H * c.W, npts = c.B * P, pairs = (long)c.Cout * c.Cin;
    long nchunk = std::max(1L, std::min((2048 + pairs - 1) / pairs, npts / 4096));
    WgradDims d = {c.B, c.Cin, c.Cout, c.D, c.H, c.W};
    d.chunk = (npts + nchunk - 1) / nchunk;
    nchunk = (npts + d.chunk - 1) / d.chunk;
    d.nchunk = (int)nchunk;
    d.sx = kWThreads % c.W;
    d.sy = kWThreads / c.W % c.H;
    d.sz = kWThreads / c.W / c.H;
    const long n = pairs * 27;
    float* part = nullptr;
    hipError_t e = hipMallocAsync((void**)&part, sizeof(float) * (n + c.Cout) * nchunk, st);
    if (e != hipSuccess) {
        set_last_error(hipGetErrorString(e));
        return GPD_ERR_HIP;
    }
    float* partb = part + n * nchunk;
    const auto launch = [&](auto kernel, int ob, int ib) {
        const long nwork = nchunk * 3 * ((c.Cin + ib - 1) / ib) * ((c.Cout + ob - 1) / ob);
        hipLaunchKernelGGL(kernel, dim3(xcd_grid_size(nwork)), dim3(kWThreads), 0, st, x, gy, part,
                           partb, d);
    };
    const bool fits = 4 * npts * std::max(c.Cin, c.Cout) < (1L << 32);
    if (c.Cout <= 2)
        fits ? launch(wgrad_kernel<1, 4, unsigned>, 1, 4) : launch(wgrad_kernel<1, 4, size_t>, 1, 4);
    else
        fits ? launch(wgrad_kernel<8, 1, unsigned>, 8, 1) : launch(wgrad_kernel<8, 1, size_t>, 8, 1);
    int rc = last_error_to_status(hipGetLastError());
    if (!rc) {
        hipLaunchKernelGGL(wgrad_reduce_kernel, dim3((unsigned)((n + c.Cout + 63) / 64)), dim3(64),
                           0, st, part, partb, gw, gb, n, c.Cout, d.nchunk);
        rc = last_error_to_status(hipGetLastError());
    }
    (void)hipFreeAsync(part, st);
    return rc;
}

// leaky ReLU and its gradient (slope a for x < 0), elementwise
__global__ void leaky_relu_kernel(long n, float a, const float* __restrict__ x,
                                  float* __restrict__ y)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) {
        const float v = x[i];
        y[i] = v > 0.f ? v : a * v;
    }
}

__global__ void leaky_relu_grad_kernel(long n, float a, const float* __restrict__ x,
                                       const float* __restrict__ gy, float* __restrict__ gx)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) gx[i] = x[i] > 0.f ? gy[i] : a * gy[i];
}

// Adam step on n parameters (bias-corrected learning rate lr_t)
__global__ void adam_kernel(long n, float lr_t, float b1, float b2, float eps,
                            float* __restrict__ w, const float* __restrict__ g,
                            float* __restrict__ m, float* __restrict__ v)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const float gi = g[i];
    const float mi = b1 * m[i] + (1.f - b1) * gi;
    const float vi = b2 * v[i] + (1.f - b2) * gi * gi;
    m[i] = mi;
    v[i] = vi;
    w[i] -= lr_t * mi / (sqrtf(vi) + eps);
}

}  // namespace gpd

using namespace gpd;

static bool conv_dims_ok(int B, int Cin, int Cout, int D, int H, int W)
{
    return B > 0 && Cin > 0 && Cout > 0 && D > 0 && H > 0 && W > 0 && B <= 65535 &&
           (long)D * H * W < (1L << 31);
}

static int conv_forward(int B, int Cin, int Cout, int D, int H, int W, const float* d_x,
                        const float* d_w, const float* d_bias, float* d_y, const ConvEpi& ep,
                        void* stream)
{
    GPD_REQUIRE(conv_dims_ok(B, Cin, Cout, D, H, W), GPD_ERR_ARG, "bad conv sizes");
    GPD_REQUIRE(d_x && d_w && d_y && d_x != d_y, GPD_ERR_ARG, "bad arrays");
    GPD_REQUIRE((long)B * ((Cout + 15) / 16) <= 65535, GPD_ERR_ARG, "batch too large");
    return launch_conv<0>(ConvDims{B, Cin, Cout, D, H, W}, d_x, d_w, d_bias, d_y, ep,
                          (hipStream_t)stream);
}

extern "C" int gpd_conv3d_forward(int B, int Cin, int Cout, int D, int H, int W,
                                  const float* d_x, const float* d_w, const float* d_bias,
                                  float* d_y, int accumulate, void* stream)
{
    return conv_forward(B, Cin, Cout, D, H, W, d_x, d_w, d_bias, d_y, {accumulate, 1.f, nullptr},
                        stream);
}

extern "C" int gpd_conv3d_forward_leaky(int B, int Cin, int Cout, int D, int H, int W,
                                        const float* d_x, const float* d_w, const float* d_bias,
                                        float slope, float* d_y, void* stream)
{
    return conv_forward(B, Cin, Cout, D, H, W, d_x, d_w, d_bias, d_y, {0, slope, nullptr},
                        stream);
}

static int conv_backward_data(int B, int Cin, int Cout, int D, int H, int W, const float* d_gy,
                              const float* d_w, float* d_gx, const ConvEpi& ep, void* stream)
{
    GPD_REQUIRE(conv_dims_ok(B, Cin, Cout, D, H, W), GPD_ERR_ARG, "bad conv sizes");
    GPD_REQUIRE(d_gy && d_w && d_gx && d_gy != d_gx && ep.act != d_gx, GPD_ERR_ARG,
                "bad arrays");
    GPD_REQUIRE((long)B * ((Cin + 15) / 16) <= 65535, GPD_ERR_ARG, "batch too large");
    return launch_conv<1>(ConvDims{B, Cin, Cout, D, H, W}, d_gy, d_w, nullptr, d_gx, ep,
                          (hipStream_t)stream);
}

extern "C" int gpd_conv3d_backward_data(int B, int Cin, int Cout, int D, int H, int W,
                                        const float* d_gy, const float* d_w, float* d_gx,
                                        int accumulate, void* stream)
{
    return conv_backward_data(B, Cin, Cout, D, H, W, d_gy, d_w, d_gx,
                              {accumulate, 1.f, nullptr}, stream);
}

extern "C" int gpd_conv3d_backward_data_leaky(int B, int Cin, int Cout, int D, int H, int W,
                                              const float* d_gy, const float* d_w,
                                              const float* d_act, float slope, float* d_gx,
                                              void* stream)
{
    return conv_backward_data(B, Cin, Cout, D, H, W, d_gy, d_w, d_gx, {0, slope, d_act}, stream);
}

extern "C" int gpd_conv3d_backward_weight(int B, int Cin, int Cout, int D, int H, int W,
                                          const float* d_x, const float* d_gy, float* d_gw,
                                          float* d_gb, void* stream)
{
    GPD_REQUIRE(conv_dims_ok(B, Cin, Cout, D, H, W), GPD_ERR_ARG, "bad conv sizes");
    GPD_REQUIRE(d_x && d_gy && d_gw, GPD_ERR_ARG, "bad arrays");
    GPD_REQUIRE((long)Cout * Cin <= (1L << 30), GPD_ERR_ARG, "too many channel pairs");
    ConvDims d = {B, Cin, Cout, D, H, W};
    hipStream_t st = (hipStream_t)stream;
    return launch_wgrad(d, d_x, d_gy, d_gw, d_gb, st);
}

extern "C" int gpd_leaky_relu(long n, float slope, const float* d_x, float* d_y, void* stream)
{
    GPD_REQUIRE(n >= 0 && (n == 0 || (d_x && d_y)), GPD_ERR_ARG, "bad arrays");
    if (n == 0) return GPD_OK;
    hipLaunchKernelGGL(leaky_relu_kernel, dim3((n + 255) / 256), dim3(256), 0,
                       (hipStream_t)stream, n, slope, d_x, d_y);
    return last_error_to_status(hipGetLastError());
}

extern "C" int gpd_leaky_relu_backward(long n, float slope, const float* d_x, const float* d_gy,
                                       float* d_gx, void* stream)
{
    GPD_REQUIRE(n >= 0 && (n == 0 || (d_x && d_gy && d_gx)), GPD_ERR_ARG, "bad arrays");
    if (n == 0) return GPD_OK;
    hipLaunchKernelGGL(leaky_relu_grad_kernel, dim3((n + 255) / 256), dim3(256), 0,
                       (hipStream_t)stream, n, slope, d_x, d_gy, d_gx);
    return last_error_to_status(hipGetLastError());
}

extern "C" int gpd_adam_step(long n, float lr_t, float beta1, float beta2, float eps, float* d_w,
                             const float* d_g, float* d_m, float* d_v, void* stream)
{
    GPD_REQUIRE(n >= 0 && (n == 0 || (d_w && d_g && d_m && d_v)), GPD_ERR_ARG, "bad arrays");
    if (n == 0) return GPD_OK;
    hipLaunchKernelGGL(adam_kernel, dim3((n + 255) / 256), dim3(256), 0, (hipStream_t)stream, n,
                       lr_t, beta1, beta2, eps, d_w, d_g, d_m, d_v);
    return last_error_to_status(hipGetLastError());
}

// ------------------------------------------------------------------ //
// Forward convolution on MFMA with bfloat16 operands (inference).
//
// Implicit GEMM per workgroup tile of 256 output points (one z-plane, TY
// rows, TX columns; TX = 32 when 32 divides W, else 16): D[o][p] =
// sum_{t, c} W[o, c, t] x[c, p + d_t] on v_mfma_f32_32x32x8_bf16 with
// A = weights (rows o), B = gathered inputs (columns p), k = 8 channels at
// one tap.  Input channels are staged 8 at a time: the tile's input points
// with their 1-point halo (3 planes) and the weights of those channels go
// to LDS as bfloat16 (round to nearest even); the FP32 accumulators hold
// all 27 taps and all channels.  Each wave owns 64 points (two 32-point
// column blocks) for NOB blocks of 32 output channels.  Requires Cin % 8 ==
// 0, Cout <= 32 NOB, W % 16 == 0 and H divisible by TY.
namespace gpd {

constexpr int kMCh = 8;   // channels per LDS stage (one MFMA k-step)

template <int TX, int NOB>
__global__ __launch_bounds__(256) void conv3d_fwd_mfma_kernel(const float* __restrict__ x,
                                                             const float* __restrict__ Wt,
                                                             const float* __restrict__ bias,
                                                             float* __restrict__ y, ConvDims d)
{
    constexpr int TY = 256 / TX;
    constexpr int HX = TX + 2, HY = TY + 2;
    constexpr int NPTS = 3 * HY * HX;
    constexpr int NO = 32 * NOB;
    __shared__ __align__(16) short xs[NPTS * kMCh];
    __shared__ __align__(16) short ws[27 * NO * kMCh];

    const int P = d.D * d.H * d.W;
    const int ntx = d.W / TX, nty = d.H / TY;
    const long nwork = (long)d.B * d.D * nty * ntx;
    const long w = xcd_work_index(blockIdx.x, nwork);
    if (w < 0) return;
    const int tx_i = (int)(w % ntx);
    long r = w / ntx;
    const int ty_i = (int)(r % nty);
    r /= nty;
    const int z = (int)(r % d.D);
    const int b = (int)(r / d.D);
    const int x0 = tx_i * TX, y0 = ty_i * TY;
    const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;

    f32x16 acc[2][NOB];
#pragma unroll
    for (int pb = 0; pb < 2; pb++)
#pragma unroll
        for (int ob = 0; ob < NOB; ob++)
#pragma unroll
            for (int v = 0; v < 16; v++) acc[pb][ob][v] = 0.f;

    // this lane's output points (column of the B operand) in each block
    int qy[2], qx[2];
#pragma unroll
    for (int pb = 0; pb < 2; pb++) {
        const int q = wave * 64 + pb * 32 + lane % 32;
        qy[pb] = q / TX;
        qx[pb] = q % TX;
    }
    const int cq = 4 * (lane / 32);   // this lane's 4 channels of the k-step

    for (int c0 = 0; c0 < d.Cin; c0 += kMCh) {
        __syncthreads();
        for (int s = threadIdx.x; s < NPTS * kMCh; s += 256) {
            const int c = s / NPTS, pt = s % NPTS;
            const int hz = pt / (HY * HX), rem = pt % (HY * HX);
            const int hy = rem / HX, hx = rem % HX;
            const int gz = wrapp(z - 1 + hz, d.D);
            const int gy = wrapp(y0 - 1 + hy, d.H);
            const int gx = wrapp(x0 - 1 + hx, d.W);
            const float v = x[((long)b * d.Cin + c0 + c) * P + ((long)gz * d.H + gy) * d.W + gx];
            xs[pt * kMCh + c] = (short)bf16_bits(v);
        }
        for (int s = threadIdx.x; s < 27 * NO * kMCh; s += 256) {
            const int c = s % kMCh, rem = s / kMCh;
            const int o = rem % NO, t = rem / NO;
            const float v = o < d.Cout ? Wt[((long)o * d.Cin + c0 + c) * 27 + t] : 0.f;
            ws[(t * NO + o) * kMCh + c] = (short)bf16_bits(v);
        }
        __syncthreads();
#pragma unroll 3
        for (int t = 0; t < 27; t++) {
            const int dz = t / 9, dy = (t / 3) % 3, dx = t % 3;
            bf16x4 bop[2];
#pragma unroll
            for (int pb = 0; pb < 2; pb++) {
                const int pt = (dz * HY + qy[pb] + dy) * HX + qx[pb] + dx;
                bop[pb] = *reinterpret_cast<const bf16x4*>(&xs[pt * kMCh + cq]);
            }
#pragma unroll
            for (int ob = 0; ob < NOB; ob++) {
                const int o = ob * 32 + lane % 32;
                const bf16x4 aop = *reinterpret_cast<const bf16x4*>(&ws[(t * NO + o) * kMCh + cq]);
#pragma unroll
                for (int pb = 0; pb < 2; pb++)
                    acc[pb][ob] = __builtin_amdgcn_mfma_f32_32x32x8bf16_1k(aop, bop[pb],
                                                                          acc[pb][ob], 0, 0, 0);
            }
        }
    }
    // D: column = point lane % 32, row = output channel 8 (v / 4) + 4 (lane / 32) + v % 4
#pragma unroll
    for (int pb = 0; pb < 2; pb++) {
        const long p = ((long)z * d.H + y0 + qy[pb]) * d.W + x0 + qx[pb];
#pragma unroll
        for (int ob = 0; ob < NOB; ob++)
#pragma unroll
            for (int v = 0; v < 16; v++) {
                const int o = ob * 32 + 8 * (v / 4) + 4 * (lane / 32) + v % 4;
                if (o < d.Cout)
                    y[((long)b * d.Cout + o) * P + p] = acc[pb][ob][v] + (bias ? bias[o] : 0.f);
            }
    }
}

}  // namespace gpd

extern "C" int gpd_conv3d_forward_bf16(int B, int Cin, int Cout, int D, int H, int W,
                                       const float* d_x, const float* d_w, const float* d_bias,
                                       float* d_y, void* stream)
{
    GPD_REQUIRE(conv_dims_ok(B, Cin, Cout, D, H, W), GPD_ERR_ARG, "bad conv sizes");
    GPD_REQUIRE(d_x && d_w && d_y && d_x != d_y, GPD_ERR_ARG, "bad arrays");
    const int TX = W % 32 == 0 ? 32 : 16;
    const int TY = 256 / TX;
    if (Cin % kMCh != 0 || Cout > 64 || W % 16 != 0 || H % TY != 0) {
        set_last_error("shape not supported by the bfloat16 MFMA convolution");
        return GPD_ERR_UNSUPPORTED;
    }
    ConvDims d = {B, Cin, Cout, D, H, W};
    const long nwork = (long)B * D * (H / TY) * (W / TX);
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid(xcd_grid_size(nwork)), block(256);
    if (TX == 32) {
        if (Cout <= 32)
            hipLaunchKernelGGL((conv3d_fwd_mfma_kernel<32, 1>), grid, block, 0, st, d_x, d_w,
                               d_bias, d_y, d);
        else
            hipLaunchKernelGGL((conv3d_fwd_mfma_kernel<32, 2>), grid, block, 0, st, d_x, d_w,
                               d_bias, d_y, d);
    } else {
        if (Cout <= 32)
            hipLaunchKernelGGL((conv3d_fwd_mfma_kernel<16, 1>), grid, block, 0, st, d_x, d_w,
                               d_bias, d_y, d);
        else
            hipLaunchKernelGGL((conv3d_fwd_mfma_kernel<16, 2>), grid, block, 0, st, d_x, d_w,
                               d_bias, d_y, d);
    }
    return last_error_to_status(hipGetLastError());
}
