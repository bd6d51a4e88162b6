// Fused pseudo-Hamiltonian apply and projector coefficients (gfx950).
//
// H psi = T psi + v psi + sum_a p_a (P_a dH_a)  -- the composite of
// FDWaveFunctions.apply_pseudo_hamiltonian (gpaw/wavefunctions/fd.py:77-83)
// and Hamiltonian.apply (gpaw/hamiltonian.py:426-460).  The kinetic stencil
// kernel adds the local potential in its epilogue; the projector terms
// follow in a second launch over the covered points.  The per-point
// rounding sequence is the reference's (stencil sum, + psi*v, then the
// projector terms in volume order).
#include <type_traits>

#include "common.hpp"
#include "fd.hpp"
#include "lfc.hpp"

namespace gpd {

// c = P dH of an atom's functions, summed over i in order.  Bound by the
// latency of its loads: a workgroup takes an atom and 16 bands, 16 lanes of a
// band a function each, and a lane has eight terms' loads in flight.  4 bands
// of 24^3 4.4 us, 50 FP32 bands and 11 atoms 4.1, 64 complex bands 5.2, 256 bands
// and 32 atoms 22 (a thread a band and atom, one term at a time: 10, 13, 19 and
// 75 us).
template <typename T> __device__ __forceinline__ T term(T s, T p, T h) { return madd<T>(s, p, h); }
__device__ __forceinline__ double2 term(double2 s, double2 p, double h)
{
    return make_double2(madd<double>(s.x, p.x, h), madd<double>(s.y, p.y, h));
}

template <typename T, typename H>
__global__ __launch_bounds__(256) void projector_coefs_kernel(
    long nb, int Mmax, int natoms, const int* __restrict__ M_a, const int* __restrict__ ni_a,
    const int* __restrict__ dH_off, const H* __restrict__ dH, const T* __restrict__ P,
    T* __restrict__ c)
{
    constexpr int NB = 8;
    const int a = (int)(blockIdx.x % natoms);
    const long x = (long)(blockIdx.x / natoms) * 16 + threadIdx.x / 16;
    if (x >= nb) return;
    const int ni = ni_a[a];
    const T* Pa = P + x * Mmax + M_a[a];
    const H* h = dH + dH_off[a];
    T* ca = c + x * Mmax + M_a[a];
    for (int j = threadIdx.x % 16; j < ni; j += 16) {
        T s = T{};
        for (int i0 = 0; i0 < ni; i0 += NB) {
            T pv[NB];
            H hv[NB];
#pragma unroll
            for (int k = 0; k < NB; k++) {
                const int i = min(i0 + k, ni - 1);
                pv[k] = Pa[i];
                hv[k] = h[i * ni + j];
            }
#pragma unroll
            for (int k = 0; k < NB; k++)
                if (i0 + k < ni) s = term(s, pv[k], hv[k]);
        }
        ca[j] = s;
    }
}

template <typename T>
__global__ void local_potential_kernel(long nb, long nG, const T* __restrict__ psi,
                                       const T* __restrict__ v, T* __restrict__ hpsi)
{
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nb * nG) return;
    hpsi[idx] = madd<T>(hpsi[idx], psi[idx], v[idx % nG]);
}

// complex bands (k-points): psi, P and c complex, v and dH real.  The
// potential term is the reference's numpy psit * vt (each part times v),
// then added.
__global__ void local_potential_z_kernel(long nb, long nG, const double2* __restrict__ psi,
                                         const double* __restrict__ v,
                                         double2* __restrict__ hpsi)
{
    long idx = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (idx >= nb * nG) return;
    const double2 p = psi[idx];
    const double w = v[idx % nG];
    double2 h = hpsi[idx];
    h.x = madd<double>(h.x, p.x, w);
    h.y = madd<double>(h.y, p.y, w);
    hpsi[idx] = h;
}

template <typename T>
__global__ void fill_zero_kernel(long n, T* __restrict__ p)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) p[i] = T(0);
}

// an event of one call, without timing
struct Event {
    hipEvent_t e = nullptr;
    ~Event()
    {
        if (e) (void)hipEventDestroy(e);
    }
    // `second` goes on after what `first` has now
    hipError_t order(hipStream_t first, hipStream_t second)
    {
        if (first == second) return hipSuccess;
        hipError_t rc = hipEventCreateWithFlags(&e, hipEventDisableTiming);
        if (rc == hipSuccess) rc = hipEventRecord(e, first);
        return rc == hipSuccess ? hipStreamWaitEvent(second, e, 0) : rc;
    }
};

// Stencil + v psi in one launch, then the projector terms: FP64 per
// covered point in the reference's order (the same roundings as adding
// them inside the stencil's epilogue, which measured slower: 5.2 ms against
// 1.25 + 2.3 ms at 96^3 x 256), FP32 by colours of disjoint atom groups.
template <typename T>
static int ham_apply(gpd_operator* kin, gpd_lfc* lfc, long nb, const T* psi, const T* v,
                     const T* c, T* out, hipStream_t st)
{
    FdEpilogue<T> ep = {};
    ep.aux = v;
    int rc = fd_apply_typed<T>(kin, EPI_POT, nb, psi, out, ep, st);
    if (rc || !lfc || !c) return rc;
    if (std::is_same<T, float>::value)
        return lfc_add_f32(lfc, nb, (const float*)c, (float*)out, st);
    return lfc_add_exact_f64(lfc, nb, (const double*)c, (double*)out, st);
}

}  // namespace gpd

using namespace gpd;

extern "C" int gpd_hamiltonian_apply(gpd_operator* kin, gpd_lfc* lfc, int dtype, long nb,
                                     const void* d_psi, const void* d_v, const void* d_c,
                                     void* d_out, void* stream)
{
    GPD_REQUIRE(kin, GPD_ERR_ARG, "null kinetic operator");
    GPD_REQUIRE(nb >= 0, GPD_ERR_ARG, "negative batch");
    if (nb == 0) return GPD_OK;
    GPD_REQUIRE(d_psi && d_v && d_out && d_psi != d_out, GPD_ERR_ARG, "bad arrays");
    if (lfc) {
        GPD_REQUIRE(lfc->nG == (long)kin->n[0] * kin->n[1] * kin->n[2], GPD_ERR_ARG,
                    "projector grid does not match the operator grid");
        GPD_REQUIRE(d_c, GPD_ERR_ARG, "projector coefficients missing");
    }
    hipStream_t st = (hipStream_t)stream;
    if (dtype == GPD_F64)
        return ham_apply<double>(kin, lfc, nb, (const double*)d_psi, (const double*)d_v,
                                 (const double*)d_c, (double*)d_out, st);
    if (dtype == GPD_F32)
        return ham_apply<float>(kin, lfc, nb, (const float*)d_psi, (const float*)d_v,
                                (const float*)d_c, (float*)d_out, st);
    GPD_REQUIRE(false, GPD_ERR_ARG, "unknown dtype");
}

extern "C" int gpd_hamiltonian_apply_projected(gpd_operator* kin, gpd_lfc* lfc, int dtype,
                                               long nb, const void* d_psi, const void* d_v,
                                               int Mmax, int natoms, const int* d_M_a,
                                               const int* d_ni_a, const int* d_dH_off,
                                               const void* d_dH, long nP, void* d_P, void* d_c,
                                               void* d_out, void* stream, void* side)
{
    GPD_REQUIRE(dtype == GPD_F64 || dtype == GPD_F32, GPD_ERR_ARG, "unknown dtype");
    GPD_REQUIRE(nb >= 0 && nP >= 0, GPD_ERR_ARG, "bad sizes");
    if (nb == 0 && nP == 0) return GPD_OK;
    GPD_REQUIRE(kin && lfc && d_P && d_c && Mmax > 0 && nP / Mmax >= nb, GPD_ERR_ARG,
                "bad projector arrays");
    hipStream_t main = (hipStream_t)stream, st = (hipStream_t)side;
    Event fork, join;
    GPD_CHECK_HIP(fork.order(main, st));
    if (dtype == GPD_F64)
        hipLaunchKernelGGL(fill_zero_kernel<double>, dim3((unsigned)((nP + 255) / 256)),
                           dim3(256), 0, st, nP, (double*)d_P);
    else
        hipLaunchKernelGGL(fill_zero_kernel<float>, dim3((unsigned)((nP + 255) / 256)), dim3(256),
                           0, st, nP, (float*)d_P);
    int rc = last_error_to_status(hipGetLastError());
    if (!rc) rc = gpd_lfc_integrate(lfc, dtype, nb, d_psi, d_P, side);
    if (!rc)
        rc = gpd_projector_coefs(dtype, nP / Mmax, Mmax, natoms, d_M_a, d_ni_a, d_dH_off, d_dH,
                                 d_P, d_c, side);
    // the caller's stream waits for the second one whatever has failed
    const int rc2 = rc ? GPD_OK
                       : gpd_hamiltonian_apply(kin, nullptr, dtype, nb, d_psi, d_v, nullptr,
                                               d_out, stream);
    GPD_CHECK_HIP(join.order(st, main));
    if (rc || rc2) return rc ? rc : rc2;
    return gpd_lfc_add(lfc, dtype, nb, d_c, d_out, stream);
}

extern "C" int gpd_hamiltonian_apply_z(gpd_operator* kin, long nb, long nG, const void* d_psi,
                                       const void* d_v, void* d_out, const double* phases,
                                       void* stream)
{
    GPD_REQUIRE(kin, GPD_ERR_ARG, "null kinetic operator");
    GPD_REQUIRE(nb >= 0, GPD_ERR_ARG, "negative batch");
    GPD_REQUIRE(nG == (long)kin->n[0] * kin->n[1] * kin->n[2], GPD_ERR_ARG,
                "grid size does not match the kinetic operator");
    if (nb == 0) return GPD_OK;
    GPD_REQUIRE(d_psi && d_v && d_out && d_psi != d_out, GPD_ERR_ARG, "bad arrays");
    hipStream_t st = (hipStream_t)stream;
    const double2* psi = (const double2*)d_psi;
    const double* v = (const double*)d_v;
    double2* out = (double2*)d_out;
    int rc = fd_apply_complex(kin, nb, psi, out, phases, v, st);
    if (rc != kNotFused) return rc;
    // stencils the streaming kernel does not take: stencil, then + psi v
    rc = fd_apply_complex(kin, nb, psi, out, phases, nullptr, st);
    if (rc) return rc;
    const long n = nb * nG;
    hipLaunchKernelGGL(local_potential_z_kernel, dim3((n + 255) / 256), dim3(256), 0, st, nb, nG,
                       psi, v, out);
    return last_error_to_status(hipGetLastError());
}

extern "C" int gpd_projector_coefs(int dtype, long nb, int Mmax, int natoms, const int* d_M_a,
                                   const int* d_ni_a, const int* d_dH_off, const void* d_dH,
                                   const void* d_P, void* d_c, void* stream)
{
    GPD_REQUIRE(nb >= 0 && natoms >= 0 && Mmax >= 0, GPD_ERR_ARG, "bad sizes");
    if (nb == 0 || natoms == 0) return GPD_OK;
    GPD_REQUIRE(d_M_a && d_ni_a && d_dH_off && d_dH && d_P && d_c && d_P != d_c, GPD_ERR_ARG,
                "bad arrays");
    hipStream_t st = (hipStream_t)stream;
    const dim3 grid((unsigned)((nb + 15) / 16 * natoms));
    if (dtype == GPD_F64) {
        hipLaunchKernelGGL((projector_coefs_kernel<double, double>), grid, dim3(256), 0, st, nb,
                           Mmax, natoms, d_M_a, d_ni_a, d_dH_off, (const double*)d_dH,
                           (const double*)d_P, (double*)d_c);
        return last_error_to_status(hipGetLastError());
    }
    if (dtype == GPD_F32) {
        hipLaunchKernelGGL((projector_coefs_kernel<float, float>), grid, dim3(256), 0, st, nb,
                           Mmax, natoms, d_M_a, d_ni_a, d_dH_off, (const float*)d_dH,
                           (const float*)d_P, (float*)d_c);
        return last_error_to_status(hipGetLastError());
    }
    if (dtype == GPD_C128) {
        hipLaunchKernelGGL((projector_coefs_kernel<double2, double>), grid, dim3(256), 0, st, nb,
                           Mmax, natoms, d_M_a, d_ni_a, d_dH_off, (const double*)d_dH,
                           (const double2*)d_P, (double2*)d_c);
        return last_error_to_status(hipGetLastError());
    }
    GPD_REQUIRE(false, GPD_ERR_ARG, "unknown dtype");
}

extern "C" int gpd_add_local_potential(int dtype, long nb, long nG, const void* d_psi,
                                       const void* d_v, void* d_hpsi, void* stream)
{
    GPD_REQUIRE(nb >= 0 && nG > 0, GPD_ERR_ARG, "bad sizes");
    if (nb == 0) return GPD_OK;
    GPD_REQUIRE(d_psi && d_v && d_hpsi, GPD_ERR_ARG, "null array");
    hipStream_t st = (hipStream_t)stream;
    long n = nb * nG;
    if (dtype == GPD_F64) {
        hipLaunchKernelGGL(local_potential_kernel<double>, dim3((n + 255) / 256), dim3(256), 0, st,
                           nb, nG, (const double*)d_psi, (const double*)d_v, (double*)d_hpsi);
        return last_error_to_status(hipGetLastError());
    }
    if (dtype == GPD_F32) {
        hipLaunchKernelGGL(local_potential_kernel<float>, dim3((n + 255) / 256), dim3(256), 0, st,
                           nb, nG, (const float*)d_psi, (const float*)d_v, (float*)d_hpsi);
        return last_error_to_status(hipGetLastError());
    }
    if (dtype == GPD_C128) {
        hipLaunchKernelGGL(local_potential_z_kernel, dim3((n + 255) / 256), dim3(256), 0, st, nb,
                           nG, (const double2*)d_psi, (const double*)d_v, (double2*)d_hpsi);
        return last_error_to_status(hipGetLastError());
    }
    GPD_REQUIRE(false, GPD_ERR_ARG, "unknown dtype");
}
