/*
 * gpawdft_amd -- C ABI of the MI355X (gfx950) real-space grid Hamiltonian
 * path.  Plain pointers and sizes only.  Array arguments named d_* are
 * device pointers (HIP global memory); everything else is host memory.
 * `stream` is a hipStream_t passed as void* (NULL = the default stream).
 *
 * Grids are C-contiguous (..., n0, n1, n2) with n2 the contiguous axis;
 * a batch of nb grids is nb consecutive grids.  dtype selects the element
 * type of the device arrays: GPD_F64 (bit-compatible with the reference's
 * FP64 C code), GPD_F32, or, where an entry point says so, GPD_C128
 * (complex128, interleaved re, im).
 *
 * Every function returns an int status: 0 on success, < 0 for a bad
 * argument or a HIP failure (gpd_last_error() gives the message), > 0 for
 * a LAPACK-style info from the dense FP64 routines.  Calls are stream
 * ordered: they return once the work is queued.
 */
#ifndef GPAWDFT_AMD_H
#define GPAWDFT_AMD_H

#ifdef __cplusplus
extern "C" {
#endif

enum {
    GPD_OK = 0,
    GPD_ERR_ARG = -1,
    GPD_ERR_HIP = -2,
    GPD_ERR_UNSUPPORTED = -3,
    GPD_ERR_NOMEM = -4
};

enum { GPD_F64 = 0, GPD_F32 = 1, GPD_C128 = 2 };

/* Message of the last failed call on this thread ("" if none). */
const char* gpd_last_error(void);

/* Library version string. */
const char* gpd_version(void);

/* ------------------------------------------------------------------ */
/* Finite-difference operator.
 * Replaces _gpaw.Operator(coefs, offsets, size, range, neighbors, real,
 * comm, cfd) (c/operators.c:462-495): `offsets` are flat offsets with the
 * padded strides [(n1+2r)(n2+2r), n2+2r, 1] that gpaw/fd_operators.py:43-52
 * builds; neighbors[c][d] >= 0 marks a periodic axis (a single rank is its
 * own neighbour), -1 a zero boundary.  One operator serves every dtype:
 * pass real = 1 (other values return GPD_ERR_UNSUPPORTED); complex grids
 * and their Bloch phases are given per call to gpd_operator_apply with
 * GPD_C128.                                                            */
typedef struct gpd_operator gpd_operator;

int gpd_operator_create(const double* coefs, const long* offsets, int ncoefs,
                        const long size[3], int range,
                        const long neighbors[6], int real, int cfd,
                        gpd_operator** out);

/* Operator.apply(in, out, phases) (c/operators.c:316-405): out = A in for
 * nin grids.  For GPD_F64 / GPD_F32 phases must be NULL.  For GPD_C128
 * (interleaved re, im) phases is a host array of 12 doubles, the (3, 2)
 * complex phase_cd: [axis][0] multiplies the periodic image above the
 * cell, [axis][1] the image below (c/bc.c:227-247 with
 * c/bmgs/translate.c:27-47), a corner carrying axis 0's phase first; NULL
 * means all ones (Gamma).  Bit-compatible with the reference's complex
 * Operator in every dtype.                                             */
int gpd_operator_apply(gpd_operator* op, int dtype, long nin,
                       const void* d_in, void* d_out, const void* phases,
                       void* stream);

/* Operator.relax(relax_method, func, source, nrelax, w) (c/operators.c:
 * 49-91, c/bmgs/relax.c): nrelax sweeps on nin grids of d_fun in place for
 * the equation "operator f = src", bit-compatible in FP64.
 * relax_method 2: weighted Jacobi (the Poisson solver's default).
 * relax_method 1: Gauss-Seidel, the reference's lexicographic sweep, run
 * one hyperplane i0 + i1 + i2 = const at a time (w is ignored, as there);
 * stencils with off-axis points return GPD_ERR_UNSUPPORTED for it.
 * Allocates one stream-ordered temporary grid set. */
int gpd_operator_relax(gpd_operator* op, int dtype, int relax_method, long nin,
                       void* d_fun, const void* d_src, int nrelax, double w,
                       void* stream);

/* Operator.get_diagonal_element() (c/operators.c:408-421). */
int gpd_operator_get_diagonal_element(const gpd_operator* op, double* diag);

/* Launch shape of the streaming stencil: split axis 0 into chunks until
 * about wg_target workgroups run (default 8192).  No counterpart in the
 * reference (its stencil is a serial loop); the ragged-batch autotuner sets
 * it per grid and band count.  Results do not depend on it. */
int gpd_operator_set_launch(gpd_operator* op, long wg_target);

int gpd_operator_destroy(gpd_operator* op);

/* ------------------------------------------------------------------ */
/* Restriction / interpolation between grids of 2:1 spacing.
 * Replaces _gpaw.Transformer(size_in, size_out, k, paddings, npaddings,
 * skip, neighbors, real, comm, interpolate) (c/transformers.c:219-262);
 * paddings/npaddings/skip/neighbors are [3][2] as computed by
 * gpaw/transformers.py:20-76.  k = 2, 4, 6 or 8.                       */
typedef struct gpd_transformer gpd_transformer;

int gpd_transformer_create(const long size_in[3], const long size_out[3],
                           int k, const long paddings[6],
                           const long npaddings[6], const long skip[6],
                           const long neighbors[6], int real, int interpolate,
                           gpd_transformer** out);

/* Transformer.apply(in, out, phases) (c/transformers.c:127-185).  For
 * GPD_F64 / GPD_F32 phases must be NULL; for GPD_C128 it is the (3, 2)
 * complex phase_cd as in gpd_operator_apply (12 host doubles, NULL for
 * Gamma), bit-compatible with the reference's complex Transformer.    */
int gpd_transformer_apply(gpd_transformer* t, int dtype, long nin,
                          const void* d_in, void* d_out, const void* phases,
                          void* stream);

/* Second-order transfer of FP32 grids with what follows it in a network:
 * out = d (add + alpha T(in)), d = act > 0 ? 1 : slope, each step rounded;
 * add and act are arrays of out's shape (not out itself) or NULL.  k != 2
 * returns GPD_ERR_UNSUPPORTED.                                          */
int gpd_transformer_apply_affine(gpd_transformer* t, long nin,
                                 const float* d_in, float alpha,
                                 const float* d_add, const float* d_act,
                                 float slope, float* d_out, void* stream);

int gpd_transformer_destroy(gpd_transformer* t);

/* One V-cycle of the FD Poisson solver's multigrid from level 0
 * (PoissonSolver.iterate2, gpaw/poisson.py:278-311): on each level l <
 * levels, relax presmooths[l] sweeps, residual = op phi - rho, restrict
 * it to rho[l+1], phi[l+1] = 0, recurse, phi -= interpolated phi[l+1];
 * then relax postsmooths[l] sweeps; at level 0 finally residual = op phi
 * - rho and d_norm[0] = dv * sum(residual^2).  ops: levels + 1 operators,
 * restrictors / interpolators: levels transformers; phis, rhos,
 * residuals: levels + 1 FP64 device grids of one band; presmooths,
 * postsmooths, weights: host arrays of levels + 1; relax_method as in
 * gpd_operator_relax; d_minus_one: an FP64 device -1.0 (must be given; the
 * differences no longer read it); d_norm: FP64 device output.  The
 * reference issues these calls one at a time from Python; here one call
 * walks the levels, so the host keeps ahead of the GPU.  The differences
 * are formed in the stencil and in the interpolation, and the coarsest
 * levels run in one launch where they fit a workgroup's LDS.  phi of level 0,
 * its residual and the norm get the bits of the single calls; the other
 * levels' grids are scratch: those inside the launch of the coarsest levels
 * are not written but for the first one's phi, and a level's sweeps alternate
 * between its phi and its residual.  A level's phi, rho and residual, its
 * residual and the next level's rho and phi, and the phi of consecutive
 * levels must be distinct; below level 0 the coarsest level's residual is not
 * used.  Allocates only the stream-ordered temporaries of relax and the dot. */
int gpd_poisson_vcycle(int levels, gpd_operator* const* ops,
                       gpd_transformer* const* restrictors,
                       gpd_transformer* const* interpolators,
                       double* const* phis, double* const* rhos,
                       double* const* residuals, const int* presmooths,
                       const int* postsmooths, const double* weights,
                       int relax_method, double dv, const double* d_minus_one,
                       double* d_norm, void* stream);

/* ------------------------------------------------------------------ */
/* Radial cubic spline (FP64, host).  Replaces _gpaw.Spline(l, rcut, f_g)
 * (c/spline.c:121-135, c/bmgs/spline.c:11-39).  f[npts-1] is used as
 * given (gpaw/spline.py:25 sets it to zero before the call).          */
typedef struct gpd_spline gpd_spline;

int gpd_spline_create(int l, double rcut, const double* f, int npts,
                      gpd_spline** out);
double gpd_spline_value(const gpd_spline* s, double r);
double gpd_spline_get_cutoff(const gpd_spline* s);
int gpd_spline_get_angular_momentum_number(const gpd_spline* s);
int gpd_spline_destroy(gpd_spline* s);

/* spline_to_grid (c/lfc.c:785-875), host FP64.  Tabulates f(r) r^l Y_lm
 * over the box [beg, end) of the local grid (corner gdcorner, size n) for
 * points with r < rcut.  A_gm must hold (box points) x (2l+1) doubles and
 * G_B 2 * (box rows) ints; *ng receives the rows written and *nB the
 * number of G_B entries.                                               */
int gpd_spline_to_grid(const gpd_spline* s, const long beg[3],
                       const long end[3], const double pos_v[3],
                       const double h_cv[9], const long n[3],
                       const long gdcorner[3], double* A_gm, int* G_B,
                       long* ng, long* nB);

/* ------------------------------------------------------------------ */
/* Localized functions (PAW projectors) on the grid.
 * Replaces _gpaw.LFC(A_Wgm, M_W, G_B, W_B, dv, phase_qW) (c/lfc.c:106-186);
 * the phases of complex functions are set per k-point by
 * gpd_lfc_set_phases.  Volume W has ng_W[W] rows of nm_W[W]
 * values, concatenated row-major in A (host, FP64); (G_B, W_B) is the
 * boundary list sorted by G (gpaw/lfc.py:276-350).  nG is the number of
 * points of one grid and Mmax the number of functions.  The object keeps
 * device copies of everything it needs.                                */
typedef struct gpd_lfc gpd_lfc;

int gpd_lfc_create(int nW, const double* A, const int* ng_W, const int* nm_W,
                   const int* M_W, int nB, const int* G_B, const int* W_B,
                   double dv, long nG, int Mmax, gpd_lfc** out);

/* LFC.integrate (c/lfc.c:361-425): c_xM += dv * sum_G a_xG A_GM for nx
 * grids; c_xM is (nx, Mmax) of the same dtype.  In FP64 and complex128 the
 * sums run in the reference's order, point by point, and nothing is
 * allocated.  In FP32 the object keeps a workspace for per-segment
 * partial sums, allocated (hipMalloc) by the first call with a larger nx
 * than before: a caller that captures the call into a graph runs it once
 * eagerly with that nx first.                                          */
int gpd_lfc_integrate(gpd_lfc* lfc, int dtype, long nx, const void* d_a_xG,
                      void* d_c_xM, void* stream);

/* LFC.add (c/lfc.c:724-783): a_xG += sum_M A_GM c_xM, per point in the
 * reference's volume order.                                            */
int gpd_lfc_add(gpd_lfc* lfc, int dtype, long nx, const void* d_c_xM,
                void* d_a_xG, void* stream);

/* The k-point of the complex (GPD_C128) integrate and add: phase_W holds
 * nW complex values (interleaved re, im; host), phase_qW[q] of
 * gpaw/lfc.py:336-343, exp(2 pi i k_q . sdisp_W) for the periodic image of
 * each volume.  integrate then sums a * (phase dv) * A and add adds
 * (sum_m A c) * conj(phase) (c/lfc.c:400-423, 758-781); NULL sets all
 * ones (Gamma).                                                        */
int gpd_lfc_set_phases(gpd_lfc* lfc, const double* phase_W);

/* Launch knob of the exact (FP64, complex) integrate: 16, 32 or 64 (the
 * more, the more bands a workgroup takes), or 0 for the automatic choice,
 * which goes by the number of workgroups.  Results do not depend on it.  No
 * counterpart in the reference (a tuning parameter of this library's
 * kernels).                                                            */
int gpd_lfc_set_launch(gpd_lfc* lfc, int exact_bands);

int gpd_lfc_destroy(gpd_lfc* lfc);

/* The whole of Htpsit = T psi + v psi + sum_a p_a (P dH)_a for nb bands
 * (GPD_F64, GPD_F32) in one call: P (nP values, at least nb rows of Mmax)
 * cleared and filled with the projections and c = P dH (the tables of
 * gpd_projector_coefs) on stream `side` while the stencil and v psi run on
 * `stream`, which then waits for it and adds the projector terms; one after
 * the other where side is stream.  Not for use under graph capture.     */
int gpd_hamiltonian_apply_projected(gpd_operator* kin, gpd_lfc* lfc, int dtype,
                                    long nb, const void* d_psi,
                                    const void* d_v, int Mmax, int natoms,
                                    const int* d_M_a, const int* d_ni_a,
                                    const int* d_dH_off, const void* d_dH,
                                    long nP, void* d_P, void* d_c,
                                    void* d_out, void* stream, void* side);

/* ------------------------------------------------------------------ */
/* Fused pseudo-Hamiltonian apply: out = T psi + v psi + sum_a p_a c_a for
 * nb bands, the composite of FDWaveFunctions.apply_pseudo_hamiltonian
 * (gpaw/wavefunctions/fd.py:77-83) and Hamiltonian.apply
 * (gpaw/hamiltonian.py:426-460).  kin is the kinetic operator; d_v the
 * local potential (one grid, dtype); lfc/d_c may be NULL for no projector
 * term, else d_c holds c_xM = P_xM dH (nb, Mmax).  The per-point rounding
 * sequence is the reference's: stencil sum, then + psi*v, then the
 * projector terms in volume order.                                     */
int gpd_hamiltonian_apply(gpd_operator* kin, gpd_lfc* lfc, int dtype, long nb,
                          const void* d_psi, const void* d_v,
                          const void* d_c, void* d_out, void* stream);

/* Complex bands at a k-point: out = T psi + v psi for nb complex128 grids
 * (interleaved re, im) of nG points each, the first two steps of
 * Hamiltonian.apply (gpaw/hamiltonian.py:426-460): kin.apply(psi, out,
 * phase_cd), then out += psi * vt.  d_v is the real FP64 potential of nG
 * points; phases as in gpd_operator_apply; nG must equal the operator's
 * grid size (GPD_ERR_ARG otherwise).  Bit-identical to the two separate
 * calls (the product rounded, then added); fused into the stencil's
 * epilogue for orthorhombic stencils of range 1-3.                     */
int gpd_hamiltonian_apply_z(gpd_operator* kin, long nb, long nG, const void* d_psi,
                            const void* d_v, void* d_out,
                            const double* phases, void* stream);

/* Htpsit_nG += psit_nG * vt_G for nb grids of nG points
 * (Hamiltonian.apply_local_potential, gpaw/hamiltonian.py:397-424): the
 * product is rounded, then added, as the reference's numpy expression.
 * For GPD_C128 psi and hpsi are complex and v is real FP64 (each part
 * times v).                                                            */
int gpd_add_local_potential(int dtype, long nb, long nG, const void* d_psi,
                            const void* d_v, void* d_hpsi, void* stream);

/* c_xM = P_xM dH for block-diagonal dH: atom a owns columns
 * [M_a[a], M_a[a] + ni_a[a]) and the ni x ni matrix at dH[dH_off[a]]
 * (row-major, dtype).  Sums run over i in order (gpaw/hamiltonian.py:456,
 * there via numpy/BLAS).  d_M_a, d_ni_a, d_dH_off are device int arrays.
 * For GPD_C128 P and c are complex and dH is real FP64.               */
int gpd_projector_coefs(int dtype, long nb, int Mmax, int natoms,
                        const int* d_M_a, const int* d_ni_a,
                        const int* d_dH_off, const void* d_dH,
                        const void* d_P, void* d_c, void* stream);

/* ------------------------------------------------------------------ */
/* Multigrid preconditioner (gpaw/preconditioner.py:11-60): a 3-level
 * V-cycle with kin0 on the fine grid, 7-point kin1/kin2 on the coarse
 * grids, restrictors r0 (fine->1), r1 (1->2), interpolators i2 (2->1),
 * i1 (1->fine), step = 0.66666666 / diag(kin0).  The object owns device
 * scratch for up to `block` bands.                                     */
typedef struct gpd_precond gpd_precond;

int gpd_precond_create(gpd_operator* kin0, gpd_operator* kin1,
                       gpd_operator* kin2, gpd_transformer* r0,
                       gpd_transformer* r1, gpd_transformer* i2,
                       gpd_transformer* i1, double step, long block,
                       gpd_precond** out);

/* __call__(residuals) -> d0: out = preconditioned correction for nb <=
 * block residuals.                                                     */
int gpd_precond_apply(gpd_precond* pc, int dtype, long nb, const void* d_R,
                      void* d_out, void* stream);

/* __call__(residuals, kpt) for complex128 bands at a k-point
 * (gpaw/preconditioner.py:34-60 with kpt.phase_cd): every stencil and
 * transformer with the Bloch phases (host [3][2] complex as in
 * gpd_operator_apply, NULL for Gamma), the elementwise steps folded into
 * the kernels as in gpd_precond_apply.  GPD_ERR_UNSUPPORTED (nothing done)
 * unless the three stencils have the axis form of range 1-3 and the
 * transformers are nn = 1.  Allocates its workspace on first use.      */
int gpd_precond_apply_z(gpd_precond* pc, long nb, const void* d_R,
                        void* d_out, const double* phases, void* stream);

/* The same V-cycle, allocating nothing.  No counterpart in the reference:
 * it is for callers that cannot allocate device memory (code under HIP
 * graph capture, tight eigensolver loops, harnesses that forbid
 * hipMalloc).  The intermediates live in a fixed 192 MiB device array of
 * the library (one per GPU, held until the process ends), so a call takes
 * at most floor(192 MiB / ((g0 + 3 g1 + 3 g2) * sizeof(T))) bands, g0..g2
 * the points of the three levels (20 FP64 bands at 96^3); larger batches
 * return GPD_ERR_ARG.  The block size of gpd_precond_create does not
 * apply.  Every call on one GPU shares that array: calls that overlap on
 * one GPU (other streams, other threads) race.  Stencils without a fused
 * epilogue (non axis-form, range > 3) return GPD_ERR_UNSUPPORTED.  Same
 * results as gpd_precond_apply.                                        */
int gpd_precond_apply_noalloc(gpd_precond* pc, int dtype, long nb,
                              const void* d_R, void* d_out, void* stream);

int gpd_precond_destroy(gpd_precond* pc);

/* ------------------------------------------------------------------ */
/* Subspace matrices and rotations (MatrixOperator, gpaw/hs_operators.py).
 *
 * gpd_inner_products: out[i][j] = alpha * sum_k X[i][k] Y[j][k] for i, j <
 * N (full N x N, FP64, row-major); hermitian != 0 gives
 * 0.5 alpha (T + T^T) -- the rk / r2k calls of GridDescriptor.integrate
 * (gpaw/grid_descriptor.py:300-306, c/blas.c:290-353), both triangles
 * filled.  X, Y: (N, K) of dtype.  FP32 runs split-bfloat16 MFMA
 * (hi+mid+lo per operand, six products, FP32 accumulation over 64 values
 * of k, then FP64); FP64 runs FP64 MFMA.  GPD_C128 (complex bands at a
 * k-point; the zherk / zher2k / zgemm('c') calls, c/blas.c:137,183,322,348):
 * out is complex128 (N, N) interleaved, out[i][j] = alpha * sum_k X[i][k]
 * conj(Y[j][k]), hermitian 0.5 alpha (T + T^H), exactly Hermitian when X
 * and Y are the same array.  d_work (may be NULL) is device scratch for the
 * per-chunk partials; if too small, the call allocates.                 */
int gpd_inner_products(int dtype, int N, long K, const void* d_X,
                       const void* d_Y, double alpha, int hermitian,
                       void* d_work, long work_bytes, double* d_out,
                       void* stream);

/* gpd_rotate: Y[n][k] = sum_m C[n][m] X[m][k] -- MatrixOperator.
 * matrix_multiply / GridDescriptor.gemm (gpaw/hs_operators.py:453-466,
 * c/blas.c:95-145).  C: FP64 (N, N) row-major (complex128, interleaved,
 * for GPD_C128: zgemm); X, Y: (N, K) of dtype, distinct.                */
int gpd_rotate(int dtype, int N, long K, const double* d_C, const void* d_X,
               void* d_Y, void* stream);

/* gpd_paw_matrix_add: A[i][j] += sum_a (P2 dA_a P1^H)[i][j] over atoms
 * (gemm(1.0, P1_ni, dA(a, P2_ni), 1.0, A_NN, 'c'), gpaw/hs_operators.py:
 * 309-311).  P1, P2: (N, Mmax) of dtype; dA blocks FP64 row-major ni x ni
 * at dA_off[a]; A: FP64 (N, N), complex128 for GPD_C128.                */
int gpd_paw_matrix_add(int dtype, int N, int Mmax, int natoms,
                       const int* d_M_a, const int* d_ni_a,
                       const int* d_dA_off, const double* d_dA,
                       const void* d_P1, const void* d_P2, double* d_A,
                       void* stream);

/* gpd_inverse_cholesky: inverse_cholesky(a) (c/lapack.c:324-370): the
 * lower triangle of the FP64 (n, n) matrix holds S; on return it holds
 * L^-1 with S = L L^T and the upper triangle is zero.  *info > 0 (LAPACK
 * dpotrf convention) if S is not positive definite.  Synchronises the
 * stream.                                                               */
int gpd_inverse_cholesky(int n, double* d_A, int* info, void* stream);

/* gpd_inverse_cholesky_z: the complex128 inverse_cholesky (zpotrf +
 * ztrtri, c/lapack.c:354-357): the lower triangle of the Hermitian
 * (n, n) interleaved matrix holds S; on return L^-1 with S = L L^H, the
 * upper triangle zero; info as above.                                   */
int gpd_inverse_cholesky_z(int n, double* d_A, int* info, void* stream);

/* gpd_diagonalize: diagonalize(a, w) (c/lapack.c:129-160): eigenvalues of
 * the symmetric FP64 (n, n) matrix whose lower triangle is given, in
 * ascending order into d_w; eigenvectors into the rows of d_A.  Jacobi
 * sweeps; *sweeps receives their number (may be NULL).  Synchronises the
 * stream once per sweep.                                                */
int gpd_diagonalize(int n, double* d_A, double* d_w, int* sweeps,
                    void* stream);

/* gpd_diagonalize_z: the complex128 diagonalize (zheev("V", "U") on the C
 * view, c/lapack.c:152): eigenvalues of the Hermitian matrix whose lower
 * triangle is given (interleaved), ascending into d_w; row k of d_A
 * receives conj(u_k) for the eigenvector u_k -- the Fortran-view
 * eigenvector zheev stores there.  Hermitian Jacobi sweeps.             */
int gpd_diagonalize_z(int n, double* d_A, double* d_w, int* sweeps,
                      void* stream);

/* ------------------------------------------------------------------ */
/* Band-wise vector operations of the eigensolver (the per-band BLAS axpy
 * and dot calls of gpaw/eigensolvers/rmmdiis.py:107-122, 199-228 and
 * eigensolver.py:88-89), batched over nb grids of nG points.
 * gpd_axpy_batched: y_x += coef[x] * x_x  (coef: FP64 device, nb; for
 * GPD_C128 complex coefficients, 2 nb interleaved).
 * gpd_dots: out[x] = alpha * sum_G a_x[G] b_x[G], FP64 accumulation in a
 * fixed order (out: FP64 device, nb <= 65535); for GPD_C128 the sum is of
 * conj(a) b and out holds 2 nb values: the real parts, then the
 * imaginary ones.                                                       */
int gpd_axpy_batched(int dtype, long nb, long nG, const double* d_coef,
                     const void* d_x, void* d_y, void* stream);
int gpd_dots(int dtype, long nb, long nG, double alpha, const void* d_a,
             const void* d_b, double* d_out, void* stream);

/* The same with the coefficients in host memory, read before the call
 * returns (nothing waits for the stream): y_x += coef[x] x_x, and y2 = y
 * where y2 is not NULL.                                                 */
int gpd_axpy_host(int dtype, long nb, long nG, const double* coef,
                  const void* d_x, void* d_y, void* d_y2, void* stream);
/* y_x = sum_i coef[x][i] x_i,x from zero in order, i < m <= 8 (complex
 * coefficients for GPD_C128), coef in host memory: what zeroing y and m
 * calls of axpy give, in one pass.                                      */
int gpd_combine(int dtype, long nb, long nG, int m, const double* coef,
                const void* const* d_x, void* d_y, void* stream);
/* gpd_dots of npairs <= 16 pairs of arrays in one launch; out holds the
 * pairs' results one after the other.                                   */
int gpd_dots_pairs(int dtype, int npairs, long nb, long nG, double alpha,
                   const void* const* d_a, const void* const* d_b,
                   double* d_out, void* stream);

/* ------------------------------------------------------------------ */
/* Learned preconditioner kernels (no counterpart in the reference: the
 * network stands beside the multigrid Preconditioner).  FP32 tensors
 * (B, C, D, H, W), C-contiguous; periodic 3x3x3 convolutions with weights
 * (Cout, Cin, 27) and tap t = 9 dz + 3 dy + dx (offsets -1..1).
 * accumulate != 0 adds into y (or gx) instead of overwriting.           */
int gpd_conv3d_forward(int B, int Cin, int Cout, int D, int H, int W,
                       const float* d_x, const float* d_w,
                       const float* d_bias, float* d_y, int accumulate,
                       void* stream);
/* The same followed by a leaky ReLU: y = v > 0 ? v : slope v.           */
int gpd_conv3d_forward_leaky(int B, int Cin, int Cout, int D, int H, int W,
                             const float* d_x, const float* d_w,
                             const float* d_bias, float slope, float* d_y,
                             void* stream);
/* Forward convolution for inference on MFMA with bfloat16 operands (inputs
 * and weights rounded to nearest even, FP32 accumulation and output).
 * Requires Cin % 8 == 0, Cout <= 64, W % 16 == 0 and H % (256 / TX) == 0
 * with TX = 32 if 32 divides W, else 16; other shapes return
 * GPD_ERR_UNSUPPORTED (use gpd_conv3d_forward). */
int gpd_conv3d_forward_bf16(int B, int Cin, int Cout, int D, int H, int W,
                            const float* d_x, const float* d_w,
                            const float* d_bias, float* d_y, void* stream);
int gpd_conv3d_backward_data(int B, int Cin, int Cout, int D, int H, int W,
                             const float* d_gy, const float* d_w,
                             float* d_gx, int accumulate, void* stream);
/* The data gradient taken on through the leaky ReLU that made the input:
 * gx = act > 0 ? v : slope v, act (B, Cin, D, H, W) being that input.   */
int gpd_conv3d_backward_data_leaky(int B, int Cin, int Cout, int D, int H,
                                   int W, const float* d_gy,
                                   const float* d_w, const float* d_act,
                                   float slope, float* d_gx, void* stream);
/* gw (Cout, Cin, 27) and gb (Cout, may be NULL) are overwritten.        */
int gpd_conv3d_backward_weight(int B, int Cin, int Cout, int D, int H, int W,
                               const float* d_x, const float* d_gy,
                               float* d_gw, float* d_gb, void* stream);
int gpd_leaky_relu(long n, float slope, const float* d_x, float* d_y,
                   void* stream);
/* Apart from a convolution or a transfer (UNet takes it in their epilogues). */
int gpd_leaky_relu_backward(long n, float slope, const float* d_x,
                            const float* d_gy, float* d_gx, void* stream);
/* Adam: m = b1 m + (1-b1) g; v = b2 v + (1-b2) g^2; w -= lr_t m/(sqrt v+eps) */
int gpd_adam_step(long n, float lr_t, float beta1, float beta2, float eps,
                  float* d_w, const float* d_g, float* d_m, float* d_v,
                  void* stream);

#ifdef __cplusplus
}
#endif

#endif /* GPAWDFT_AMD_H */
