/*
 * oa_ortho.h -- C ABI of the MI355X orthonormalization library
 * (openatom_amd/liboa_ortho.so).
 *
 * Two layers:
 *
 *  1. BLAS drop-ins with the exact Fortran ABI the reference's path calls
 *     (dgemm_).  A Charm++ build links this library ahead of src_mathlib (the
 *     reference already links with -Wl,--allow-multiple-definition,
 *     makefiles/config.mk:32), and every DGEMM on the path runs on the GPU.
 *     Host or device pointers are accepted; the call is synchronous.
 *
 *  2. Path-level entry points (oa_*) over device-resident buffers, on the
 *     handle's HIP stream.  They replace the PairCalculator forward/backward
 *     DGEMM tuples and the Ortho S->T loop with single calls.
 *
 * Layouts (both layers' path calls): a block of n states is row-major
 * [n][ld] doubles holding 2*npw interleaved (re, im) coefficients per row --
 * the collated layout the reference hands to DGEMM (MessageDataCollator.h:222,
 * ckPairCalculator.C:871-872).  n x n matrices (S, T, Lambda) are row-major
 * [x][y] with leading dimension n (ckPairCalculator.C:889: outData[x*nY + y]).
 *
 * Status codes: 0 success; > 0 the 1-based index of an invalid argument
 * (BLAS INFO convention, dgemm.f:169-194); < 0 one of OA_ERR_*.
 * Every entry point is reentrant: no global mutable state other than the
 * per-thread default handle used by dgemm_.
 */
#ifndef OA_ORTHO_H
#define OA_ORTHO_H

#include <stddef.h>
#include <stdint.h>

#ifdef __cplusplus
extern "C" {
#endif

#define OA_SUCCESS 0
#define OA_ERR_HIP (-1)           /* a HIP runtime call failed               */
#define OA_ERR_NOT_CONVERGED (-2) /* S->T reached maxit (ortho.C:129-133)    */
#define OA_ERR_NO_DEVICE (-3)     /* no usable gfx950 device                 */
#define OA_ERR_UNSUPPORTED (-4)   /* precision/variant not available         */
#define OA_ERR_CAPACITY (-5)      /* request exceeds a documented limit      */
#define OA_ERR_IO (-6)            /* a state file cannot be opened or parsed */

/* Arithmetic of the O(n^2 npw) products (overlap, Lambda, back-multiply).
 * S->T, the G=0 term and all reductions stay FP64 in every mode.
 *   OA_PREC_FP64      FP64 MFMA (v_mfma_f64_16x16x4), the drop-in form.
 *   OA_PREC_INT8      Ozaki digit slices on int8 MFMA, exact int32 sums.
 *   OA_PREC_FP16      Ozaki digit slices on fp16 MFMA, exact fp32 sums.
 *   OA_PREC_BF16      Ozaki digit slices on bf16 MFMA, exact fp32 sums.
 *   OA_PREC_FP32      Ozaki digit slices on fp32 MFMA, exact fp32 sums.
 * For the slice modes, OA_PREC_SLICES(p, s) selects s digit slices
 * (2 <= s <= 6); the default is 3.  The overlap keeps the products of
 * levels p + q <= s + 1.  The back-multiply splits T = D + X, applies D in
 * FP64 to psi rebuilt from all s digits and keeps levels p + q <= s of the
 * X * psi digit products, or p + q <= s - 1 with OA_PREC_LEAN_BACKMUL. */
#define OA_PREC_FP64 0
#define OA_PREC_INT8 1
#define OA_PREC_FP16 2
#define OA_PREC_BF16 3
#define OA_PREC_FP32 4
#define OA_PREC_SLICES(p, s) ((p) | ((s) << 8))
#define OA_PREC_LEAN_BACKMUL (1 << 12)
/* Adaptive slice counts (OA_PREC_INT8 with 4 <= s <= 6): every K chunk z
 * gets its own count s_z in [2, s], chosen on the device from the chunk
 * maxima alone.  With W_z = K_z 4^(e_z) (K_z columns, chunk exponent e_z)
 * and W = sum_z W_z, chunk z drops d slices while
 * W_z 254^d <= (254 / 4) W / nz.  The element-wise truncation bound of S
 * (and of the residual after T psi) is then at most 64.5 times the bound of
 * s uniform slices, i.e. about a quarter of the bound of s - 1 uniform
 * slices: OA_PREC_SLICES(OA_PREC_INT8, 6) | OA_PREC_ADAPTIVE is more
 * accurate than 5 uniform slices, and chunks whose coefficients are small
 * next to the largest chunk run 2-5 slices instead of 6.  Applies to
 * oa_overlap_sym, oa_backmul, oa_lambda_force, oa_ortho_step and batches;
 * the Lambda product and the complex calls return OA_ERR_UNSUPPORTED. */
#define OA_PREC_ADAPTIVE (1 << 13)
/* oa_backmul / oa_lambda_force: reuse the digit slices of psi left in the
 * handle's workspace by the preceding split slicing on this handle (an
 * oa_overlap_sym or a back-multiply of the same psi).  A hint: when the
 * workspace no longer holds digits of this psi pointer, ld, n, npw and
 * precision (any other call that used the workspace in between), psi is
 * sliced again.  The caller guarantees psi's contents are unchanged. */
#define OA_PREC_REUSE_DIGITS (1 << 16)

typedef struct oa_context *oa_handle_t;

/* Device-side S->T report, written by the asynchronous S->T entry points. */
typedef struct oa_ns_report {
  int32_t iterations; /* iterations performed                          */
  int32_t done;       /* 1 once the loop has stopped                   */
  int32_t status;     /* OA_SUCCESS or OA_ERR_NOT_CONVERGED            */
  int32_t pad;
  double error;       /* sqrt(sum (T_old - T_new)^2 / n^2), last iterate */
} oa_ns_report;

/* ---- handles ---------------------------------------------------------- */

/* Create a handle on HIP device `device`, with its own non-blocking stream.
 * No counterpart in the reference (a Charm++ PE's BLAS has no handle). */
int oa_create(oa_handle_t *h, int device);
int oa_destroy(oa_handle_t h);
/* Run the handle's work on `stream` (a hipStream_t); NULL selects the
 * device's default (null) stream, as everywhere in HIP.  A new handle starts
 * on a non-blocking stream of its own. */
int oa_set_stream(oa_handle_t h, void *stream);
void *oa_get_stream(oa_handle_t h);
/* Block until the handle's stream is idle. */
int oa_synchronize(oa_handle_t h);
/* Pre-size the handle's workspace for instances up to (n, npw) so that later
 * calls allocate nothing (needed before hipGraph capture). */
int oa_reserve(oa_handle_t h, int n, int npw);
/* Same, including the digit-slice workspace of a split precision `prec`. */
int oa_reserve_prec(oa_handle_t h, int n, int npw, int prec);
const char *oa_status_string(int status);

/* ---- BLAS drop-ins (Fortran ABI) --------------------------------------- */

/* Replaces the reference's DGEMM (src_mathlib/dgemm.f:1-313) as declared at
 * ckPairCalculator.h:26-48 / CLA_Matrix.C:9-17 and called by
 * PairCalculator::multiplyForward (ckPairCalculator.C:889),
 * bwMultiplyHelper (:1835, :1842, :1879, :1929), bwMultiplyDynOrthoT (:2018),
 * CLA_Matrix::multiply (CLA_Matrix.C:556) and genmatmul (genmatmul.f:33).
 * Column-major, FP64 MFMA on the GPU.  Invalid arguments return silently with
 * C untouched, as the reference's empty XERBLA does (xerbla.f). */
void dgemm_(const char *transa, const char *transb, const int *m, const int *n,
            const int *k, const double *alpha, const double *a, const int *lda,
            const double *b, const int *ldb, const double *beta, double *c,
            const int *ldc);

/* Same operation on device pointers, asynchronous on the handle's stream;
 * returns the BLAS INFO value instead of discarding it. */
int oa_dgemm(oa_handle_t h, char transa, char transb, int m, int n, int k,
             double alpha, const double *a, int lda, const double *b, int ldb,
             double beta, double *c, int ldc);

/* Replaces the reference's ZGEMM (src_mathlib/zgemm.f:1-411), the GEMM of
 * the complex-math PairCalculator build (CP_PAIRCALC_USES_COMPLEX_MATH:
 * ckPairCalculator.h:26-48 declares zgemm_; myGEMM promotes alpha and beta
 * to complex, ckPairCalculator.C:56-65).  Column-major COMPLEX*16 (re, im
 * pairs); alpha and beta point at (re, im).  op in {N, T, C}.  Host or device
 * pointers, synchronous; invalid arguments return silently (xerbla.f). */
void zgemm_(const char *transa, const char *transb, const int *m, const int *n,
            const int *k, const double *alpha, const double *a, const int *lda,
            const double *b, const int *ldb, const double *beta, double *c,
            const int *ldc);

/* Same operation on device pointers (alpha, beta in host memory),
 * asynchronous on the handle's stream; returns the BLAS INFO value. */
int oa_zgemm(oa_handle_t h, char transa, char transb, int m, int n, int k,
             const double *alpha, const double *a, int lda, const double *b,
             int ldb, const double *beta, double *c, int ldc);

/* ---- path level (device pointers, asynchronous on the handle's stream) -- */

/* Symmetric PairCalculator forward: S = alpha * sum_k w_k psi_x[k] psi_y[k]
 * with w_k = 1/2 on the leading 2*nkx0 doubles (the kx=0 points that
 * CP_State_GSpacePlane.C:3025-3028 scales by 1/sqrt2 before the alpha=2
 * DGEMM) and 1 elsewhere.  Replaces multiplyForward + contributeSubTiles +
 * sumMatrixDouble (ckPairCalculator.C:821-1016, :20-53).  Only upper-triangle
 * tiles are computed; S is written in full (exactly symmetric).  psi rows have
 * leading dimension ldpsi >= 2*npw.  If maxdev != NULL it receives
 * max_ij |S_ij - diag*delta_ij| (Ortho::array_diag_max, ortho.h:282-313). */
int oa_overlap_sym(oa_handle_t h, int n, int npw, const double *psi,
                   long ldpsi, int nkx0, double alpha, int prec, double *S,
                   double diag, double *maxdev);

/* The per chunk digit counts an adaptive split precision (OA_PREC_ADAPTIVE)
 * assigns to psi: chunk maxima and the count rule on the device, then a
 * synchronous copy of nchunks ints into counts (host).  *nchunks and *kchunk
 * (columns per chunk, in doubles) are set even when capacity is too small
 * (OA_ERR_CAPACITY).  No counterpart in the reference: it reports what the
 * split chose (tests, benchmark histograms). */
int oa_slice_counts(oa_handle_t h, int n, int npw, const double *psi,
                    long ldpsi, int nkx0, int prec, int *counts, int capacity,
                    int *nchunks, int *kchunk);

/* Asymmetric PairCalculator forward (the Lambda instance, alpha = 1 in the
 * reference, cpaimd.C:2510-2516): L[x][y] = alpha * sum_k psi_x[k] F_y[k]
 * over all 2*npw doubles.  Replaces ckPairCalculator.C:889 for the asymmetric
 * instance.  Slice modes split psi and F into digits with their own chunk
 * exponents and form all tiles of the product. */
int oa_lambda(oa_handle_t h, int n, int npw, const double *psi, long ldpsi,
              const double *F, long ldF, double alpha, int prec, double *L);

/* Ortho S -> T (ortho.C:153-971): B = S/2 (nspin == 1) or S (nspin == 2,
 * lsda), A = I; C = 3I - A*B; B = B*C/2; A = C*A/2 until
 * sqrt(sum (A_old - A_new)^2 / n^2) <= tol or the iteration count reaches
 * maxit.  Returns OA_ERR_NOT_CONVERGED when the count reached maxit at exit
 * (the reference aborts there, ortho.C:129-133); T then holds the last
 * iterate.  Synchronous: iters / err are host pointers (may be NULL). */
int oa_s_to_t(oa_handle_t h, int n, const double *S, int nspin, double tol,
              int maxit, double *T, int *iters, double *err);

/* Asynchronous S->T: fixed launch sequence of maxit guarded iterations that
 * become no-ops once converged (capturable in a hipGraph).  The report is a
 * device pointer. */
int oa_s_to_t_async(oa_handle_t h, int n, const double *S, int nspin,
                    double tol, int maxit, double *T, oa_ns_report *report);

/* Backward PairCalculator multiply (bwMultiplyHelper, ckPairCalculator.C:
 * 1835 symmetric, :1842 asymmetric; bwMultiplyDynOrthoT :2018 with
 * alpha = -1): out[y] = alpha * sum_x M[y][x] psi[x] + beta * out[y]
 * (transM == 0), or M[x][y] (transM != 0), over 2*npw doubles per row. */
int oa_backmul(oa_handle_t h, int n, int npw, const double *M, int transM,
               const double *psi, long ldpsi, double alpha, double beta,
               double *out, long ldout, int prec);

/* GSpace side of the Lambda round trip, fused into the backward multiply:
 *   force[y][c] := beta * force[y][c] + alpha * w_c * (op(M) psi)[y][c],
 * w_c = wkx0 for the leading 2*nkx0 doubles of every row (the kx = 0
 * points) and 1 elsewhere, op as in oa_backmul.  It replaces the backward
 * GEMM followed by the GSpace accumulation of its result:
 *   minimisation, partialResultMsg (CP_State_GSpacePlane.C:2168-2195):
 *     force -= w data, w = 1/2 at kx = 0 (double pack), 1/2 everywhere
 *     (single pack)  ->  alpha = -1, wkx0 = 1/2, beta = 1 (or alpha = -1/2,
 *     wkx0 = 1);
 *   minimisation, CkReductionMsg (:2068-2106): w = 1/ov at kx = 0, 2/ov
 *     elsewhere, ov = 2 (lda) or 1 (lsda)  ->  alpha = -2/ov, wkx0 = 1/2;
 *   dynamics (:2180-2183 with doLambda :2247-2252): force = -data, then the
 *     kx = 0 points scaled by 1/sqrt2  ->  alpha = -1, wkx0 = 1/sqrt2,
 *     beta = 0 for the first contribution, 1 after.
 * Returns the argument index on a bad argument (nkx0 outside [0, npw] is 8). */
int oa_lambda_force(oa_handle_t h, int n, int npw, const double *M, int transM,
                    const double *psi, long ldpsi, int nkx0, double wkx0,
                    double alpha, double beta, double *force, long ldf,
                    int prec);

/* X[r][c] *= s for c < 2*nkx0 (every row r < n): the GSpace rescaling of the
 * kx = 0 points -- psi by 1/sqrt2 and the force by sqrt2 before the dynamics
 * Lambda forward (CP_State_GSpacePlane.C:1926-1947; nkx0 = npw scales every
 * point, the single-pack form), the force by 1/sqrt2 in doLambda
 * (:2247-2252). */
int oa_scale_kx0(oa_handle_t h, int n, int npw, double *X, long ld, int nkx0,
                 double s);

/* One symmetric orthonormalisation step -- overlap, S->T, T*psi -- as the
 * reference's GSP -> PC -> Ortho -> PC -> GSP round trip performs it
 * (call stack: gspace.ci:158 -> CP_State_GSpacePlane.C:2975 ->
 * ckPairCalculator.C:821 -> ortho.C:153..971 -> ckPairCalculator.C:1201 ->
 * CP_State_GSpacePlane.C:3232).  S, T (n*n) and psi_out ([n][ldout]) are
 * device outputs; psi_out must not alias psi.  Synchronous when iters/err
 * are non-NULL host pointers (S, T and the outcome are complete on return,
 * psi_out in the order of the stream), else asynchronous. */
int oa_ortho_step(oa_handle_t h, int n, int npw, const double *psi, long ldpsi,
                  int nkx0, int nspin, double tol, int maxit, int prec,
                  double *S, double *T, double *psi_out, long ldout,
                  int *iters, double *err);

/* oa_ortho_step in FP64 (prec must be OA_PREC_FP64) with no device memory
 * allocated by the call or by the library on its behalf.  No counterpart in
 * the reference: it is for callers that cannot allocate (code under HIP graph
 * capture, tight serving loops, harnesses that forbid hipMalloc).  Every
 * buffer beyond the arguments lives in one scratch array of
 * oa_noalloc_scratch_bytes() (64 MiB) that each device holds for the life of
 * the process: the S->T report and buffers (five matrices with rows padded to
 * 16, and partial sums) and, before them in time, the overlap's split-K partial
 * tiles, whose depth is capped to what 5 n^2 doubles leave (S, T and psi_out
 * then differ from oa_ortho_step's by k-sum rounding only).  Sizes
 * whose buffers do not fit (n above about 1300) return OA_ERR_CAPACITY;
 * npw must be at least 1.  Calls on one device share the array: calls that
 * overlap in time on one device race. */
int oa_ortho_step_noalloc(oa_handle_t h, int n, int npw, const double *psi, long ldpsi,
                          int nkx0, int nspin, double tol, int maxit, int prec,
                          double *S, double *T, double *psi_out, long ldout,
                          int *iters, double *err);
size_t oa_noalloc_scratch_bytes(void);

/* ---- complex-math (k-point) path --------------------------------------
 *
 * The PairCalculator built with CP_PAIRCALC_USES_COMPLEX_MATH
 * (pcFwdDeclarations.h:17-24) works on complex internal data: ZGEMM('C','N')
 * forward (ckPairCalculator.C:840-889), Ortho on complex matrices, and
 * ZGEMM('N','N') / ('N','C') backward (:1792-1842).  States are row-major
 * [n][2*npw] doubles = [n][npw] complex (re, im) over the full G set of a
 * k-point (no double packing).  n x n matrices are row-major complex [x][y],
 * 2*n*n doubles, contiguous.  Device pointers, handle stream.  prec selects
 * the products' arithmetic as for the real calls (OA_PREC_FP64 or a digit
 * split: Re S on the symmetric digit overlap, Im S and Lambda on the
 * asymmetric digit product of psi with i psi, T psi as two digit
 * back-multiplies); S -> T is FP64 in every mode. */

/* S[x][y] = alpha * sum_k psi_x[k] conj(psi_y[k])  (ZGEMM('C','N') with
 * right = left, ckPairCalculator.C:840-889), written exactly Hermitian.  If
 * maxdev != NULL (device pointer) it receives Ortho::array_diag_max of S
 * (ortho.h:282-313 with myabs = std::abs): the largest of |S_ij| off the
 * diagonal and ||S_ii| - diag| on it. */
int oa_zoverlap(oa_handle_t h, int n, int npw, const double *psi, long ldpsi,
                double alpha, double *S, int prec, double diag, double *maxdev);

/* Asymmetric complex forward: L[x][y] = alpha * sum_k psi_x[k] conj(F_y[k]). */
int oa_zlambda(oa_handle_t h, int n, int npw, const double *psi, long ldpsi,
               const double *F, long ldF, double alpha, double *L, int prec);

/* Ortho S -> T on complex matrices (ortho.C:153-971 with internalType
 * complex; CLA_Matrix products are plain complex products): B = S/2 (nspin 1)
 * or S, A = I; C = 3I - A B; B = B C / 2; A = C A / 2.  The stop rule is the
 * reference's complex one: err = sqrt(Re sum (A_old - A_new)^2 / n^2) with
 * complex squares (tolerance_check accumulates tmp * tmp, collect_error reads
 * the real part, ortho.C:109-146, 936-971); the loop ends when err <= tol, when
 * err is NaN (negative sum) or at maxit.  modulus != 0 uses sum |dA|^2.
 * Synchronous; iters / err host pointers (may be NULL).  Returns
 * OA_ERR_NOT_CONVERGED when the count reached maxit. */
int oa_zs_to_t(oa_handle_t h, int n, const double *S, int nspin, double tol,
               int maxit, int modulus, double *T, int *iters, double *err);

/* out[y] = alpha * sum_x M[y][x] psi[x] + beta * out[y] (transM == 0,
 * ZGEMM('N','N'), ckPairCalculator.C:1835) or conj(M[x][y]) (transM != 0,
 * ZGEMM('N','C'), :1842). */
int oa_zbackmul(oa_handle_t h, int n, int npw, const double *M, int transM,
                const double *psi, long ldpsi, double alpha, double beta,
                double *out, long ldout, int prec);

/* One complex step: S = psi psi^H, S -> T (the reference's stop rule, or
 * sum |dA|^2 when modulus != 0), out = T psi.  Under lsda (B = S) the
 * reference rule often ends after one iteration: Re sum (dA)^2 of a Hermitian
 * dA is negative when its off-diagonal imaginary parts dominate. */
int oa_zortho_step(oa_handle_t h, int n, int npw, const double *psi,
                   long ldpsi, int nspin, double tol, int maxit, int modulus,
                   double *S, double *T, double *psi_out, long ldout,
                   int *iters, double *err, int prec);

/* ---- state files and the kx = 0 plane layout -----------------------------
 *
 * A state file (utility/util.C:1107-1330 readState, :1955-2180
 * writeStateFile) is a header `ncoef nx ny nz` and one `re im kx ky kz`
 * record per plane wave.  format: 0 text, 1 binary, 2 gzip text, 3 gzip
 * binary (2 and 3 open `<path>.gz`, as the reference does).  Host calls,
 * no device work; they return OA_ERR_IO when a file cannot be opened,
 * parsed or written. */

/* Read one state.  double_pack != 0 (gamma point): the file lists the upper
 * half of the kx = 0 plane, the kx > 0 points and G = 0 last; reading stops
 * at G = 0 and the lower half of the kx = 0 plane is rebuilt by conjugate
 * symmetry (para_grp_parse.C:178-264 flip_data_set), giving the memory
 * layout [lower half | G = 0 | upper half | kx > 0]; the flip's consistency
 * checks return OA_ERR_IO.  double_pack == 0 (k-points): the records as
 * listed.  *npts receives the number of points of the layout, *nkx0 the
 * points with kx = 0 (the leading block of weight 1 in the path metric; 0
 * without double packing), grid[3] nx ny nz.  coef holds 2*capacity doubles,
 * kx/ky/kz capacity ints (may be NULL); when npts exceeds capacity the call
 * returns OA_ERR_CAPACITY after setting *npts, *nkx0 and grid. */
int oa_state_read(const char *path, int format, int double_pack, int capacity,
                  double *coef, int *kx, int *ky, int *kz, int *npts,
                  int *nkx0, int *grid);

/* Write one state as writeStateFile does: points ordered by (kx, ky, kz)
 * (sort_psi_output, util.C:2180-2215); with double_pack the points after
 * G = 0 in that order and then G = 0 (the lower half of the kx = 0 plane is
 * dropped), header count = points written.  Text records use the
 * reference's "%g %g %d %d %d \n". */
int oa_state_write(const char *path, int format, int double_pack, int npts,
                   const double *coef, const int *kx, const int *ky,
                   const int *kz, const int *grid);

/* Device form of flip_data_set for a block of n states: rows of nfile
 * points in file order (upper half of the kx = 0 plane: nhalf points,
 * kx > 0 points, G = 0 last) -> rows of nfile + nhalf points in memory order,
 * and back (contract drops the lower half).  Row-major, (re, im) pairs,
 * leading dimensions in doubles. */
int oa_kx0_expand(oa_handle_t h, int n, int nfile, int nhalf,
                  const double *in, long ldin, double *out, long ldout);
int oa_kx0_contract(oa_handle_t h, int n, int nfile, int nhalf,
                    const double *in, long ldin, double *out, long ldout);

/* ---- caller-side transport (per-(state, plane) messages) ---------------
 *
 * The Charm++ driver moves the states to the PairCalculators and the
 * results back as one message per (state, plane[, chunk]).  On one device
 * the messages become copies into and out of the resident [n][ld] block.
 * Message m covers rows row0[m] .. row0[m] + nrows[m] - 1 and doubles
 * col0[m] .. col0[m] + ncols[m] - 1 of the block; its data are nrows[m] x
 * ncols[m] contiguous doubles (row-major).  Messages must not overlap.
 * *_on_host != 0 says every message buffer is host memory (staged through
 * pinned memory of the handle), else every one is device memory.  The block
 * is device memory.  Synchronous.  Returns the index of a bad argument:
 * a message outside the block reports its row0 (3) or col0 (5). */

/* Replaces MessageDataCollator::operator() (MessageDataCollator.h:163-247),
 * which copies each paircalcInputMsg (pcMessages.h:117-153) to its sender's
 * place in the collated buffer (:222). */
int oa_collate_rows(oa_handle_t h, int count, const int *row0, const int *nrows,
                    const long *col0, const int *ncols, const double *const *src,
                    int src_on_host, double *block, long ld, int nblock_rows);

/* The return leg: sendBWResultDirect (ckPairCalculator.C:2365-2452) sends
 * one partialResultMsg per output state and plane, and the GSpace chare
 * copies the first contribution and adds later ones with fastAdd
 * (CP_State_GSpacePlane.C:3120-3126, 3197-3203; fastadd.C:34-51).  Message
 * m's destination receives its slice of the block: copied when
 * accumulate[m] == 0 (or accumulate == NULL), else added elementwise
 * (dst += slice, one FP64 add per element as in fastAdd). */
int oa_scatter_rows(oa_handle_t h, int count, const int *row0, const int *nrows,
                    const long *col0, const int *ncols, double *const *dst,
                    int dst_on_host, const int *accumulate, const double *block,
                    long ld, int nblock_rows);

/* ---- batched independent instances (grouped launches) -----------------
 *
 * Many independent orthonormalisation problems of uneven size -- path-integral
 * beads, k-points, tempering replicas, each its own GSP/PC/Ortho instance
 * set in the reference (cpaimd.C:600-664 loops over spin, temper, k-point
 * and bead; cpaimd.C:2566-2593 builds each instance's PairCalculator pair
 * and Ortho array) -- advance together: every phase
 * of the step (chunk maxima, slicing, overlap products, reduction, each S->T
 * iteration, back-multiply) is one grouped launch per tile in use over all
 * instances, reading a device table of per-instance arguments (in FP64 more
 * where one instance's buffers overlap another's).  Results, reports included,
 * are those of oa_ortho_step on each instance alone, bit for bit: every sum runs
 * in one order whatever the tile, and the chunks and the parts they are summed
 * in depend on (n, npw) and the precision's slice count only. */
typedef struct oa_instance {
  int n;              /* states                                          */
  int npw;            /* plane waves (2*npw doubles per state)           */
  int nkx0;           /* leading kx=0 points (weight 1/2 in S)           */
  int nspin;          /* 1: B = S/2; 2 (lsda): B = S                     */
  const double *psi;  /* device [n][ldpsi], read                          */
  long ldpsi;
  double *psi_out;    /* device [n][ldout], written (T psi)              */
  long ldout;
  double *S;          /* device n*n or NULL (kept in the batch workspace) */
  double *T;          /* device n*n or NULL (kept in the batch workspace) */
  double tol;         /* invsqr_tolerance                                */
  int maxit;          /* invsqr_max_iter                                 */
  int pad;
} oa_instance;

typedef struct oa_batch *oa_batch_t;

/* A batch lives on its handle's device and orders its work after the
 * handle's stream. */
int oa_batch_create(oa_handle_t h, oa_batch_t *b);
int oa_batch_destroy(oa_batch_t b);
/* (Re)plan for `count` instances at precision `prec` (OA_PREC_FP64 or a
 * slice mode).  Synchronous: waits for the batch's previous work, grows the
 * device workspace when needed and uploads the argument tables.  Tile
 * choices come from the batch's tuning table (oa_batch_tune), else from a
 * size rule. */
int oa_batch_plan(oa_batch_t b, int count, const oa_instance *inst, int prec);
/* Bytes of device memory the planned batch holds (workspace + tables). */
size_t oa_batch_footprint(oa_batch_t b);
/* Pre-size the batch's workspace and table allocations, so that later plans
 * within these sizes allocate nothing (a serving loop re-plans often). */
int oa_batch_reserve(oa_batch_t b, size_t workspace_bytes, size_t table_bytes);
/* Device bytes one instance of (n, npw) needs at `prec` (admission). */
size_t oa_instance_footprint(int n, int npw, int prec);
/* Enqueue one step of every planned instance on the handle's stream: no
 * allocation, no host synchronisation (capturable). */
int oa_batch_run(oa_batch_t b);
/* The same step as a hipGraph replay: the first call after a plan captures
 * oa_batch_run into a graph; later calls replay it. */
int oa_batch_launch(oa_batch_t b);
/* Synchronous copy of the per-instance S->T reports (count entries). */
int oa_batch_reports(oa_batch_t b, oa_ns_report *host, int count);
/* Project autotuner: for each size bucket (n rounded up to 32) pick the
 * digit-GEMM tile (128 or 64) and the S->T GEMM tile (WM 4 or 2) by timing
 * the whole planned batch `reps` times per candidate (coordinate descent
 * over buckets), keep the choices in the batch's table and re-plan. */
int oa_batch_tune(oa_batch_t b, int reps);
/* Tile choices of planned instance i (digit tile, S->T GEMM WM). */
int oa_batch_config(oa_batch_t b, int i, int *tile, int *wm);
/* Tuning table as text ("bucket tile wm" per line) and back. */
int oa_batch_get_table(oa_batch_t b, char *buf, int bytes);
int oa_batch_set_table(oa_batch_t b, const char *text);

#ifdef __cplusplus
}
#endif
#endif /* OA_ORTHO_H */
