// Complex-math (k-point) form of the orthonormalization path.
//
// CP_PAIRCALC_USES_COMPLEX_MATH (pcFwdDeclarations.h:17-24) makes the
// PairCalculator's internal type complex: the forward is ZGEMM('C','N')
// (ckPairCalculator.C:840-889), Ortho iterates on complex matrices (ortho.C
// with internalType complex, CLA_Matrix products through ZGEMM('T','T')) and
// the backward is ZGEMM('N','N') / ('N','C') (:1792-1842).  The states carry
// the full G set of a k-point: no double packing, no kx = 0 weighting.
//
// Every complex product runs as real products on the FP64-MFMA kernels:
//   * a block psi [n][npw complex] is read as the real [n][2npw] matrix of
//     interleaved (re, im) doubles, and J psi = i psi = (-im, re) per point
//     is applied to the operand fragments, so that
//       Re sum_k psi_x conj(phi_y) = psi_x . phi_y          (row dot product)
//       Im sum_k psi_x conj(phi_y) = psi_x . (J phi)_y
//       M psi = Re(M) psi + Im(M) (J psi)      (one pass over the output);
//   * n x n matrices are kept as separate real and imaginary planes, and each
//     part of a complex product sums its two real products in one tile.
// With a split precision the forward and backward products run on the digit
// kernels instead (Re S on the symmetric overlap, Im S and Lambda on the
// asymmetric product, T psi as two back-multiplies); S -> T stays FP64.
#include <math.h>

#include "oa_internal.h"

namespace {

constexpr int NT = 256;

unsigned blocks_for(long elems) {
  const long b = (elems + NT - 1) / NT;
  return (unsigned)(b < 1 ? 1 : (b > 8192 ? 8192 : b));
}

// out[r][2k] = -psi[r][2k+1], out[r][2k+1] = psi[r][2k]  (J psi = i psi)
__global__ void jswap_kernel(int n, int npw, const double *__restrict__ psi, long ld,
                             double *__restrict__ out, long ldo) {
  const long total = (long)n * npw;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < total;
       i += (long)gridDim.x * blockDim.x) {
    const long r = i / npw, k = i % npw;
    const double re = psi[r * ld + 2 * k], im = psi[r * ld + 2 * k + 1];
    out[r * ldo + 2 * k] = -im;
    out[r * ldo + 2 * k + 1] = re;
  }
}

// Interleaved complex Z (n x n) -> planes re, im with leading dimension ld.
__global__ void zplanes_kernel(int n, const double *__restrict__ Z, double *__restrict__ re,
                               double *__restrict__ im, int ld) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < (long)n * n;
       i += (long)gridDim.x * blockDim.x) {
    const long k = i / n * ld + i % n;
    re[k] = Z[2 * i];
    im[k] = Z[2 * i + 1];
  }
}

// Planes -> interleaved complex Z[nn].
__global__ void zmerge_kernel(long nn, const double *__restrict__ re,
                              const double *__restrict__ im, double *__restrict__ Z) {
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < nn;
       i += (long)gridDim.x * blockDim.x) {
    Z[2 * i] = re[i];
    Z[2 * i + 1] = im[i];
  }
}

// Hermitian S from the symmetric real part Sr and the imaginary part Si of
// the upper triangle: S[x][y] = Sr[x][y] + i Si[x][y] (x < y), its conjugate
// mirror below, a real diagonal.
// With md != null it also takes Ortho::array_diag_max of the merged S
// (ortho.h:282-313 with myabs = std::abs): |S_ij| off the diagonal and
// ||S_ii| - diag| on it, maximised through atomicMax on the IEEE bits of
// non-negative doubles (md cleared beforehand).
__global__ void zherm_kernel(int n, const double *__restrict__ Sr, const double *__restrict__ Si,
                             double *__restrict__ S, double diag, unsigned long long *md) {
  const long nn = (long)n * n;
  double mx = 0.0;
  for (long i = (long)blockIdx.x * blockDim.x + threadIdx.x; i < nn;
       i += (long)gridDim.x * blockDim.x) {
    const long x = i / n, y = i % n;
    const double re = Sr[i], im = (x < y) ? Si[i] : ((x > y) ? -Si[y * n + x] : 0.0);
    S[2 * i] = re;
    S[2 * i + 1] = im;
    const double a = hypot(re, im);
    mx = fmax(mx, (x == y) ? fabs(a - diag) : a);
  }
  if (md) {
    // wave maximum, then one atomic per wave
    for (int o = 32; o > 0; o >>= 1) mx = fmax(mx, __shfl_xor(mx, o));
    if ((threadIdx.x & 63) == 0) atomicMax(md, (unsigned long long)__double_as_longlong(mx));
  }
}

#define OA_KLAUNCH(kern, elems, s, ...)                                                     \
  do {                                                                                      \
    hipLaunchKernelGGL(kern, dim3(blocks_for(elems)), dim3(NT), 0, s, __VA_ARGS__);        \
    if (hipPeekAtLastError() != hipSuccess) return OA_ERR_HIP;                              \
  } while (0)

// Workspace of the complex forward and backward: J phi ([n][K]) where the
// general split forward slices it, two n x n planes (rows padded to an even
// length, for 16-byte loads), then the kernels' own workspace; every part
// starts on a 256-byte boundary.  The FP64 products apply J themselves; the
// split Hermitian forward and the split back-multiply make J psi's digits
// from psi's.
bool is_split(int prec) { return (prec & 0xff) != OA_PREC_FP64; }
size_t al256(size_t b) { return (b + 255) / 256 * 256; }
bool needs_j(bool sym_or_back, int prec) { return !sym_or_back && is_split(prec); }
int plane_ld(int n) { return (n + 1) / 2 * 2; }
size_t off_planes(int n, int K, bool jn) { return jn ? al256((size_t)n * K * sizeof(double)) : 0; }
size_t plane_bytes(int n) { return al256((size_t)n * plane_ld(n) * sizeof(double)); }
size_t off_kws(int n, int K, bool jn) { return off_planes(n, K, jn) + 2 * plane_bytes(n); }

size_t zoverlap_ws_bytes(int n, int K, int prec, bool sym) {
  size_t kws = oa_overlap_f64_ws_bytes(n, K);
  if (oa_ntsplit_f64_ws_bytes(n, n, K) > kws) kws = oa_ntsplit_f64_ws_bytes(n, n, K);
  if (is_split(prec)) {
    if (oa_split_ws_bytes(prec, n, K) > kws) kws = oa_split_ws_bytes(prec, n, K);
    if (oa_split_lambda_ws_bytes(prec, n, K) > kws) kws = oa_split_lambda_ws_bytes(prec, n, K);
    if (oa_split_zimag_ws_bytes(prec, n, K) > kws) kws = oa_split_zimag_ws_bytes(prec, n, K);
  }
  return off_kws(n, K, needs_j(sym, prec)) + kws;
}

size_t zbackmul_ws_bytes(int n, int K, int prec) {
  return off_kws(n, K, needs_j(true, prec)) + (is_split(prec) ? oa_split_ws_bytes(prec, n, K) : 0);
}

// Hermitian (sym) or general (!sym) product L[x][y] = alpha sum_k psi_x[k]
// conj(phi_y[k]); J phi ([n][K], where needed), the real and imaginary planes
// and the kernel workspace follow each other in ws.
int zforward(hipStream_t s, bool sym, int n, int npw, const double *psi, long ld,
             const double *phi, long ldphi, double alpha, double *L, char *ws, size_t ws_bytes,
             int prec, double diag = 0.0, double *maxdev = nullptr) {
  const int K = 2 * npw;
  const bool jn = needs_j(sym, prec);
  double *J = jn ? reinterpret_cast<double *>(ws) : nullptr;
  double *Lr = reinterpret_cast<double *>(ws + off_planes(n, K, jn));
  double *Li = reinterpret_cast<double *>(ws + off_planes(n, K, jn) + plane_bytes(n));
  char *kws = ws + off_kws(n, K, jn);
  const size_t kbytes = ws_bytes - off_kws(n, K, jn);
  if (jn)
    OA_KLAUNCH(jswap_kernel, (long)n * npw, s, n, npw, phi, ldphi, J, (long)K);
  int st;
  if (is_split(prec)) {
    if (sym) {
      // psi is sliced once: Re S on its digits, Im S on them and on J psi's
      // made from them; psi's digits (both layouts) stay in the kernel
      // workspace, where a following back-multiply can reuse them
      st = oa_launch_overlap_split(s, prec, n, K, psi, ld, 0, alpha, Lr, 0.0, nullptr, kws,
                                   kbytes);
      if (st) return st;
      st = oa_launch_zimag_split(s, prec, n, K, alpha, Li, kws, kbytes);
    } else {
      st = oa_launch_lambda_split(s, prec, n, K, psi, ld, J, K, alpha, Li, kws, kbytes);
      if (st) return st;
      st = oa_launch_lambda_split(s, prec, n, K, psi, ld, phi, ldphi, alpha, Lr, kws, kbytes);
    }
  } else {
    if (sym) {
      st = oa_launch_overlap_f64(s, n, K, psi, ld, 0, alpha, Lr, 0.0, nullptr, kws, kbytes);
      if (st) return st;
      // the Hermitian merge reads only Im S's strict upper triangle
      st = oa_launch_overlap_j_f64(s, n, K, psi, ld, alpha, Li, kws, kbytes);
    } else {
      st = oa_launch_ntsplit_f64(s, n, n, K, psi, ld, phi, ldphi, alpha, Lr, n, kws, kbytes);
      if (st) return st;
      st = oa_launch_ntsplit_f64(s, n, n, K, psi, ld, phi, ldphi, alpha, Li, n, kws, kbytes, true);
    }
  }
  if (st) return st;
  if (sym) {
    auto *md = reinterpret_cast<unsigned long long *>(maxdev);
    if (md && oa_fill_u64(s, md, 1)) return OA_ERR_HIP;
    OA_KLAUNCH(zherm_kernel, (long)n * n, s, n, Lr, Li, L, diag, md);
  } else
    OA_KLAUNCH(zmerge_kernel, (long)n * n, s, (long)n * n, Lr, Li, L);
  return OA_SUCCESS;
}

// out = alpha op(M) psi + beta out, op(M) = M or M^H; with reuse_psi the kernel
// workspace holds psi's digits from a symmetric split forward on the same psi
// (no re-slicing).
int zbackward(hipStream_t s, int n, int npw, const double *M, int transM, const double *psi,
              long ld, double alpha, double beta, double *out, long ldo, char *ws,
              size_t ws_bytes, int prec, bool reuse_psi = false) {
  const int K = 2 * npw;
  const bool jn = needs_j(true, prec);
  double *Mr = reinterpret_cast<double *>(ws + off_planes(n, K, jn));
  double *Mi = reinterpret_cast<double *>(ws + off_planes(n, K, jn) + plane_bytes(n));
  // the split back-multiply reads an n x n matrix with leading dimension n
  const int ldm = is_split(prec) ? n : plane_ld(n);
  OA_KLAUNCH(zplanes_kernel, (long)n * n, s, n, M, Mr, Mi, ldm);
  // Re(M^H) = Mr^T and Im(M^H) = -Mi^T
  if (is_split(prec)) {
    char *kws = ws + off_kws(n, K, jn);
    const size_t kbytes = ws_bytes - off_kws(n, K, jn);
    const int p = prec & ~OA_PREC_REUSE_DIGITS;
    int st = oa_launch_backmul_split(s, reuse_psi ? (p | OA_PREC_REUSE_DIGITS) : p, n, K, Mr,
                                     transM, psi, ld, 0, alpha, beta, out, ldo, kws, kbytes);
    if (st) return st;
    // J psi's digits from psi's (left by the first product), in place,
    // instead of slicing J psi; the second product reuses them
    st = oa_launch_jswap_db(s, p, n, K, kws, kbytes);
    if (st) return st;
    // psi's pointer and pitch stand in for J psi's: with the digits reused
    // the product reads neither
    return oa_launch_backmul_split(s, p | OA_PREC_REUSE_DIGITS, n, K, Mi, transM, psi, ld, 0,
                                   transM ? -alpha : alpha, 1.0, out, ldo, kws, kbytes);
  }
  return oa_launch_zback_f64(s, transM != 0, n, K, Mr, Mi, ldm, transM != 0, psi, ld, alpha, beta,
                             out, ldo);
}

// Ortho's loop on complex planes, with the stop rule of the reference's
// complex tolerance_check (ortho.C:950-953 accumulates tmp * tmp as a complex
// square; the sum_double reduction and collect_error, :113, keep its real
// part): err = sqrt(Re sum (dA)^2 / n^2), NaN when that sum is negative, which
// ends the loop because `err > tol` is then false.  modulus != 0 uses
// sum |dA|^2 instead.
int zs_to_t_run(oa_context *c, int n, const double *S, int nspin, double tol, int maxit,
                int modulus, double *T, int *iters, double *err) {
  return oa_s_to_t_sync(c, n, S, nspin, tol, maxit, T, iters, err, c->ns.ptr, c->report, true,
                        modulus);
}

size_t zs_to_t_ws_bytes(int n) { return oa_ns_ws_bytes(n, true); }

}  // namespace

extern "C" {

int oa_zoverlap(oa_handle_t c, int n, int npw, const double *psi, long ldpsi, double alpha,
                double *S, int prec, double diag, double *maxdev) {
  if (!c) return OA_ERR_NO_DEVICE;
  if (prec & OA_PREC_ADAPTIVE) return OA_ERR_UNSUPPORTED;  // uniform slices only
  if (n < 0) return 2;
  if (npw < 0) return 3;
  if (n > 0 && npw > 0 && !psi) return 4;
  if (ldpsi < 2L * npw) return 5;
  if (n > 0 && !S) return 7;
  if (n == 0) return OA_SUCCESS;
  DeviceGuard g(c->device);
  if (npw == 0) {
    OA_HIP_CHECK(hipMemsetAsync(S, 0, 2 * (size_t)n * n * sizeof(double), c->stream));
    if (maxdev) {
      // S = 0: array_diag_max is |0 - diag| on the diagonal
      const double d = fabs(diag);
      OA_HIP_CHECK(hipMemcpyAsync(maxdev, &d, sizeof(double), hipMemcpyHostToDevice, c->stream));
      OA_HIP_CHECK(hipStreamSynchronize(c->stream));
    }
    return OA_SUCCESS;
  }
  const int st = oa_ws_require(c, zoverlap_ws_bytes(n, 2 * npw, prec, true));
  if (st) return st;
  return zforward(c->stream, true, n, npw, psi, ldpsi, psi, ldpsi, alpha, S, (char *)c->ws.ptr,
                  c->ws.bytes, prec, diag, maxdev);
}

int oa_zlambda(oa_handle_t c, int n, int npw, const double *psi, long ldpsi, const double *F,
               long ldF, double alpha, double *L, int prec) {
  if (!c) return OA_ERR_NO_DEVICE;
  if (prec & OA_PREC_ADAPTIVE) return OA_ERR_UNSUPPORTED;  // uniform slices only
  if (n < 0) return 2;
  if (npw < 0) return 3;
  if (n > 0 && npw > 0 && !psi) return 4;
  if (ldpsi < 2L * npw) return 5;
  if (n > 0 && npw > 0 && !F) return 6;
  if (ldF < 2L * npw) return 7;
  if (n > 0 && !L) return 9;
  if (n == 0) return OA_SUCCESS;
  DeviceGuard g(c->device);
  if (npw == 0) {
    OA_HIP_CHECK(hipMemsetAsync(L, 0, 2 * (size_t)n * n * sizeof(double), c->stream));
    return OA_SUCCESS;
  }
  const int st = oa_ws_require(c, zoverlap_ws_bytes(n, 2 * npw, prec, false));
  if (st) return st;
  return zforward(c->stream, false, n, npw, psi, ldpsi, F, ldF, alpha, L, (char *)c->ws.ptr,
                  c->ws.bytes, prec);
}

int oa_zs_to_t(oa_handle_t c, int n, const double *S, int nspin, double tol, int maxit,
               int modulus, double *T, int *iters, double *err) {
  if (!c) return OA_ERR_NO_DEVICE;
  if (n < 0) return 2;
  if (n > 0 && !S) return 3;
  if (nspin != 1 && nspin != 2) return 4;
  if (maxit < 1) return 6;
  if (n > 0 && !T) return 8;
  if (n == 0) return OA_SUCCESS;
  DeviceGuard g(c->device);
  const int st = oa_ws_require_into(c, c->ns, zs_to_t_ws_bytes(n));
  if (st) return st;
  const int st_ns = zs_to_t_run(c, n, S, nspin, tol, maxit, modulus, T, iters, err);
  OA_HIP_CHECK(hipStreamSynchronize(c->stream));
  return st_ns;
}

int oa_zbackmul(oa_handle_t c, int n, int npw, const double *M, int transM, const double *psi,
                long ldpsi, double alpha, double beta, double *out, long ldout, int prec) {
  if (!c) return OA_ERR_NO_DEVICE;
  if (prec & OA_PREC_ADAPTIVE) return OA_ERR_UNSUPPORTED;  // uniform slices only
  if (n < 0) return 2;
  if (npw < 0) return 3;
  if (n > 0 && !M) return 4;
  if (n > 0 && npw > 0 && !psi) return 6;
  if (ldpsi < 2L * npw) return 7;
  if (n > 0 && npw > 0 && !out) return 10;
  if (ldout < 2L * npw) return 11;
  if (n == 0 || npw == 0) return OA_SUCCESS;
  DeviceGuard g(c->device);
  const int st = oa_ws_require(c, zbackmul_ws_bytes(n, 2 * npw, prec));
  if (st) return st;
  return zbackward(c->stream, n, npw, M, transM, psi, ldpsi, alpha, beta, out, ldout,
                   (char *)c->ws.ptr, c->ws.bytes, prec);
}

int oa_zortho_step(oa_handle_t c, int n, int npw, const double *psi, long ldpsi, int nspin,
                   double tol, int maxit, int modulus, double *S, double *T, double *psi_out,
                   long ldout, int *iters, double *err, int prec) {
  if (!c) return OA_ERR_NO_DEVICE;
  if (prec & OA_PREC_ADAPTIVE) return OA_ERR_UNSUPPORTED;  // uniform slices only
  if (n < 0) return 2;
  if (npw < 1) return 3;
  if (n > 0 && !psi) return 4;
  if (ldpsi < 2L * npw) return 5;
  if (nspin != 1 && nspin != 2) return 6;
  if (maxit < 1) return 8;
  if (n > 0 && (!S || !T || !psi_out)) return 10;
  if (ldout < 2L * npw) return 13;
  if (n == 0) return OA_SUCCESS;
  DeviceGuard g(c->device);
  const int K = 2 * npw;
  size_t need = zoverlap_ws_bytes(n, K, prec, true);
  if (zbackmul_ws_bytes(n, K, prec) > need) need = zbackmul_ws_bytes(n, K, prec);
  int st = oa_ws_require(c, need);
  if (!st) st = oa_ws_require_into(c, c->ns, zs_to_t_ws_bytes(n));
  if (st) return st;
  char *ws = (char *)c->ws.ptr;
  st = zforward(c->stream, true, n, npw, psi, ldpsi, psi, ldpsi, 1.0, S, ws, c->ws.bytes, prec);
  if (st) return st;
  const int st_ns = zs_to_t_run(c, n, S, nspin, tol, maxit, modulus, T, iters, err);
  if (st_ns != OA_SUCCESS && st_ns != OA_ERR_NOT_CONVERGED) return st_ns;
  // a split forward left psi's digits in the kernel workspace (S->T has
  // buffers of its own), from which the back-multiply makes J psi's
  st = oa_ns_mark(c->stream, &c->host->drained);
  if (st == OA_SUCCESS)
    st = zbackward(c->stream, n, npw, T, 0, psi, ldpsi, 1.0, 0.0, psi_out, ldout, ws, c->ws.bytes,
                   prec, is_split(prec));
  const int st_dr = oa_ns_drain(c);
  return st ? st : (st_dr ? st_dr : st_ns);
}

}  // extern "C"
