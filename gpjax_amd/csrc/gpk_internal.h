// Internal declarations shared by the libgpk HIP sources (gfx950 only).
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>
#include <type_traits>

#include "../../include/gpk.h"

namespace gpk {

// Block size of the recursive factorisation: leaves are NB x NB diagonal
// blocks factored in LDS, and every GEMM tile is NB x NB.  Internal matrices
// are padded to a multiple of NB with an identity tail.
constexpr int NB = 128;
// Largest input dimension of the exact-GP kernels (the Sigma products keep a
// point's coordinates in registers; the gradient epilogue stages them in LDS in
// chunks of 32).
constexpr int MAX_D = 64;

void set_error(const char* fmt, ...);

#define GPK_HIP_TRY(call)                                                            \
  do {                                                                               \
    hipError_t e_ = (call);                                                          \
    if (e_ != hipSuccess) {                                                          \
      ::gpk::set_error("%s failed: %s (%s:%d)", #call, hipGetErrorString(e_), __FILE__, \
                       __LINE__);                                                    \
      return GPK_ERR_HIP;                                                            \
    }                                                                                \
  } while (0)

#define GPK_LAUNCH_CHECK()                                                           \
  do {                                                                               \
    hipError_t e_ = hipGetLastError();                                               \
    if (e_ != hipSuccess) {                                                          \
      ::gpk::set_error("kernel launch failed: %s (%s:%d)", hipGetErrorString(e_),     \
                       __FILE__, __LINE__);                                          \
      return GPK_ERR_HIP;                                                            \
    }                                                                                \
  } while (0)

inline int64_t round_up(int64_t a, int64_t b) { return (a + b - 1) / b * b; }

// ---------------------------------------------------------------------------
// Batches of independent problems of one padded size, one member per
// blockIdx.z.  The workspace of member z sits ws_stride bytes after that of
// member z - 1, so every workspace pointer of a kernel is shifted by
// z * ws_stride.  Inputs and outputs are addressed through the member's
// problem index p = gp[z]: rows xoff[p] .. xoff[p+1]-1 of the concatenated
// x (and y), hyperparameter row theta + p * theta_stride, output row p.  The
// default (gp == nullptr, ws_stride == 0, one member) is a single problem.
// ---------------------------------------------------------------------------
struct Batch {
  int64_t ws_stride = 0;
  const int* gp = nullptr;
  const int64_t* xoff = nullptr;
  int64_t theta_stride = 0;
  unsigned count = 1;
  // Optional device flag (member z's at skip + z * ws_stride bytes): the
  // vector kernels of an iterative refinement step return at once when it is
  // set, so a converged refinement skips its remaining steps without a host
  // sync.
  const int* skip = nullptr;
};

// True when this member's refinement has converged (see Batch::skip).
__device__ __forceinline__ bool bskip(const Batch& b) {
  if (!b.skip) return false;
  const int* p = b.skip;
  if (b.ws_stride)
    p = reinterpret_cast<const int*>(reinterpret_cast<const char*>(p) +
                                     (int64_t)blockIdx.z * b.ws_stride);
  return *p != 0;
}

// The shift is byte arithmetic on the pointer itself (not through an integer),
// so the compiler keeps the global address space and emits global (not flat)
// loads and stores.
template <typename T>
__device__ __forceinline__ T* bws(T* p, const Batch& b) {
  if (!p || !b.ws_stride) return p;
  typedef typename std::conditional<std::is_const<T>::value, const char, char>::type Byte;
  return reinterpret_cast<T*>(reinterpret_cast<Byte*>(p) + (int64_t)blockIdx.z * b.ws_stride);
}
// Problem index of this member (0 for a single problem).
__device__ __forceinline__ int64_t bprob(const Batch& b) {
  return b.gp ? (int64_t)b.gp[blockIdx.z] : 0;
}
// Rebase this member's inputs: x rows, n and the hyperparameter row.
template <typename PX, typename PT>
__device__ __forceinline__ void bmember(const Batch& b, int d, PX& x, int64_t& n, PT& theta) {
  if (!b.gp) return;
  const int64_t p = b.gp[blockIdx.z];
  const int64_t r0 = b.xoff[p];
  x += r0 * d;
  n = b.xoff[p + 1] - r0;
  theta += p * b.theta_stride;
}

// ---------------------------------------------------------------------------
// Stationary kernel formulas (unit variance), from rho^2 of the
// lengthscale-scaled inputs.  kval_of() is k(rho); kval_fac_of() also F(rho) with
// dK/dl_d = var * F(rho) * u_d / l_d, u_d = (x_d - z_d)^2 / l_d^2.
//   RBF        gpjax/kernels/stationary/rbf.py:43          k = exp(-rho^2/2)
//   Matern-1/2 gpjax/kernels/stationary/matern12.py:47     k = exp(-rho)
//   Matern-3/2 gpjax/kernels/stationary/matern32.py:48-53  k = (1+s3 rho) exp(-s3 rho)
//   Matern-5/2 gpjax/kernels/stationary/matern52.py:47-52  k = (1+s5 rho+5/3 rho^2) exp(-s5 rho)
// Matern distances are sqrt(max(rho^2, 1e-36)) (stationary/utils.py:67).
// ---------------------------------------------------------------------------
// The kernel kind is a template argument here: a switch per element puts every
// exponential into a branch of its own, one dependent chain after the other with its
// coefficients moved in again each time.  with_kind() takes the switch once around a
// loop of elements, whose chains then overlap.
template <int KIND>
__device__ __forceinline__ double kval_of(double d2) {
  if constexpr (KIND == GPK_KERNEL_RBF) return exp(-0.5 * d2);
  const double t = sqrt(fmax(d2, 1e-36));
  if constexpr (KIND == GPK_KERNEL_MATERN12) return exp(-t);
  if constexpr (KIND == GPK_KERNEL_MATERN32) {
    const double s3 = 1.7320508075688772;
    return (1.0 + s3 * t) * exp(-s3 * t);
  }
  const double s5 = 2.23606797749979;
  return (1.0 + s5 * t + (5.0 / 3.0) * t * t) * exp(-s5 * t);
}

// kval_of in float32 arithmetic (rho^2 formed in float64 by the caller), for
// entries that are stored in float32 anyway: a few float32 ulps of relative
// error instead of the half ulp of rounding a float64 value.
template <int KIND>
__device__ __forceinline__ float kvalf_of(float d2) {
  if constexpr (KIND == GPK_KERNEL_RBF) return expf(-0.5f * d2);
  const float t = sqrtf(fmaxf(d2, 1e-36f));
  if constexpr (KIND == GPK_KERNEL_MATERN12) return expf(-t);
  if constexpr (KIND == GPK_KERNEL_MATERN32) {
    const float s3 = 1.7320508f;
    return (1.0f + s3 * t) * expf(-s3 * t);
  }
  const float s5 = 2.2360680f;
  return (1.0f + s5 * t + (5.0f / 3.0f) * t * t) * expf(-s5 * t);
}

// Both k(rho) and F(rho) with one exponential.
template <int KIND>
__device__ __forceinline__ void kval_fac_of(double d2, double& k, double& f) {
  if constexpr (KIND == GPK_KERNEL_RBF) {
    k = exp(-0.5 * d2);
    f = k;
    return;
  }
  const double t = sqrt(fmax(d2, 1e-36));
  if constexpr (KIND == GPK_KERNEL_MATERN12) {
    const double e = exp(-t);
    k = e;
    f = d2 > 1e-36 ? e / t : 0.0;
  } else if constexpr (KIND == GPK_KERNEL_MATERN32) {
    const double s3 = 1.7320508075688772;
    const double e = exp(-s3 * t);
    k = (1.0 + s3 * t) * e;
    f = 3.0 * e;
  } else {
    const double s5 = 2.23606797749979;
    const double e = exp(-s5 * t);
    k = (1.0 + s5 * t + (5.0 / 3.0) * t * t) * e;
    f = (5.0 / 3.0) * (1.0 + s5 * t) * e;
  }
}

// kval_fac_of in float32 arithmetic (the mixed collapsed ELBO's gradient pass).
template <int KIND>
__device__ __forceinline__ void kval_facf_of(float d2, float& k, float& f) {
  if constexpr (KIND == GPK_KERNEL_RBF) {
    k = expf(-0.5f * d2);
    f = k;
    return;
  }
  const float t = sqrtf(fmaxf(d2, 1e-36f));
  if constexpr (KIND == GPK_KERNEL_MATERN12) {
    const float e = expf(-t);
    k = e;
    f = d2 > 1e-36f ? e / t : 0.0f;
  } else if constexpr (KIND == GPK_KERNEL_MATERN32) {
    const float s3 = 1.7320508f;
    const float e = expf(-s3 * t);
    k = (1.0f + s3 * t) * e;
    f = 3.0f * e;
  } else {
    const float s5 = 2.2360680f;
    const float e = expf(-s5 * t);
    k = (1.0f + s5 * t + (5.0f / 3.0f) * t * t) * e;
    f = (5.0f / 3.0f) * (1.0f + s5 * t) * e;
  }
}

// f(std::integral_constant<int, kind>()).
template <typename F>
__device__ __forceinline__ void with_kind(int kind, F&& f) {
  if (kind == GPK_KERNEL_RBF) f(std::integral_constant<int, GPK_KERNEL_RBF>());
  else if (kind == GPK_KERNEL_MATERN12) f(std::integral_constant<int, GPK_KERNEL_MATERN12>());
  else if (kind == GPK_KERNEL_MATERN32) f(std::integral_constant<int, GPK_KERNEL_MATERN32>());
  else f(std::integral_constant<int, GPK_KERNEL_MATERN52>());
}

// By runtime kind, for loops that one element at a time is enough for (the collapsed
// ELBO's data pass, with 2 d + 1 sums per thread: a kernel per kind was no faster).
__device__ __forceinline__ void kval_fac(int kind, double d2, double& k, double& f) {
  with_kind(kind, [&](auto K) { kval_fac_of<K()>(d2, k, f); });
}
__device__ __forceinline__ void kval_facf(int kind, float d2, float& k, float& f) {
  with_kind(kind, [&](auto K) { kval_facf_of<K()>(d2, k, f); });
}

// ---------------------------------------------------------------------------
// Host-side launchers (each defined next to its kernels).
// ---------------------------------------------------------------------------

// Gram / cross-covariance tiles.  Rows i < rows_total, cols j < cols_total are
// written; entries with i >= n or j >= m are the identity pad (1 on i == j,
// else 0).  diag_mode & KM_DIAG_MASK: 0 none, 1 add jitter, 2 add jitter +
// obs_sd^2 (i == j < n); diag_mode | KM_ZERO_PAD makes the pad all zeros.
constexpr int KM_DIAG_MASK = 3;
constexpr int KM_ZERO_PAD = 4;
// lower_only: only 128-tiles on or below the diagonal (rows_total == cols_total).
// dblk (optional, lower_only mode): every diagonal NB x NB block is also
// written in float64 to dblk[b][NB][NB].
// spk (optional, lower_only mode): every lower NB-tile (I >= J) is also written
// in float64, packed: tile I(I+1)/2 + J at spk + (I(I+1)/2 + J) * NB * NB.
template <typename TS>
int launch_kernel_matrix(int kind, const double* x, int64_t n, const double* z, int64_t m,
                         int d, const double* theta, int nls, double jitter, int diag_mode,
                         TS* out, int64_t ldo, int64_t rows_total, int64_t cols_total,
                         bool lower_only, hipStream_t s, double* dblk = nullptr,
                         const Batch& bt = Batch(), double* spk = nullptr);

// Cross-covariance K[i][j] = var k(x_i, z_j) (i < n, j < m; zero elsewhere up
// to rows_total x cols_total) for long point streams (the collapsed ELBO's Kzx
// chunks: x = inducing inputs, z = the chunk's points; the predictive's test
// points).  Entries equal launch_kernel_matrix's (d > 32 runs it); f32k
// (float32 output only, d <= 32) evaluates the kernel function in float32
// arithmetic from the float64 squared distances (kvalf).
template <typename TS>
int launch_cross(int kind, const double* x, int64_t n, const double* z, int64_t m, int d,
                 const double* theta, int nls, bool f32k, TS* out, int64_t ldo,
                 int64_t rows_total, int64_t cols_total, hipStream_t s);

// Leaf: factor the NB x NB diagonal block at (o, o) of A in float64 in LDS,
// write L (lower, zero upper) to A, L^-1 to X (lower, zero upper) and to
// leafinv (float64), 2*sum(log diag) to *logdet, first bad pivot to *info.
// dsrc (optional): read the block from this float64 NB x NB array instead of A.
template <typename TS>
int launch_leaf(TS* A, TS* X, int64_t ld, int64_t o, double* leafinv, double* logdet, int* info,
                const double* dsrc, hipStream_t s, const Batch& bt = Batch());

// The float64 leaf with one FMA per entry and column, in order (Factor::seq).
int launch_leaf_sweep(double* A, double* X, int64_t ld, int64_t o, double* leafinv,
                      double* logdet, int* info, hipStream_t s);
// The float64 leaf at o >= NB together with the update C -= P P^T of the `rest` rows
// and columns beyond it (lower NB-tiles) by the NB columns P before o and, with
// `inverse`, of the unfinished rows of the inverse by the finished row before o.
int launch_leaf_update(double* A, double* X, int64_t ld, int64_t o, int64_t rest, bool inverse,
                       double* leafinv, double* logdet, int* info, hipStream_t s);
// After a leaf with inverse `inv`: B (`rows` x NB) <- B inv^T and N (NB x `cols`) <-
// inv N, both in place.
int launch_step_solve(double* B, double* N, int64_t ld, int64_t rows, int64_t cols,
                      const double* inv, hipStream_t s);

// k-range modes of the tile GEMM.
enum KRange { KR_FULL = 0, KR_GE_N = 1, KR_LE_M = 2, KR_GE_M = 3 };
// Product arithmetic of the tile GEMM.  AR_FP16X3: float32 operands scaled by a
// power of two (so that every entry sits well inside the fp16 range), split
// into fp16 hi + lo planes, products hi*hi + hi*lo + lo*hi.
// AR_F64_SEQ: float64 on 128-tiles alone, four consecutive k per matrix-core product
// (Factor::seq).
enum Arith { AR_F64 = 0, AR_F64_SEQ = 1, AR_BF16X3 = 3, AR_FP16X3 = 4, AR_BF16X6 = 6 };

// Tile rule of the FP64 products (double operands, no diagonal side buffer), by the
// number of 128-tiles of the launch (every tile width sums k in the same order, so
// the choice changes no bit): up to SMALL_TILES run on 64 x 64 tiles, up to
// TINY_TILES on 32 x 32.  The line lies where 128-tiles fill the chip's two
// workgroups per CU; MLL + gradient at n = 5,000: 6.57 ms with 160, 6.45 with 384,
// 6.19 with 512, 6.27 with 1,024 (10.9 without), n = 16,384: 86.5 / 86.8 / 86.7 /
// 87.3 (100.9).  The 32-wide ones (none / up to 8 / 24 / 64 tiles): n = 500 296 / 279 /
// 278 / 279 us, n = 2,000 933 / 889 / 846 / 846, n = 4,000 3,332 / 3,290 / 3,235 / 3,221,
// predictive at n = 2,000 with 500 points 1,247 / 1,189 / 1,107 / 1,120.  In a batch the other
// pieces' launches fill the chip, so there only launches of few tiles take the small
// ones (512 GPs of up to 600 rows: 3.17 ms with 512, 2.96 with 96).
constexpr int64_t SMALL_TILES = 512, SMALL_TILES_BATCH = 96;
constexpr int64_t TINY_TILES = 24;

// C[M x N] = alpha * sum_k A(m, k) B(n, k) (+ C if beta_one), M, N, K multiples
// of NB.  A(m, k) is A[m*lda + k] (a_km = false) or A[k*lda + m] (a_km = true);
// B(n, k) is B[n*ldb + k] (b_kn = false) or B[k*ldb + n] (b_kn = true).
// lower_tiles: only tiles with mt >= nt.  krange restricts k per tile.
// fscale (AR_FP16X3 only): device pointer to the power-of-two scales of A and B.
template <typename TA, typename TB, typename TC>
int launch_gemm(int arith, bool a_km, bool b_kn, const TA* A, int64_t lda, const TB* B,
                int64_t ldb, TC* C, int64_t ldc, int64_t M, int64_t N, int64_t K, double alpha,
                bool beta_one, bool lower_tiles, int krange, hipStream_t s,
                double* cdiag = nullptr, const Batch& bt = Batch(),
                const float* fscale = nullptr);

// One level of the recursive triangular inverse as one launch: the 2^depth nodes of
// that depth of the recursion over rows o .. o + n (splits as tri_split), a node
// per z index.  Every node wider than `unit` computes T = L21 X11 (product 1) or
// X21 = -X22 T (product 2); its T sits at T + (node's o - o) * tstride.
struct TriLevel {
  unsigned nodes = 0;  // nodes of this launch; 0: not a level of the inverse
  unsigned first = 0;  // the first of them (a level may take several launches)
  int depth = 0;
  int product = 0;
  int o = 0, n = 0, unit = NB;  // 32 bits: a kernel argument of every tile GEMM
  int ld = 0, tstride = 0;
};
__host__ __device__ inline int tri_split(int n, int unit) {
  const int hu = n / unit / 2;
  return (hu > 0 ? hu : 1) * unit;
}
// Node `node` of the level: rows o .. o + n, split at h; false if it is a leaf (or
// below one).
__host__ __device__ inline bool tri_node(const TriLevel& t, unsigned node, int& o, int& n,
                                         int& h) {
  o = t.o;
  n = t.n;
  for (int d = t.depth - 1; d >= 0; --d) {
    if (n <= t.unit) return false;
    h = tri_split(n, t.unit);
    if ((node >> d) & 1) {
      o += h;
      n -= h;
    } else {
      n = h;
    }
  }
  if (n <= t.unit) return false;
  h = tri_split(n, t.unit);
  return true;
}
// max_m x max_n: the largest node's T.  A, B, C as the product names them.
template <typename TS>
int launch_tri_level(int arith, const TriLevel& lev, int64_t max_m, int64_t max_n, const TS* A,
                     int64_t lda, const TS* B, int64_t ldb, TS* C, int64_t ldc, hipStream_t s,
                     const Batch& bt, const float* fscale);

// Y = B L11^-T in place: m rows x NB columns (float64), inv = L11^-1 (NB x NB).
int launch_trsm_strip(double* B, int64_t ld, int64_t m, const double* inv, hipStream_t s,
                      const Batch& bt = Batch());

// True when the FP64 pass below runs on 64-tiles (which read X down its columns, never
// its transpose), and the number of partial records a call writes (each nls + 2
// doubles): one per tile.  Up to 600 128-tiles, about where those fill the chip's two
// workgroups per CU: MLL + gradient at n = 2,000 1.60 -> 1.47 ms and n = 4,000 even, but
// n = 6,000 (1,128 tiles) 8.5 -> 8.9 ms with the small tiles.  By np and d alone: the
// width is part of the order of the sums, and a batch member's must not depend on how
// many members share a launch.  Batches, 128-wide / 64-wide (MLL + gradient): 8 GPs of
// 1,024 rows 1.15 / 1.00 ms, 400 of 512 3.36 / 3.19 ms, 50 of 2,048 11.94 / 11.86 ms,
// 400 of 1,024 15.5 / 15.8 ms (d = 8: 18.3 / 16.9), 4,096 of 32 to 1,024 57.5 / 58.7 ms.
constexpr int64_t ADJ_SMALL_TILES = 600;
inline bool adjoint_small(int64_t np, int d) {
  const int64_t T = np / NB;
  return d <= 32 && T * (T + 1) / 2 <= ADJ_SMALL_TILES;
}
inline int64_t adjoint_tiles(bool f64, int64_t np, int d) {
  const int64_t T = f64 && adjoint_small(np, d) ? np / 64 : np / NB;
  return T * (T + 1) / 2;
}

// Fused LAUUM + adjoint: for every lower NB-tile of Sinv = X^T X (X = L^-1,
// lower, Np x Np), reduce 1/2 tr(W dSigma/dtheta) contributions with
// W = alpha alpha^T - Sinv against kernel tiles recomputed from x.
// partial: [adjoint_tiles][nls + 2] float64.
// beta (optional): W = alpha beta^T + beta alpha^T - X^T X instead; dense: X is
// a dense Np x Np matrix (every k) rather than lower triangular (k >= row).
// fscale (AR_FP16X3 only): device pointer to the power-of-two scale of X.
template <typename TS>
int launch_adjoint(int kind, int arith, const TS* X, int64_t ld, int64_t np, const double* x,
                   int64_t n, int d, const double* theta, int nls, const double* alpha,
                   double* partial, hipStream_t s, const Batch& bt = Batch(),
                   const double* beta = nullptr, bool dense = false,
                   const float* fscale = nullptr, bool xt = false);
// xt: the operand passed is U = X^T (upper, row-major) from launch_lower_to_upper
// (refused where adjoint_small).

// U = X^T for lower-triangular X (np x np, np a multiple of NB): upper U with
// zeros below the diagonal inside its diagonal NB-tiles.
template <typename TS>
int launch_lower_to_upper(const TS* X, TS* U, int64_t ld, int64_t np, hipStream_t s,
                          const Batch& bt = Batch());

// Row chunk of launch_trmv's transposed form over its 64-column blocks: the widest of
// 1,024 .. 128 rows whose grid (column blocks x chunks) has at least 1,024 workgroups,
// 128 if none has; and the chunks it makes of np rows.  By np alone (as the two rules
// below and colreduce_rows): the members of a batch add to the grid, but a member's sums
// must not depend on how many others are computed with it.
inline int64_t trmv_t_rows(int64_t np) {
  const int64_t blocks = (np + 63) / 64;
  int64_t rc = 1024;
  while (rc > 128 && blocks * ((np + rc - 1) / rc) < 1024) rc /= 2;
  return rc;
}
inline int64_t trmv_max_chunks(int64_t np) {
  const int64_t rc = trmv_t_rows(np);
  return (np + rc - 1) / rc;
}
// Row chunk of launch_colreduce, by the number of rows alone: a column's sum does not
// depend on how many columns come with it (the predictive's passes).
inline int64_t colreduce_rows(int64_t rows) { return rows <= 4096 ? 128 : rows <= 16384 ? 256 : 1024; }
inline int64_t colreduce_chunks(int64_t rows) {
  const int64_t rc = colreduce_rows(rows);
  return (rows + rc - 1) / rc;
}

// y = X r (trans = false) or y = X^T r (trans = true; add: y += X^T r), X lower
// triangular np x np (only k <= i is read); float64 accumulation through `partial`
// (nv x trmv_max_chunks(np) x np doubles).  nv = 1 or 3 right-hand sides, stored
// np apart in r and in y, share each pass over X.  rows: the transposed form's row
// chunk (at least trmv_t_rows, at most 1,024), 0 for the rule above.
template <typename TS>
int launch_trmv(const TS* X, int64_t ld, int64_t np, const double* r, double* y, bool trans,
                double* partial, hipStream_t s, const Batch& bt = Batch(), int nv = 1,
                bool add = false, int64_t rows = 0);

// Columns per chunk of the recomputed Sigma product below: the widest power of two
// (64 .. 1,024) whose grid, ceil(np / 256) row blocks x chunks, has at least 1,024
// workgroups (four waves per SIMD), 64 if none has.
inline int64_t sigma_mv_chunk(int64_t np) {
  const int64_t rows = (np + 255) / 256;
  int64_t cw = 1024;
  while (cw > 64 && rows * ((np + cw - 1) / cw) < 1024) cw /= 2;
  return cw;
}
inline int64_t sigma_mv_max_chunks(int64_t np) {
  const int64_t cw = sigma_mv_chunk(np);
  return (np + cw - 1) / cw;
}

// v = Sigma a, Sigma recomputed from x in float64 (identity pad for i >= n);
// nv = 1 or 3 vectors np apart share each kernel evaluation.  partial holds
// nv x sigma_mv_max_chunks(np) x np doubles.  res (optional) = r - v (first vector).
int launch_sigma_matvec(int kind, const double* x, int64_t n, int64_t np, int d,
                        const double* theta, int nls, double jitter, const double* a, double* v,
                        double* partial, hipStream_t s, const Batch& bt = Batch(), int nv = 1,
                        const double* r = nullptr, double* res = nullptr);

// Library-owned streams (default priority, non-blocking) and events for the
// calling thread on the current device, created on first use and kept for the
// process.  The look-ahead Cholesky takes stream 0 and events 0..2 (never
// inside a batched call); the batched driver takes the streams and events
// 3..3+AUX_STREAMS; the collapsed ELBO takes stream 0 and events 6 and 7
// (joined before its M x M factor, which alone may run the look-ahead Cholesky).
constexpr int AUX_STREAMS = 3;
constexpr int AUX_EVENTS = 8;
int aux_streams(hipStream_t* streams, hipEvent_t* events);
int lookahead_resources(hipStream_t* s2, hipEvent_t* ev3);

// Joins a forked library stream back into the caller's: at scope exit (an
// early error return included) `s` waits for everything issued to `s2` so far,
// so no work of a call is left unjoined.
struct StreamJoin {
  hipStream_t s, s2;
  hipEvent_t e;
  ~StreamJoin() {
    if (hipEventRecord(e, s2) == hipSuccess) (void)hipStreamWaitEvent(s, e, 0);
  }
};

// v = S a for a symmetric S held as its packed lower NB-tiles in float64 (the
// spk layout of launch_kernel_matrix), np x np; nv = 1 or 3 vectors np apart
// share each read of S.  partial holds 2 * nv * T(T+1)/2 * NB doubles, T = np/NB.
// res (optional) = r - v (first vector).
int launch_packed_symv(const double* S, int64_t np, const double* a, double* v,
                       double* partial, hipStream_t s, const Batch& bt = Batch(), int nv = 1,
                       const double* r = nullptr, double* res = nullptr);

// y_j = sum_i M[i][j] v_i (v non-null) or sum_i M[i][j]^2 (v null), dense
// rows x cols (float64 or float32 entries, float64 sums); partial holds
// colreduce_chunks(rows) x cols doubles.  lower: only rows i >= j enter column j.
template <typename TM>
int launch_colreduce(const TM* M, int64_t ld, int64_t rows, int64_t cols, const double* v,
                     double* y, double* partial, hipStream_t s, bool lower = false);

int launch_mfma_selftest(double* out64, float* outbf, hipStream_t s);

}  // namespace gpk
