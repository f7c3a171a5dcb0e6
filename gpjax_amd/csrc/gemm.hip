// Tile GEMM used by the recursive Cholesky, triangular solve and triangular
// inverse:  C = alpha * A B^T (+ C), with per-tile k-ranges for triangular
// operands and an optional lower-triangular tile set (SYRK).  These replace the
// LAPACK/BLAS work behind jnp.linalg.cholesky / solve / slogdet
// (gpjax/linalg/operations.py:54-55,109-111,163-165).
#include <type_traits>

#include "factor.h"
#include "gemm_core.h"

namespace gpk {
namespace {

struct GemmParams {
  const void* A;
  int64_t lda;
  const void* B;
  int64_t ldb;
  void* C;
  int64_t ldc;
  int64_t K;
  double alpha;
  int beta_one;
  int lower_tiles;
  int krange;
  double* cdiag;  // lower_tiles: diagonal tiles update this float64 [tile][NB][NB] instead of C
  Batch bt;       // batch of same-shape problems, member blockIdx.z (operands in workspaces)
  const float* fscale;  // AR_FP16X3: power-of-two scales of A and B (device)
  int64_t tiles_m;      // M / TILE (the lower-tile decode needs the side)
  int64_t tiles_n;      // N / TILE
  TriLevel tri;         // tri.nodes > 0: one level of the triangular inverse
};

// Member and (for a level of the triangular inverse) node of this workgroup, and
// the operands rebased to them; false when the node has no work here.
template <typename TA, typename TB, typename TC>
__device__ __forceinline__ bool gemm_rebase(GemmParams& p) {
  unsigned member = blockIdx.z;
  if (p.tri.nodes > 0) {
    const unsigned node = p.tri.first + blockIdx.z % p.tri.nodes;
    member = blockIdx.z / p.tri.nodes;
    int o32, n, h;
    if (!tri_node(p.tri, node, o32, n, h)) return false;
    const int64_t o = o32;
    // p.A = L (product 1) or X (product 2), p.B = X or T, p.C = T or X
    const int64_t ld = p.tri.ld, toff = (o - p.tri.o) * (int64_t)p.tri.tstride;
    if (p.tri.product == 1) {  // T = L21 X11
      p.A = static_cast<const TA*>(p.A) + (o + h) * ld + o;
      p.B = static_cast<const TB*>(p.B) + o * ld + o;
      p.C = static_cast<TC*>(p.C) + toff;
      p.ldc = h;
      p.K = h;
    } else {  // X21 = -X22 T
      p.A = static_cast<const TA*>(p.A) + (o + h) * ld + o + h;
      p.B = static_cast<const TB*>(p.B) + toff;
      p.ldb = h;
      p.C = static_cast<TC*>(p.C) + (o + h) * ld + o;
      p.K = n - h;
    }
    p.tiles_m = (n - h) / TILE;
    p.tiles_n = h / TILE;
  }
  if (p.bt.ws_stride) {
    const int64_t sh = (int64_t)member * p.bt.ws_stride;
    p.A = static_cast<const char*>(p.A) + sh;
    p.B = static_cast<const char*>(p.B) + sh;
    p.C = static_cast<char*>(p.C) + sh;
    if (p.cdiag) p.cdiag = reinterpret_cast<double*>(reinterpret_cast<char*>(p.cdiag) + sh);
  }
  return true;
}

// 128-tile (mt, nt) of the flat index b, in the banded orders (16 x 16 blocks of
// tiles resident together share their operand panels in L2); false past the end.
__device__ __forceinline__ bool gemm_tile(const GemmParams& p, int64_t b, int64_t& mt,
                                          int64_t& nt) {
  if (p.lower_tiles) {
    lower_tile_banded(b, p.tiles_m, mt, nt);
    return true;
  }
  if (b >= p.tiles_m * p.tiles_n) return false;
  if (p.krange == KR_GE_N) {
    // k >= column tile: the first tile columns carry the most work, so band
    // by columns and dispatch them first.
    grid_tile_banded(b, p.tiles_n, p.tiles_m, nt, mt);
  } else {
    grid_tile_banded(b, p.tiles_m, p.tiles_n, mt, nt);
    // k <= row tile: the last tile rows carry the most work, so dispatch them first.
    if (p.krange == KR_LE_M) mt = p.tiles_m - 1 - mt;
  }
  return true;
}

template <int AR, typename TA, typename TB, typename TC, bool A_KM, bool B_KN, bool SEQ>
__global__ __launch_bounds__(WaveLayout<AR>::NT) void gemm_kernel(GemmParams p) {
  typedef WaveLayout<AR> WL;
  __shared__ __align__(16) char smem[smem_bytes<AR>()];
  if (!gemm_rebase<TA, TB, TC>(p)) return;
  int64_t mt, nt;
  if (!gemm_tile(p, blockIdx.x, mt, nt)) return;
  int64_t kb, ke;
  k_range(p.krange, mt, nt, p.K, kb, ke);
  const int64_t m0 = mt * TILE, n0 = nt * TILE;
  typename AccT<AR>::vec acc[4][WL::NJ];
  if constexpr (AR == AR_F64) {
    mainloop_f64<TA, TB, A_KM, B_KN, SEQ>(static_cast<const TA*>(p.A), p.lda,
                                     static_cast<const TB*>(p.B), p.ldb, m0, n0, kb, ke, acc,
                                     smem);
  } else {
    float sa = 1.f, sb = 1.f;
    if constexpr (AR == AR_FP16X3) {
      sa = p.fscale[0];
      sb = p.fscale[1];
    }
    mainloop_bf16<AR, A_KM, B_KN>(static_cast<const float*>(p.A), p.lda,
                                  static_cast<const float*>(p.B), p.ldb, m0, n0, kb, ke, acc,
                                  smem, sa, sb);
  }
  TC* C = static_cast<TC*>(p.C);
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int wm = w / WL::WN, wn = w % WL::WN;
  if (p.cdiag && p.lower_tiles && mt == nt) {
    double* cd = p.cdiag + mt * TILE * TILE;
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
      for (int j = 0; j < WL::NJ; ++j)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int row = wm * 64 + i * 16 + acc_row<AR>(lane, r);
          const int colx = wn * WL::WC + j * 16 + (lane & 15);
          double* c = cd + row * TILE + colx;
          double v = p.alpha * (double)acc[i][j][r];
          if (p.beta_one) v += *c;
          *c = v;
        }
    return;
  }
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < WL::NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int64_t row = m0 + wm * 64 + i * 16 + acc_row<AR>(lane, r);
        const int64_t colx = n0 + wn * WL::WC + j * 16 + (lane & 15);
        TC* c = C + row * p.ldc + colx;
        double v = p.alpha * (double)acc[i][j][r];
        if (p.beta_one) v += (double)*c;
        *c = (TC)v;
      }
}

// ---- small FP64 products ----
// The same products on (32 MI) x (32 NJ) tiles for grids that leave most of the
// chip idle at 128 x 128 (one such tile takes 14 us per 128 of k on its one CU).
// Four independent waves, 16 MI x 16 NJ each, read their matrix-core operands
// straight from global memory: lane (lr, lc) = (lane / 16, lane % 16) takes row lc
// and k = 4 lr .. 4 lr + 3 of a 16-deep slab, and the four products of a slab use
// its q-th values, so both operands see the same k.  No LDS and no barrier: four
// slabs per operand are in flight in registers (SETS), which covers the latency a
// lone wave per SIMD would otherwise wait out.  The k-ranges of triangular operands
// are cut at 64 instead of 128.  Bound by the matrix cores' own chain: 16 products
// of 64 cycles per slab and wave.  Measured per launch: K = 128, one to sixteen
// 128-tiles 24 -> 6 us; the 1,024 x 1,024 x 1,024 products of the triangular
// inverse 142 -> 51 us.
template <bool A_KM, bool B_KN, int MI, int NJ>
__global__ __launch_bounds__(256, 2) void gemm_small_kernel(GemmParams p) {
  constexpr int BM = 32 * MI, BN = 32 * NJ;
  constexpr int SM = TILE / BM, SN = TILE / BN;
  if (!gemm_rebase<double, double, double>(p)) return;
  int64_t mt, nt;
  if (!gemm_tile(p, blockIdx.x / (SM * SN), mt, nt)) return;
  const int sub = blockIdx.x % (SM * SN);
  const int64_t m0 = mt * TILE + (sub / SN) * BM, n0 = nt * TILE + (sub % SN) * BN;
  int64_t kb = 0, ke = p.K;
  if (p.krange == KR_GE_N) kb = n0 / KG * KG;
  else if (p.krange == KR_LE_M) ke = min(p.K, (m0 + BM + KG - 1) / KG * KG);
  else if (p.krange == KR_GE_M) kb = m0 / KG * KG;

  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane >> 4, lc = lane & 15;
  const int64_t mw = m0 + (w >> 1) * 16 * MI, nw = n0 + (w & 1) * 16 * NJ;
  const double* A = static_cast<const double*>(p.A);
  const double* B = static_cast<const double*>(p.B);
  double* C = static_cast<double*>(p.C);
  f64x4 acc[MI][NJ];
  DirectLoop<A_KM, B_KN, MI, NJ> loop(A, p.lda, B, p.ldb, mw, nw, lane, kb, ke);
  double cv[MI][NJ][4];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cv[i][j][r] =
            p.beta_one ? C[(mw + 16 * i + lr + 4 * r) * p.ldc + nw + 16 * j + lc] : 0.0;
  loop.run(acc);
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        C[(mw + 16 * i + lr + 4 * r) * p.ldc + nw + 16 * j + lc] =
            p.alpha * acc[i][j][r] + cv[i][j][r];
}

// 128-tiles of a launch (the largest node's, for a level of the inverse) and
// its z extent.
inline int64_t tile_count(const GemmParams& p) {
  return p.lower_tiles ? p.tiles_m * (p.tiles_m + 1) / 2 : p.tiles_m * p.tiles_n;
}
inline unsigned z_count(const GemmParams& p) {
  return p.bt.count * (p.tri.nodes > 0 ? p.tri.nodes : 1u);
}

template <int MI, int NJ>
int launch_small(bool a_km, bool b_kn, const GemmParams& p, hipStream_t s) {
  const dim3 grid((unsigned)(tile_count(p) * (TILE / (32 * MI)) * (TILE / (32 * NJ))), 1,
                  z_count(p));
#define GPK_SMALL(AK, BK) \
  hipLaunchKernelGGL((gemm_small_kernel<AK, BK, MI, NJ>), grid, dim3(256), 0, s, p)
  if (!a_km && !b_kn) GPK_SMALL(false, false);
  else if (!a_km && b_kn) GPK_SMALL(false, true);
  else if (a_km && !b_kn) GPK_SMALL(true, false);
  else GPK_SMALL(true, true);
#undef GPK_SMALL
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

// Y = B L11^-T in place for `m` rows (a multiple of NB) of NB columns, from the
// leaf's float64 inverse (row-major NB x NB, lower): the column block of a
// triangular solve.  One workgroup per 16 MI rows: its four waves read all of the
// rows' operands into registers, pass a barrier, and then overwrite them; wave w
// computes column blocks w and 7 - w (of 16), k only up to the diagonal, so every
// wave issues nine slabs.  15 blocks of 128 rows: 24 us as 128 x 128 tiles, 7 us.
template <int MI>
__device__ __forceinline__ void trsm_strip(double* B, int64_t ld, const double* __restrict__ inv,
                                           int64_t r0) {
  constexpr int NS = NB / SLAB;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane >> 4, lc = lane & 15;
  double av[NS][MI][4], bv[NS + 1][4];
#pragma unroll
  for (int s = 0; s < NS; ++s)
#pragma unroll
    for (int i = 0; i < MI; ++i)
      frag_load<false>(B, ld, r0 + 16 * i + lc, s * SLAB + 4 * lr, av[s][i]);
  // slabs 0 .. 7 - w of column block 7 - w, then 0 .. w of column block w
#pragma unroll
  for (int t = 0; t <= NS; ++t) {
    const int second = t >= NS - w;
    const int J = second ? w : NS - 1 - w, s = second ? t - (NS - w) : t;
    frag_load<false>(inv, NB, J * 16 + lc, s * SLAB + 4 * lr, bv[t]);
  }
  __syncthreads();
  f64x4 acc[2][MI];
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < MI; ++i) acc[c][i] = f64x4{0.0, 0.0, 0.0, 0.0};
  // w is uniform: one of four straight-line schedules
  auto products = [&](auto wc) {
    constexpr int W = decltype(wc)::value;
#pragma unroll
    for (int t = 0; t <= NS; ++t) {
      constexpr int split = NS - W;
      const int c = t >= split ? 1 : 0, s = t >= split ? t - split : t;
#pragma unroll
      for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int i = 0; i < MI; ++i)
          acc[c][i] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[s][i][q], bv[t][q], acc[c][i], 0, 0,
                                                           0);
    }
  };
  if (w == 0) products(std::integral_constant<int, 0>());
  else if (w == 1) products(std::integral_constant<int, 1>());
  else if (w == 2) products(std::integral_constant<int, 2>());
  else products(std::integral_constant<int, 3>());
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        B[(r0 + 16 * i + lr + 4 * r) * ld + (c ? w : NS - 1 - w) * 16 + lc] = acc[c][i][r];
}

template <int MI>
__global__ __launch_bounds__(256) void trsm_strip_kernel(double* B, int64_t ld,
                                                         const double* __restrict__ inv,
                                                         Batch bt) {
  trsm_strip<MI>(bws(B, bt), ld, bws(inv, bt), (int64_t)blockIdx.x * 16 * MI);
}

// X = L11^-1 N in place for the 16 columns from c0 of NB rows (the same roles with the
// inverse on the left): wave w computes row blocks w and 7 - w.
__device__ __forceinline__ void inverse_strip(double* N, int64_t ld,
                                              const double* __restrict__ inv, int64_t c0) {
  constexpr int NS = NB / SLAB;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int lr = lane >> 4, lc = lane & 15;
  double av[NS + 1][4], bv[NS][4];
#pragma unroll
  for (int s = 0; s < NS; ++s) frag_load<true>(N, ld, c0 + lc, s * SLAB + 4 * lr, bv[s]);
#pragma unroll
  for (int t = 0; t <= NS; ++t) {
    const int second = t >= NS - w;
    const int I = second ? w : NS - 1 - w, s = second ? t - (NS - w) : t;
    frag_load<false>(inv, NB, I * 16 + lc, s * SLAB + 4 * lr, av[t]);
  }
  __syncthreads();
  f64x4 acc[2] = {f64x4{0.0, 0.0, 0.0, 0.0}, f64x4{0.0, 0.0, 0.0, 0.0}};
  auto products = [&](auto wc) {
    constexpr int split = NS - decltype(wc)::value;
#pragma unroll
    for (int t = 0; t <= NS; ++t) {
      const int c = t >= split ? 1 : 0, s = t >= split ? t - split : t;
#pragma unroll
      for (int q = 0; q < 4; ++q)
        acc[c] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[t][q], bv[s][q], acc[c], 0, 0, 0);
    }
  };
  if (w == 0) products(std::integral_constant<int, 0>());
  else if (w == 1) products(std::integral_constant<int, 1>());
  else if (w == 2) products(std::integral_constant<int, 2>());
  else products(std::integral_constant<int, 3>());
#pragma unroll
  for (int c = 0; c < 2; ++c)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      N[((c ? w : NS - 1 - w) * 16 + lr + 4 * r) * ld + c0 + lc] = acc[c][r];
}

// What follows a leaf whose inverse is `inv`: the solve of the column block B below it
// (`rows` rows, the first rows / 16 workgroups) and the inverse's row block N left of
// it (`cols` columns, the others).
__global__ __launch_bounds__(256) void step_solve_kernel(double* B, double* N, int64_t ld,
                                                         const double* __restrict__ inv,
                                                         int64_t rows) {
  const int64_t nb = rows / 16;
  if (blockIdx.x < nb) trsm_strip<1>(B, ld, inv, (int64_t)blockIdx.x * 16);
  else inverse_strip(N, ld, inv, ((int64_t)blockIdx.x - nb) * 16);
}

template <int AR, typename TA, typename TB, typename TC, bool A_KM, bool B_KN, bool SEQ>
int launch_t(const GemmParams& p, hipStream_t s) {
  const dim3 grid((unsigned)tile_count(p), 1, z_count(p));
  hipLaunchKernelGGL((gemm_kernel<AR, TA, TB, TC, A_KM, B_KN, SEQ>), grid,
                     dim3(WaveLayout<AR>::NT), 0, s, p);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

template <int AR, typename TA, typename TB, typename TC, bool SEQ = false>
int dispatch_layout(bool a_km, bool b_kn, const GemmParams& p, hipStream_t s) {
  if (!a_km && !b_kn) return launch_t<AR, TA, TB, TC, false, false, SEQ>(p, s);
  if (!a_km && b_kn) return launch_t<AR, TA, TB, TC, false, true, SEQ>(p, s);
  if (a_km && !b_kn) return launch_t<AR, TA, TB, TC, true, false, SEQ>(p, s);
  return launch_t<AR, TA, TB, TC, true, true, SEQ>(p, s);
}

template <typename TA, typename TB, typename TC>
int launch_arith(int arith, bool a_km, bool b_kn, const GemmParams& p, hipStream_t s) {
  if (tile_count(p) > 0x7fffffff / 16 || z_count(p) > 65535) {
    set_error("gemm: %lld tiles x %u members exceed one launch", (long long)tile_count(p),
              z_count(p));
    return GPK_ERR_BAD_ARG;
  }
  if (arith == AR_F64) {
    if constexpr (std::is_same<TA, double>::value && std::is_same<TB, double>::value &&
                  std::is_same<TC, double>::value) {
      const int64_t tiles = tile_count(p) * z_count(p);
      if (!p.cdiag && tiles <= TINY_TILES) return launch_small<1, 1>(a_km, b_kn, p, s);
      if (!p.cdiag && tiles <= (p.bt.gp ? SMALL_TILES_BATCH : SMALL_TILES))
        return launch_small<2, 2>(a_km, b_kn, p, s);
    }
    return dispatch_layout<AR_F64, TA, TB, TC>(a_km, b_kn, p, s);
  }
  if constexpr (std::is_same<TA, double>::value && std::is_same<TB, double>::value &&
                std::is_same<TC, double>::value) {
    if (arith == AR_F64_SEQ) return dispatch_layout<AR_F64, TA, TB, TC, true>(a_km, b_kn, p, s);
  }
  if constexpr (std::is_same<TA, float>::value && std::is_same<TB, float>::value) {
    if (arith == AR_BF16X3)
      return dispatch_layout<AR_BF16X3, float, float, TC>(a_km, b_kn, p, s);
    if (arith == AR_BF16X6)
      return dispatch_layout<AR_BF16X6, float, float, TC>(a_km, b_kn, p, s);
    if (arith == AR_FP16X3) {
      if (!p.fscale) {
        set_error("gemm: fp16 products need the operand scales");
        return GPK_ERR_BAD_ARG;
      }
      return dispatch_layout<AR_FP16X3, float, float, TC>(a_km, b_kn, p, s);
    }
  }
  set_error("gemm: unsupported arithmetic %d for these operand types", arith);
  return GPK_ERR_BAD_ARG;
}

}  // namespace

template <typename TA, typename TB, typename TC>
int launch_gemm(int arith, bool a_km, bool b_kn, const TA* A, int64_t lda, const TB* B,
                int64_t ldb, TC* C, int64_t ldc, int64_t M, int64_t N, int64_t K, double alpha,
                bool beta_one, bool lower_tiles, int krange, hipStream_t s, double* cdiag,
                const Batch& bt, const float* fscale) {
  if (M <= 0 || N <= 0) return GPK_OK;
  if (M % TILE || N % TILE || K % TILE || K < 0) {
    set_error("gemm: extents %lld x %lld x %lld not multiples of %d", (long long)M,
              (long long)N, (long long)K, TILE);
    return GPK_ERR_BAD_ARG;
  }
  if (lower_tiles && M != N) {
    set_error("gemm: lower tile set needs M == N");
    return GPK_ERR_BAD_ARG;
  }
  GemmParams p{A, lda, B, ldb, C, ldc, K, alpha, beta_one ? 1 : 0, lower_tiles ? 1 : 0, krange,
               cdiag, bt, fscale, M / TILE, N / TILE, TriLevel()};
  return launch_arith<TA, TB, TC>(arith, a_km, b_kn, p, s);
}

template <typename TS>
int launch_tri_level(int arith, const TriLevel& lev, int64_t max_m, int64_t max_n, const TS* A,
                     int64_t lda, const TS* B, int64_t ldb, TS* C, int64_t ldc, hipStream_t s,
                     const Batch& bt, const float* fscale) {
  GemmParams p{A, lda, B, ldb, C, ldc, 0, lev.product == 1 ? 1.0 : -1.0, 0, 0,
               lev.product == 1 ? (int)KR_GE_N : (int)KR_LE_M, nullptr, bt, fscale,
               max_m / TILE, max_n / TILE, lev};
  // as many nodes per launch as the grid's z extent takes with these members
  const unsigned per = bt.count >= 65535 ? 1u : 65535u / bt.count;
  for (unsigned q = 0; q < lev.nodes; q += per) {
    p.tri.first = lev.first + q;
    p.tri.nodes = lev.nodes - q < per ? lev.nodes - q : per;
    GPK_TRY(launch_arith<TS, TS, TS>(arith, false, true, p, s));
  }
  return GPK_OK;
}
template int launch_tri_level<double>(int, const TriLevel&, int64_t, int64_t, const double*,
                                      int64_t, const double*, int64_t, double*, int64_t,
                                      hipStream_t, const Batch&, const float*);
template int launch_tri_level<float>(int, const TriLevel&, int64_t, int64_t, const float*,
                                     int64_t, const float*, int64_t, float*, int64_t, hipStream_t,
                                     const Batch&, const float*);

int launch_step_solve(double* B, double* N, int64_t ld, int64_t rows, int64_t cols,
                      const double* inv, hipStream_t s) {
  if (rows + cols <= 0) return GPK_OK;
  if (rows % NB || cols % NB) {
    set_error("step solve: %lld rows, %lld columns not multiples of %d", (long long)rows,
              (long long)cols, NB);
    return GPK_ERR_BAD_ARG;
  }
  hipLaunchKernelGGL(step_solve_kernel, dim3((unsigned)((rows + cols) / 16)), dim3(256), 0, s, B,
                     N, ld, inv, rows);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

int launch_trsm_strip(double* B, int64_t ld, int64_t m, const double* inv, hipStream_t s,
                      const Batch& bt) {
  if (m <= 0) return GPK_OK;
  if (m % NB || m / 16 > 0x7fffffff) {
    set_error("trsm: %lld rows not a multiple of %d", (long long)m, NB);
    return GPK_ERR_BAD_ARG;
  }
  // 16 rows per workgroup until that fills the chip, then 32 (half the reads of
  // the inverse)
  if (m / 16 * bt.count <= 512)
    hipLaunchKernelGGL(trsm_strip_kernel<1>, dim3((unsigned)(m / 16), 1, bt.count), dim3(256), 0,
                       s, B, ld, inv, bt);
  else
    hipLaunchKernelGGL(trsm_strip_kernel<2>, dim3((unsigned)(m / 32), 1, bt.count), dim3(256), 0,
                       s, B, ld, inv, bt);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

#define GPK_GEMM_INST(TA, TB, TC)                                                            \
  template int launch_gemm<TA, TB, TC>(int, bool, bool, const TA*, int64_t, const TB*,       \
                                       int64_t, TC*, int64_t, int64_t, int64_t, int64_t, double, \
                                       bool, bool, int, hipStream_t, double*, const Batch&, \
                                       const float*);
GPK_GEMM_INST(double, double, double)
GPK_GEMM_INST(float, float, float)
GPK_GEMM_INST(float, double, float)
GPK_GEMM_INST(float, double, double)
GPK_GEMM_INST(float, float, double)
#undef GPK_GEMM_INST

}  // namespace gpk
