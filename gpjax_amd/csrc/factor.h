// Recursive Cholesky / triangular-solve / triangular-inverse driver on the tile
// GEMM, shared by the exact-GP and collapsed-ELBO paths.
//
//   potrf(A):   potrf(A11); L21 = A21 L11^-T (trsm); A22 -= L21 L21^T; potrf(A22)
//   trsm(B, L): Y L^T = B by recursion on the columns, leaves multiplying by the
//               float64 inverse of an NB x NB diagonal block
//   trtri(L):   X = L^-1 with X21 = -X22 (L21 X11), both halves recursively
// A single float64 problem up to STEPS_MAX rows instead goes leaf by leaf, factor and
// inverse in one sweep (Factor::potrf_steps); larger single problems go by panels.
// These replace jnp.linalg.cholesky, jsp.linalg.solve_triangular and the
// LU-based slogdet/solve behind gpjax/linalg/operations.py:54-55,105-111,163-165.
// Splits fall on multiples of NB; leaves (NB x NB) are factored and inverted
// in float64 in LDS (leaf.hip).
#pragma once

#include "gpk_internal.h"

namespace gpk {

#define GPK_TRY(...)               \
  do {                             \
    int rc_ = (__VA_ARGS__);       \
    if (rc_ != GPK_OK) return rc_; \
  } while (0)

inline int64_t split_point(int64_t n) { return (n / NB / 2) * NB; }

// 128-row blocks x members up to which a triangular solve's leaf runs in strips
// (wide batches take the 128 x 128 tiles: 4,096 small GPs 62.3 -> 61.1 ms).
constexpr int64_t TRSM_STRIP_TILES = 512;
static_assert(TRSM_STRIP_TILES >= SMALL_TILES, "an in-place product on small tiles would race");

// Largest single float64 problem factored leaf by leaf on one stream
// (Factor::potrf_steps).  Beyond it the trailing updates, a rank-128 step each, take
// longer than the leaf they run beside.  MLL + gradient (two streams with the
// look-ahead and the inverse after it / leaf by leaf with the inverse in the sweep, ms):
// n = 2,000 1.41 / 0.85, n = 3,000 2.42 / 1.75, n = 4,000 3.81 / 3.23, n = 4,500 5.14 /
// 4.55, n = 5,000 6.12 / 5.91, n = 6,000 8.56 / 8.89, n = 8,000 15.6 / 19.6.
constexpr int64_t STEPS_MAX = 4096;

// Panel width of the look-ahead Cholesky (Factor::potrf_lookahead) for a single
// np x np problem, np >= 2,048 (float64: > STEPS_MAX): np/32 with float32 storage, np/64
// in float64, rounded down to a multiple of NB, at least NB.  Wider panels put more of the
// update into large rank-B GEMMs; narrower ones shorten the second stream's
// chain per panel, which the first and last panels wait for.  Measured (ms per
// MLL + gradient; * = the rule's choice):
//   float32 storage   np =  2,048: no look-ahead 1.87, B = 128 1.64*, 256 1.86
//                     np =  4,096: no look-ahead 4.13, 128 3.24*, 256 3.75
//                     np =  8,192: no look-ahead 11.6, 128 9.81, 256 9.35*, 512 9.99
//                     np = 16,384: 128 53.4, 256 42.2, 512 39.0*, 1,024 39.7
//                     np = 32,768: 512 230.8, 1,024 217.7*, 2,048 218.1
//                     np = 65,536: 1,024 1,576, 2,048 1,525*, 4,096 1,521
//   float64           np =  8,192: no look-ahead 17.8, 128 16.1*, 256 15.5, 512 16.3
//                     np = 16,384: 128 95.6, 256 87.3*, 512 88.0, 1,024 88.6
//                     np = 32,768: 512 596.9*, 1,024 592.3, 2,048 594.9
//                     np = 65,536: 1,024 4,592*, 2,048 4,589, 4,096 4,602
// (65,536: with the column-sweep leaf.  In float64 np/32 would now be 4 % better at 8,192
// and no worse above.)
// GPK_LOOKAHEAD_B set at build time fixes the width (0 turns the look-ahead off).
#ifndef GPK_LOOKAHEAD_B
#define GPK_LOOKAHEAD_B -1
#endif
inline int64_t lookahead_width(int64_t np, bool f32) {
  if (GPK_LOOKAHEAD_B >= 0) return np >= 4 * GPK_LOOKAHEAD_B ? GPK_LOOKAHEAD_B : 0;
  if (np < 2048) return 0;
  const int64_t b = (np / (f32 ? 32 : 64)) / NB * NB;
  return b < NB ? NB : b;
}

// Depth of the triangular inverse's recursion over n rows with leaves of `unit`.
inline int tri_depth(int n, int unit) {
  int d = 0;
  while (n > unit) {
    n -= tri_split(n, unit);  // the larger half
    ++d;
  }
  return d;
}
// Largest T (rows, columns) of a level's nodes.
inline void tri_extents(const TriLevel& lev, int& mm, int& mn) {
  mm = mn = 0;
  for (unsigned q = 0; q < lev.nodes; ++q) {
    int o, n, h;
    if (!tri_node(lev, q, o, n, h)) continue;
    if (n - h > mm) mm = n - h;
    if (h > mn) mn = h;
  }
}

template <typename T>
inline T* at(void* ws, size_t off) {
  return reinterpret_cast<T*>(static_cast<char*>(ws) + off);
}

template <typename TS>
struct Factor {
  TS* L;             // matrix in, factor out (lower NB-tiles), leading dimension ld
  TS* X;             // L^-1 out (lower)
  int64_t ld;
  TS* T;             // scratch of factor_scratch_elems(n) elements
  double* leafinv;   // n/NB blocks of NB x NB float64 leaf inverses
  double* leafld;    // n/NB leaf log-determinants
  int* leafinfo;     // n/NB leaf pivot status
  int ar_potrf, ar_trtri;
  hipStream_t s;
  // Optional float64 copy of the diagonal NB-blocks ([n/NB][NB][NB]): when set
  // (float32 storage), SYRK updates those blocks in float64 and the leaves
  // factor them from there, so no pivot block is ever rounded to float32.
  double* dblk = nullptr;
  // Optional batch: all pointers above are member 0's; member z's are
  // bt.ws_stride bytes further per z (same padded size for every member).
  Batch bt = Batch();
  // fp16 operand scales (device, AR_FP16X3 only): [sL, sL, sX, sT] with sL for
  // entries of L and the trailing matrix, sX for X = L^-1, sT for L21 X11; the
  // GEMMs read the (A, B) pair at fscale + 0 (POTRF), + 1 and + 2 (TRTRI).
  const float* fscale = nullptr;
  // Diagonal blocks of this width (at multiples of it) already hold their
  // inverse in X when trtri runs (potrf_lookahead inverts each panel's
  // diagonal block on its second stream); NB = only the leaves.
  int64_t tri_unit = NB;

  double* dblk_at(int64_t o) const { return dblk ? dblk + (o / NB) * NB * NB : nullptr; }
  // Float64 with one fixed grouping of its sums (ar_potrf = ar_trtri = AR_F64_SEQ, no
  // batch): the column-sweep leaf, 128-tiles whose products take four consecutive k, the
  // recursion or the look-ahead.  For the mixed collapsed bound, which rounds G_P, made
  // of these inverses, to float32: another grouping moves some of its entries to the
  // other float32 neighbour, and the gradient in Z, a difference of large terms, by
  // 1e-13 to 1e-7 of its norm.  That keeps results as they were, and no more: the two
  // groupings are equally far from the float64 bound (N = 1e6, M = 2,048: 9.191e-6 of
  // the gradient in Z both, 7.0e-9 apart), and this one takes 79.4 ms there against 75.7
  // on the faster routes.
  bool seq() const { return ar_potrf == AR_F64_SEQ; }
  int factor_seq(int64_t n, bool streams) {
    GPK_TRY(factor_only(n, streams));
    return trtri(0, n);
  }
  int leaf(int64_t o) {
    if constexpr (std::is_same<TS, double>::value) {
      if (seq())
        return launch_leaf_sweep(L, X, ld, o, leafinv + (o / NB) * NB * NB, leafld + o / NB,
                                 leafinfo + o / NB, s);
    }
    return launch_leaf<TS>(L, X, ld, o, leafinv + (o / NB) * NB * NB, leafld + o / NB,
                           leafinfo + o / NB, dblk_at(o), s, bt);
  }
  // Solve Y L^T = B in place, B = L[row0 : row0+m, o : o+n], triangle L[o:o+n, o:o+n].
  int trsm(int64_t row0, int64_t m, int64_t o, int64_t n) {
    if (n == NB) {
      if (ar_potrf != AR_F64 && !seq()) {
        // float32 storage: the leaf also left L11^-1 in float32 in X's diagonal
        // block, so the product takes the Cholesky updates' split arithmetic.
        return launch_gemm<TS, TS, TS>(ar_potrf, false, false, L + row0 * ld + o, ld,
                                       X + o * ld + o, ld, L + row0 * ld + o, ld, m, NB, NB, 1.0,
                                       false, false, KR_FULL, s, nullptr, bt,
                                       fscale ? fscale + 1 : nullptr);
      }
      const double* inv = leafinv + (o / NB) * NB * NB;
      if constexpr (std::is_same<TS, double>::value) {
        if (m / NB * bt.count <= TRSM_STRIP_TILES && !seq())
          return launch_trsm_strip(L + row0 * ld + o, ld, m, inv, s, bt);
      }
      // In place: a workgroup must own its rows' NB columns, so this launch must
      // not take the FP64 products' smaller tiles (it has more tiles than they do).
      return launch_gemm<TS, double, TS>(seq() ? AR_F64_SEQ : AR_F64, false, false, L + row0 * ld + o, ld, inv, NB,
                                         L + row0 * ld + o, ld, m, NB, NB, 1.0, false, false,
                                         KR_FULL, s, nullptr, bt);
    }
    const int64_t h = split_point(n);
    GPK_TRY(trsm(row0, m, o, h));
    GPK_TRY(launch_gemm<TS, TS, TS>(ar_potrf, false, false, L + row0 * ld + o, ld,
                                    L + (o + h) * ld + o, ld, L + row0 * ld + o + h, ld, m,
                                    n - h, h, -1.0, true, false, KR_FULL, s, nullptr, bt,
                                    fscale));
    return trsm(row0, m, o + h, n - h);
  }
  int potrf(int64_t o, int64_t n) {
    if (n == NB) return leaf(o);
    const int64_t h = split_point(n);
    GPK_TRY(potrf(o, h));
    GPK_TRY(trsm(o + h, n - h, o, h));
    GPK_TRY(launch_gemm<TS, TS, TS>(ar_potrf, false, false, L + (o + h) * ld + o, ld,
                                    L + (o + h) * ld + o, ld, L + (o + h) * ld + o + h, ld,
                                    n - h, n - h, h, -1.0, true, true, KR_FULL, s,
                                    dblk_at(o + h), bt, fscale));
    return potrf(o + h, n - h);
  }
  // The whole factorisation of one problem (no batch); `inverse`: X = L^-1 too.
  // `streams`: the look-ahead may use this thread's second stream.
  int factor(int64_t n, bool streams, bool inverse) {
    const bool f32 = std::is_same<TS, float>::value;
    if (!f32 && n <= STEPS_MAX) return potrf_steps(n, inverse);
    GPK_TRY(factor_only(n, streams));
    return inverse ? trtri(0, n) : GPK_OK;
  }
  int factor_only(int64_t n, bool streams) {
    const int64_t la = streams ? lookahead_width(n, std::is_same<TS, float>::value) : 0;
    return la > 0 ? potrf_lookahead(n, la) : potrf(0, n);
  }
  // Right-looking in single leaves on one stream (float64), the factor and, with
  // `inverse`, its inverse in one sweep.  Per leaf, three launches: the solve of the
  // column block below it and of the inverse's row block left of it; the next column
  // block's update; the next leaf beside everything else that panel updates.
  // The inverse's products fill CUs that the leaf leaves idle: the value and gradient
  // with the inverse after the factor, level by level, 1,026 us at n = 2,000 and 3,393 at
  // 4,000; in the sweep 852 and 3,245.
  int potrf_steps(int64_t n, bool inverse) {
    if constexpr (std::is_same<TS, double>::value) {
      GPK_TRY(leaf(0));
      for (int64_t o = 0; o < n; o += NB) {
        const int64_t o1 = o + NB, rest = n - o1 - NB;
        GPK_TRY(launch_step_solve(L + o1 * ld + o, X + o * ld, ld, n - o1, inverse ? o : 0,
                                  leafinv + (o / NB) * NB * NB, s));
        if (o1 == n) break;
        const TS* P = L + o1 * ld + o;
        GPK_TRY(launch_gemm<TS, TS, TS>(AR_F64, false, false, P, ld, P, ld, L + o1 * ld + o1, ld,
                                        NB + rest, NB, NB, -1.0, true, false, KR_FULL, s));
        GPK_TRY(launch_leaf_update(L, X, ld, o1, rest, inverse, leafinv + (o1 / NB) * NB * NB,
                                   leafld + o1 / NB, leafinfo + o1 / NB, s));
      }
      return GPK_OK;
    } else {
      return potrf(0, n);
    }
  }
  // Right-looking over panels of width B with a look-ahead of one panel: while
  // this stream applies panel j's update to the trailing columns beyond panel
  // j+1, a second stream factors panel j+1's diagonal block (the recursion's
  // latency-bound bottom: leaves and small updates) and solves its column
  // block, so that chain runs under the large update instead of after it.
  //   stream s : (a) diag block j+1 -= P_j P_j^T   -> ev0
  //              (b) column block j+1 -= P_j P_j^T -> ev1
  //              (c) columns beyond j+1 -= ...      (overlaps s2)
  //              wait ev2
  //   stream s2: wait ev0; potrf(diag j+1); wait ev1; trsm(column block j+1); -> ev2
  // The operations and their arithmetic are the recursion's; only the order of
  // the trailing updates differs (rank-B steps instead of halving splits).
  int potrf_lookahead(int64_t n, int64_t B) {
    hipStream_t s2 = nullptr;
    hipEvent_t ev[3];
    GPK_TRY(lookahead_resources(&s2, ev));
    // Whatever happens below, the calling stream ends up waiting for all the
    // second stream's work (an early error return included), so no work of
    // this call is left unjoined.
    StreamJoin join{s, s2, ev[2]};
    Factor<TS> G = *this;
    G.s = s2;
    GPK_TRY(potrf(0, B));
    GPK_TRY(trtri(0, B));
    GPK_TRY(trsm(B, n - B, 0, B));
    for (int64_t o = 0; o + B < n; o += B) {
      const int64_t o1 = o + B;
      const int64_t b1 = n - o1 < B ? n - o1 : B;
      const int64_t o2 = o1 + b1;
      const int64_t rest = n - o2;
      TS* P = L + o1 * ld + o;  // panel j below its diagonal block: (n - o1) x B
      GPK_TRY(launch_gemm<TS, TS, TS>(ar_potrf, false, false, P, ld, P, ld, L + o1 * ld + o1, ld,
                                      b1, b1, B, -1.0, true, true, KR_FULL, s, dblk_at(o1), bt,
                                      fscale));
      GPK_HIP_TRY(hipEventRecord(ev[0], s));
      if (rest > 0)
        GPK_TRY(launch_gemm<TS, TS, TS>(ar_potrf, false, false, P + b1 * ld, ld, P, ld,
                                        L + o2 * ld + o1, ld, rest, b1, B, -1.0, true, false,
                                        KR_FULL, s, nullptr, bt, fscale));
      GPK_HIP_TRY(hipEventRecord(ev[1], s));
      GPK_HIP_TRY(hipStreamWaitEvent(s2, ev[0], 0));
      GPK_TRY(G.potrf(o1, b1));
      GPK_TRY(G.trtri(o1, b1));
      GPK_HIP_TRY(hipStreamWaitEvent(s2, ev[1], 0));
      if (rest > 0) GPK_TRY(G.trsm(o2, rest, o1, b1));
      GPK_HIP_TRY(hipEventRecord(ev[2], s2));
      if (rest > 0)
        GPK_TRY(launch_gemm<TS, TS, TS>(ar_potrf, false, false, P + b1 * ld, ld, P + b1 * ld,
                                        ld, L + o2 * ld + o2, ld, rest, rest, B, -1.0, true, true,
                                        KR_FULL, s, dblk_at(o2), bt, fscale));
      GPK_HIP_TRY(hipStreamWaitEvent(s, ev[2], 0));
    }
    tri_unit = B;
    return GPK_OK;
  }
  // X = L^-1 below the leaves, whose diagonal blocks the leaves already wrote:
  // level by level from the deepest, all nodes of a level (independent of each
  // other) in one launch per product.  The inverse of a float64 factor of 2,000 rows:
  // 30 launches of one to 64 workgroups 1,217 us, eight launches 195 us.  (Node by node
  // is no faster for wide batches either: 4,096 GPs of 32 to 1,024 rows 58.9 ms, 59.1
  // by levels, and from 8 to 1,000 of 512 or 1,024 rows within 1.5 % both ways.)
  int trtri(int64_t o, int64_t n) {
    TriLevel lev;
    lev.o = (int)o;
    lev.n = (int)n;
    lev.unit = (int)tri_unit;
    lev.ld = (int)ld;
    for (int d = tri_depth((int)n, (int)tri_unit) - 1; d >= 0; --d) {
      lev.nodes = 1u << d;
      lev.depth = d;
      int mm, mn;
      tri_extents(lev, mm, mn);
      lev.tstride = d == 0 ? 0 : mn;
      // T = L21 X11   ((n-h) x h; X11 lower, so k >= column tile)
      lev.product = 1;
      GPK_TRY(launch_tri_level<TS>(ar_trtri, lev, mm, mn, L, ld, X, ld, T, mn, s, bt,
                                   fscale ? fscale + 1 : nullptr));
      // X21 = -X22 T  (X22 lower, so k <= row tile)
      lev.product = 2;
      GPK_TRY(launch_tri_level<TS>(ar_trtri, lev, mm, mn, X, ld, T, mn, X, ld, s, bt,
                                   fscale ? fscale + 2 : nullptr));
    }
    return GPK_OK;
  }
};

// Elements of the trtri scratch T for an n x n factorisation: the largest level's,
// for either width of its leaves.
inline int64_t factor_scratch_elems(int64_t n) {
  int64_t best = 1;
  for (const int64_t unit : {(int64_t)NB, lookahead_width(n, false), lookahead_width(n, true)}) {
    if (unit <= 0) continue;
    for (int depth = tri_depth((int)n, (int)unit) - 1; depth >= 0; --depth) {
      TriLevel lev;
      lev.nodes = 1u << depth;
      lev.depth = depth;
      lev.n = (int)n;
      lev.unit = (int)unit;
      int mm, mn;
      tri_extents(lev, mm, mn);
      const int64_t stride = depth == 0 ? 0 : mn;
      for (unsigned q = 0; q < lev.nodes; ++q) {
        int o, nn, h;
        if (!tri_node(lev, q, o, nn, h)) continue;
        const int64_t end = o * stride + (int64_t)(nn - h) * h;
        if (end > best) best = end;
      }
    }
  }
  return best;
}

}  // namespace gpk
