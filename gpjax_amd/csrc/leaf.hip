// Leaf of the recursive Cholesky: factor one NB x NB diagonal block in float64
// and form its inverse in the same sweep.
//
// Replaces the diagonal work of jnp.linalg.cholesky / slogdet
// (gpjax/linalg/operations.py:54-55,163-165).  Algorithm: right-looking
// Cholesky in panels of 16 columns; alongside it the numerators of X = L^-1 are
// eliminated row by row (forward substitution of L X = I, right-looking form).
// Both live in one NB x NB array S of 16 x 16 tiles: tile (I, J), I >= J, holds the
// trailing matrix / L, and tile (I, J), I < J, holds X^T (entry (i, c) is the
// numerator of X[c][i]).  Panel p is then tile column p of S with 16 identity
// rows added for block row p: every row y of it becomes y L11^-T, which gives
// the rows of L below the block, the rows of X^T above it, L11 itself from the
// block's own rows and X11^T from the identity rows.
//
// One workgroup of ten waves, two roles:
//   * Two panel waves, one of the 112 + 16 rows outside the pivot block per lane.
//     Each 16-lane row also holds the 16 pivot rows, one per lane, so no wave waits
//     for another inside a panel: a column step broadcasts the pivot and the pivot
//     rows' multipliers within each lane row (row_newbcast) and costs two FMAs and
//     a broadcast per remaining column; no LDS and no barrier.
//   * Eight update waves hold S in matrix-core accumulator layout (tile (I, J)
//     in wave (I + J) % 8, slot J: at most five of the 36 lower tiles per
//     wave).  Panel p updates tile column p + 1 first (phase B), which goes to
//     LDS as the next panel; the columns beyond it are updated, and panel p's
//     results stored to memory, while the panel waves factor panel p + 1
//     (phase A).
// What bounds it: the chain of 128 column steps on the panel waves, about 300
// cycles each (update and broadcast of the next pivot, its reciprocal root, scale),
// and within a panel the matrix-core updates, which share the SIMDs' float64 units
// (4,600 cycles a panel alone, up to 6,600 beside them).  Measured (one block,
// launch included): 26.5 us; panels of four columns factored by half-waves with
// LDS broadcasts and one barrier each 67 us; this layout with the multipliers
// broadcast as scalars (v_readlane, three panel waves) 29 us.  Inside an
// evaluation: n = 2,000 3.89 -> 3.32 ms, n = 300 0.79 -> 0.55 ms per Adam step.
//
// Outputs: L (lower, zero strict upper) into A, X = L^-1 (lower, zero strict
// upper) into X, X in float64 into leafinv, 2*sum(log L_kk) into *logdet and
// 1 + global index of the first non-positive pivot (or 0) into *info.  A
// non-positive pivot turns the rest of the block into NaN, which propagates
// to the objective.
#include "gemm_core.h"

namespace gpk {
namespace {

constexpr int PB = 16;                       // panel width = matrix-core tile edge
constexpr int NPAN = NB / PB;                // panels (and tile rows) of a block
constexpr int UPD_WAVES = NPAN;              // waves holding S
constexpr int PAN_WAVES = 2;                 // waves factoring the panel
constexpr int LEAF_THREADS = 64 * (UPD_WAVES + PAN_WAVES);
constexpr int PLD = PB + 1;                  // padded panel row (doubles)
constexpr int ROW_XT = NB;                   // panel buffer rows of X11^T
constexpr int ROW_L11 = NB + PB;             // panel buffer rows of L11
constexpr int PROWS = NB + 2 * PB;

// Lane J of each 16-lane row, in all lanes of that row.
template <int J>
__device__ __forceinline__ double rowcast(double v) {
  return __builtin_amdgcn_update_dpp(0.0, v, 0x150 + J /* row_newbcast:J */, 0xf, 0xf, true);
}

// 1 / sqrt(x) (the hardware estimate and one third-order step) and sqrt(x) with its
// residual corrected.  x <= 0, infinite and NaN give NaN.
__device__ __forceinline__ void roots(double x, double& inv, double& dk) {
  const double y = __builtin_amdgcn_rsq(x);
  const double e = fma(-x * y, y, 1.0);
  inv = fma(y * e, fma(e, 0.375, 0.5), y);
  const double t = x * inv;
  dk = fma(0.5 * inv, fma(-t, t, x), t);
}

// d -= (lane J of x in each 16-lane row) * f: one instruction, the broadcast and
// the sign being its operand modifiers.  x must have been written at least two wait
// states before (settle).  volatile keeps the steps in the order written below.
template <int J>
__device__ __forceinline__ void fnma_rowcast(double& d, double x, double f) {
  asm volatile("v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
               : "+v"(d)
               : "v"(x), "v"(f), "n"(J));
}
// The two wait states between a vector write of x and its use under a row broadcast.
__device__ __forceinline__ void settle(double& x) { asm volatile("s_nop 1" : "+v"(x)); }

// Column steps K .. 15 of a panel: u = the pivot row lane % 16 (the same in every
// 16-lane row), v = the lane's own row, (inv, dk) = roots of pivot K.
template <int J>
__device__ __forceinline__ void column_updates(double (&u)[PB], double (&v)[PB], double fu,
                                               double fv) {
  if constexpr (J < PB) {
    fnma_rowcast<J>(u[J], fu, fu);
    fnma_rowcast<J>(v[J], fu, fv);
    column_updates<J + 1>(u, v, fu, fv);
  }
}
template <int K>
__device__ __forceinline__ void column_steps(double (&u)[PB], double (&v)[PB], int lr, double inv,
                                             double dk) {
  double fu = u[K] * inv;
  settle(fu);
  const double fv = v[K] * inv;
  u[K] = lr == K ? dk : fu;
  v[K] = fv;
  if constexpr (K + 1 < PB) {
    // the next pivot's roots first: the other columns' updates fill their latency
    fnma_rowcast<K + 1>(u[K + 1], fu, fu);
    fnma_rowcast<K + 1>(v[K + 1], fu, fv);
    settle(u[K + 1]);
    double inv1, dk1;
    roots(rowcast<K + 1>(u[K + 1]), inv1, dk1);
    column_updates<K + 2>(u, v, fu, fv);
    __builtin_amdgcn_sched_barrier(0);
    column_steps<K + 1>(u, v, lr, inv1, dk1);
  }
}
// The same by plain square roots and quotients, which take every value.
template <int K>
__device__ __forceinline__ void plain_steps(double (&u)[PB], double (&v)[PB], int lr) {
  settle(u[K]);
  const double dk = sqrt(rowcast<K>(u[K])), inv = 1.0 / dk;
  double fu = u[K] * inv;
  settle(fu);
  const double fv = v[K] * inv;
  u[K] = lr == K ? dk : fu;
  v[K] = fv;
  column_updates<K + 1>(u, v, fu, fv);
  __builtin_amdgcn_sched_barrier(0);
  if constexpr (K + 1 < PB) plain_steps<K + 1>(u, v, lr);
}

// Factor panel p in place in P (PROWS x PLD), wave `a` of the panel waves.
// ident: the PB x PB identity (rows of PLD).
__device__ __forceinline__ void factor_panel(double* P, const double* ident, int p, int a,
                                             int lane) {
  const int lr = lane & (PB - 1);
  const int q = a * 64 + lane;  // the rows outside block p, then the identity rows
  const int row = q < p * PB ? q : q + PB;
  const int unit = q - (NB - PB);
  double u[PB], v[PB];
  const double* src = unit < 0 ? P + row * PLD : ident + unit * PLD;
  auto fetch = [&]() {
#pragma unroll
    for (int j = 0; j < PB; ++j) {
      u[j] = P[(p * PB + lr) * PLD + j];
      v[j] = src[j];
    }
  };
  fetch();
  double inv, dk;
  roots(rowcast<0>(u[0]), inv, dk);
  column_steps<0>(u, v, lr, inv, dk);
  // A pivot that is not positive and finite (every lane row of both waves sees the
  // same): the panel again from its untouched rows by the plain steps; a
  // non-positive pivot turns what follows into NaN.
  double dg = 1.0;
#pragma unroll
  for (int j = 0; j < PB; ++j) dg = lr == j ? u[j] : dg;
  if (__ballot(!(dg > 0.0 && dg < __builtin_inf())) != 0) {
    fetch();
    plain_steps<0>(u, v, lr);
  }
  const int dst = unit < 0 ? row : ROW_XT + unit;
#pragma unroll
  for (int j = 0; j < PB; ++j) {
    P[dst * PLD + j] = v[j];
    if (q < PB) P[(ROW_L11 + lr) * PLD + j] = u[j];
  }
}

// LDS of one leaf.
struct LeafShared {
  double buf[2][PROWS * PLD];
  double ident[PB * PLD];
  double dk_s[NB];
};

// The leaf of the block at row and column o: the whole workgroup.
template <typename TS>
__device__ __forceinline__ void leaf_block(LeafShared& sh, TS* A, TS* X, int64_t ld, int64_t o,
                                           double* __restrict__ leafinv,
                                           double* __restrict__ logdet, int* __restrict__ info,
                                           const double* __restrict__ dsrc) {
  auto& buf = sh.buf;
  auto& ident = sh.ident;
  auto& dk_s = sh.dk_s;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lr = lane >> 4, lc = lane & 15;  // accumulator element r: row lr + 4 r, column lc
  TS* Ab = A + o * ld + o;
  TS* Xb = X + o * ld + o;

  if (w >= UPD_WAVES) {
    // ---- panel waves ----
    const int a = w - UPD_WAVES;
    int bad = NB;
    for (int e = a * 64 + lane; e < PB * PB; e += 64 * PAN_WAVES)
      ident[(e / PB) * PLD + e % PB] = e / PB == e % PB ? 1.0 : 0.0;
    __syncthreads();  // panel 0 staged
#pragma unroll 1
    for (int p = 0; p < NPAN; ++p) {
      double* P = buf[p & 1];
      factor_panel(P, ident, p, a, lane);
      if (a == 0) {
        double dg = 1.0;
        if (lane < PB) dk_s[p * PB + lane] = dg = P[(ROW_L11 + lane) * PLD + lane];
        const unsigned long long m = __ballot(!(dg > 0.0));  // non-positive pivots give NaN
        if (m != 0 && bad == NB) bad = p * PB + __builtin_ctzll(m);
      }
      __syncthreads();  // panel p factored
      __syncthreads();  // panel p + 1 staged
    }
    if (a == 0) {
      double s = log(dk_s[lane]) + log(dk_s[lane + 64]);
#pragma unroll
      for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off);
      if (lane == 0) {
        *logdet = 2.0 * s;
        *info = bad < NB ? (int)(o + bad + 1) : 0;
      }
    }
    return;
  }

  // ---- update waves ----
  f64x4 acc[NPAN];  // slot J: tile ((w - J) mod 8, J)
  auto load_tiles = [&](const auto* src, int64_t lds) {
#pragma unroll
    for (int J = 0; J < NPAN; ++J) {
      const int I = (w - J) & (NPAN - 1);
      acc[J] = f64x4{0.0, 0.0, 0.0, 0.0};
      if (I >= J) {
        const auto* t = src + (I * PB + lr) * lds + J * PB + lc;
#pragma unroll
        for (int r = 0; r < 4; ++r) acc[J][r] = (double)t[4 * r * lds];
      }
    }
  };
  if (dsrc) load_tiles(dsrc, NB);
  else load_tiles(Ab, ld);
  auto stage = [&](int J, double* P) {  // tile of slot J -> panel buffer
    const int I = (w - J) & (NPAN - 1);
#pragma unroll
    for (int r = 0; r < 4; ++r) P[(I * PB + lr + 4 * r) * PLD + lc] = acc[J][r];
  };
  // acc[J] -= R(I) G(J)^T with panel p's finished rows
  auto update = [&](int J, int p, const double* P) {
    const int I = (w - J) & (NPAN - 1);
    const double* R = P + (I == p ? ROW_XT : I * PB) * PLD;
    const double* G = P + J * PB * PLD;
    double av[4], bv[4];
#pragma unroll
    for (int kk = 0; kk < 4; ++kk) {
      av[kk] = -R[lc * PLD + 4 * kk + lr];
      bv[kk] = G[lc * PLD + 4 * kk + lr];
    }
#pragma unroll
    for (int kk = 0; kk < 4; ++kk)
      acc[J] = __builtin_amdgcn_mfma_f64_16x16x4f64(av[kk], bv[kk], acc[J], 0, 0, 0);
  };
  // This wave's share of panel p's results: tile (w, p) of L (zero for w < p) and,
  // for w <= p, tile (p, w) of X and the zero tile (w, p) above X's diagonal.
  auto emit = [&](int p, const double* P) {
    const double* R = P + (w == p ? ROW_L11 : w * PB) * PLD;
    const double* Y = P + (w == p ? ROW_XT : w * PB) * PLD;
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int i = lr + 4 * r;
      const int64_t g = (int64_t)(w * PB + i) * ld + p * PB + lc;
      if (w > p) {
        Ab[g] = (TS)R[i * PLD + lc];
      } else {
        Ab[g] = w == p && lc <= i ? (TS)R[i * PLD + lc] : (TS)0.0;
        if (w < p) {
          Xb[g] = (TS)0.0;
          leafinv[(w * PB + i) * NB + p * PB + lc] = 0.0;
        }
        const double x = w == p && lc > i ? 0.0 : Y[lc * PLD + i];
        Xb[(int64_t)(p * PB + i) * ld + w * PB + lc] = (TS)x;
        leafinv[(p * PB + i) * NB + w * PB + lc] = x;
      }
    }
  };

  stage(0, buf[0]);
  __syncthreads();  // panel 0 staged
  for (int p = 0; p < NPAN; ++p) {
    // phase A: panel p - 1 into the tile columns beyond p, and its results out
    if (p > 0) {
      const double* P = buf[(p - 1) & 1];
#pragma unroll
      for (int J = 2; J < NPAN; ++J) {
        const int I = (w - J) & (NPAN - 1);
        if (J > p && (I >= J || I <= p - 1)) update(J, p - 1, P);
      }
      emit(p - 1, P);
    }
    __syncthreads();  // panel p factored
    // phase B: panel p into tile column p + 1 (all of it takes part), staged
#pragma unroll
    for (int J = 1; J < NPAN; ++J) {
      if (J == p + 1) {
        update(J, p, buf[p & 1]);
        stage(J, buf[J & 1]);
      }
    }
    __syncthreads();  // panel p + 1 staged
  }
  emit(NPAN - 1, buf[(NPAN - 1) & 1]);
}

template <typename TS>
__global__ __launch_bounds__(LEAF_THREADS) void leaf_kernel(TS* A, TS* X, int64_t ld, int64_t o,
                                                            double* __restrict__ leafinv,
                                                            double* __restrict__ logdet,
                                                            int* __restrict__ info,
                                                            const double* __restrict__ dsrc,
                                                            Batch bt) {
  __shared__ LeafShared sh;
  leaf_block(sh, bws(A, bt), bws(X, bt), ld, o, bws(leafinv, bt), bws(logdet, bt), bws(info, bt),
             bws(dsrc, bt));
}

// The leaf at o (first workgroup) beside the updates by the solved panel before it, P =
// the NB columns before o (the others): C -= P P^T over the lower NB-tiles from row and
// column o + NB on and, with `inverse`, the rows of the inverse not yet finished:
// X[J][I] -= L[J][p] X[p][I] for every block row J >= o / NB and column I <= p =
// o / NB - 1 (X[J][p] starts here: it is written without being read).  One launch
// instead of several on two streams, whose hand-over costs more than the leaf's
// dependents (see Factor::potrf_steps).  A workgroup takes a 64 x 64 quarter of a tile,
// eight of its waves 16 x 32 each straight from global memory.
__global__ __launch_bounds__(LEAF_THREADS) void leaf_update_kernel(
    double* A, double* X, int64_t ld, int64_t o, int64_t trailing, int inverse,
    double* __restrict__ leafinv, double* __restrict__ logdet, int* __restrict__ info) {
  __shared__ LeafShared sh;
  if (blockIdx.x == 0) {
    leaf_block<double>(sh, A, X, ld, o, leafinv, logdet, info, nullptr);
    return;
  }
  int b = blockIdx.x - 1;
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  if (w >= 8) return;
  const int64_t ms = ((b >> 1) & 1) * 64 + (w >> 1) * 16, ns = (b & 1) * 64 + (w & 1) * 32;
  const int lr = lane >> 4, lc = lane & 15;
  b /= 4;
  f64x4 acc[1][2];
  double cv[2][4];
  double* C;
  int64_t mw, nw;
  auto fetch = [&](bool read) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int r = 0; r < 4; ++r)
        cv[j][r] = read ? C[(mw + lr + 4 * r) * ld + nw + 16 * j + lc] : 0.0;
  };
  if (b < trailing) {
    int64_t mt, nt;
    lower_tile(b, mt, nt);
    mw = mt * NB + ms;
    nw = nt * NB + ns;
    const double* P = A + (o + NB) * ld + o - NB;
    C = A + (o + NB) * ld + o + NB;
    DirectLoop<false, false, 1, 2> loop(P, ld, P, ld, mw, nw, lane, 0, NB);
    fetch(true);
    loop.run(acc);
  } else {
    const int p = (int)(o / NB) - 1, q = b - (int)trailing;
    const int J = q / (p + 1), I = q % (p + 1);
    mw = J * NB + ms;
    nw = I * NB + ns;
    C = X + o * ld;
    DirectLoop<false, true, 1, 2> loop(A + o * ld + o - NB, ld, X + (o - NB) * ld, ld, mw, nw,
                                       lane, 0, NB);
    fetch(I < p);
    loop.run(acc);
  }
#pragma unroll
  for (int j = 0; j < 2; ++j)
#pragma unroll
    for (int r = 0; r < 4; ++r)
      C[(mw + lr + 4 * r) * ld + nw + 16 * j + lc] = cv[j][r] - acc[0][j][r];
}

// The leaf as a right-looking sweep by columns, for Factor::seq: thread t of 1,024 holds
// the 4 x 4 block at rows 4 (t % 32), columns 4 (t / 32) of one array with the trailing
// matrix / L below the diagonal and the numerators of X = L^-1, transposed, above it.
// The half-wave that owns a panel of four columns factors it among its own lanes and
// publishes it; after one barrier every thread to the right applies the rank-4 update.
// 67 us, bound by its 32 dependent panels (leaf_kernel: 26.5), but each entry takes one
// FMA per column, in order.
constexpr int SWEEP_THREADS = 1024;
constexpr int EB = 4;
constexpr int BPR = NB / EB;
__global__ __launch_bounds__(SWEEP_THREADS) void leaf_sweep_kernel(
    double* A, double* X, int64_t ld, int64_t o, double* __restrict__ leafinv,
    double* __restrict__ logdet, int* __restrict__ info) {
  // pub[buf][kk][i]: the step factors of the four columns of the last panel
  // (row factor of row i; for rows below the step's column also its column
  // factor).  Double-buffered across panels.
  __shared__ double pub[2][EB][NB];
  __shared__ double dk_s[NB];
  __shared__ double dinv_s[NB];
  __shared__ int bad_s;
  __shared__ double tr_s[NB][NB + 1];

  const int t = threadIdx.x;
  const int rb = (t % BPR) * EB;   // first row of this thread's block
  const int cb = (t / BPR) * EB;   // first column (the half-wave t / 32 owns columns cb .. cb+3)
  const int hl = t % BPR;          // lane within the half-wave: rows 4 hl .. 4 hl + 3
  const int hbase = (t & 63) & ~(BPR - 1);  // first wave lane of this half-wave
  // Stage the block through LDS so that global reads stay row-contiguous.
  for (int e = t; e < NB * NB; e += SWEEP_THREADS) {
    const int i = e / NB, j = e % NB;
    tr_s[i][j] = A[(o + i) * ld + o + j];
  }
  if (t == 0) bad_s = NB;
  __syncthreads();
  double s[EB][EB];
#pragma unroll
  for (int a = 0; a < EB; ++a)
#pragma unroll
    for (int b = 0; b < EB; ++b) s[a][b] = (cb + b <= rb + a) ? tr_s[rb + a][cb + b] : 0.0;

  for (int p = 0; p < NB / EB; ++p) {
    const int c0 = p * EB;  // the panel's columns c0 .. c0 + 3
    if (cb == c0) {
      // Factor the panel inside this half-wave.  Step k = c0 + kk: the pivot
      // and the panel's own entries of column k (rows c0 .. c0+3) sit in the
      // half-wave lane p; each is broadcast from there.  As in the unblocked
      // sweep, entry (i, j), j > k, takes one FMA with row factor
      // f_i = s_ik / d_k (1 / d_k on the diagonal) and column factor s_jk / d_k
      // when i >= j (trailing update of L) or i <= k (numerator of X[j][i]).
#pragma unroll
      for (int kk = 0; kk < EB; ++kk) {
        const int k = c0 + kk;
        double cv[EB];
#pragma unroll
        for (int a = 0; a < EB; ++a) cv[a] = __shfl(s[a][kk], hbase + p);
        const double piv = cv[kk];
        const double dk = sqrt(piv);
        const double inv = 1.0 / dk;
        double f[EB];
#pragma unroll
        for (int a = 0; a < EB; ++a) f[a] = (rb + a == k) ? inv : s[a][kk] * inv;
#pragma unroll
        for (int b = kk + 1; b < EB; ++b) {
          const double g = cv[b] * inv;  // column factor of column c0 + b
#pragma unroll
          for (int a = 0; a < EB; ++a) {
            const int i = rb + a, j = c0 + b;
            const double fa = (i >= j || i <= k) ? f[a] : 0.0;
            s[a][b] = fma(-fa, g, s[a][b]);
          }
        }
#pragma unroll
        for (int a = 0; a < EB; ++a) s[a][kk] = (rb + a == k) ? dk : f[a];
#pragma unroll
        for (int a = 0; a < EB; ++a) pub[p & 1][kk][rb + a] = f[a];
        if (hl == p) {
          dk_s[k] = dk;
          dinv_s[k] = inv;
          if (!(piv > 0.0) && k < bad_s) bad_s = k;
        }
      }
    }
    __syncthreads();
    if (cb > c0) {
      // Rank-4 update of the columns right of the panel, steps in order.
      const double* P = &pub[p & 1][0][0];
#pragma unroll
      for (int kk = 0; kk < EB; ++kk) {
        const int k = c0 + kk;
        double fr[EB], g[EB];
#pragma unroll
        for (int a = 0; a < EB; ++a) fr[a] = P[kk * NB + rb + a];
#pragma unroll
        for (int b = 0; b < EB; ++b) g[b] = P[kk * NB + cb + b];
#pragma unroll
        for (int a = 0; a < EB; ++a) {
          const int i = rb + a;
          // j = cb + b > k always here; the mask is i >= j or i <= k
          const double flo = fr[a];
          const double fhi = (i <= k) ? fr[a] : 0.0;
#pragma unroll
          for (int b = 0; b < EB; ++b) {
            const double fa = (i >= cb + b) ? flo : fhi;
            s[a][b] = fma(-fa, g[b], s[a][b]);
          }
        }
      }
    }
  }

  // L (lower incl. diagonal) and X (from the upper part, transposed) staged
  // in LDS for row-contiguous writes.
  __syncthreads();
#pragma unroll
  for (int a = 0; a < EB; ++a)
#pragma unroll
    for (int b = 0; b < EB; ++b) tr_s[rb + a][cb + b] = s[a][b];
  if (t < NB) dk_s[t] = log(dk_s[t]);
  __syncthreads();
  for (int e = t; e < NB * NB; e += SWEEP_THREADS) {
    const int i = e / NB, j = e % NB;
    A[(o + i) * ld + o + j] = (j <= i) ? tr_s[i][j] : 0.0;
    const double v = (j < i) ? tr_s[j][i] : (j == i ? dinv_s[i] : 0.0);
    X[(o + i) * ld + o + j] = v;
    leafinv[e] = v;
  }
  if (t == 0) {
    double ld_acc = 0.0;  // in column order, as the sweep produced the pivots
    for (int k = 0; k < NB; ++k) ld_acc += dk_s[k];
    *logdet = 2.0 * ld_acc;
    *info = bad_s < NB ? (int)(o + bad_s + 1) : 0;
  }
}

}  // namespace

template <typename TS>
int launch_leaf(TS* A, TS* X, int64_t ld, int64_t o, double* leafinv, double* logdet, int* info,
                const double* dsrc, hipStream_t s, const Batch& bt) {
  hipLaunchKernelGGL(leaf_kernel<TS>, dim3(1, 1, bt.count), dim3(LEAF_THREADS), 0, s, A, X, ld,
                     o, leafinv, logdet, info, dsrc, bt);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

int launch_leaf_sweep(double* A, double* X, int64_t ld, int64_t o, double* leafinv,
                      double* logdet, int* info, hipStream_t s) {
  hipLaunchKernelGGL(leaf_sweep_kernel, dim3(1), dim3(SWEEP_THREADS), 0, s, A, X, ld, o, leafinv,
                     logdet, info);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

int launch_leaf_update(double* A, double* X, int64_t ld, int64_t o, int64_t rest, bool inverse,
                       double* leafinv, double* logdet, int* info, hipStream_t s) {
  if (o < NB || o % NB || rest < 0 || rest % NB) {
    set_error("leaf update: block at %lld with %lld rows beyond it", (long long)o,
              (long long)rest);
    return GPK_ERR_BAD_ARG;
  }
  const int64_t T = rest / NB, trailing = T * (T + 1) / 2;
  const int64_t inv = inverse ? (T + 1) * (o / NB) : 0;
  hipLaunchKernelGGL(leaf_update_kernel, dim3((unsigned)(1 + 4 * (trailing + inv))),
                     dim3(LEAF_THREADS), 0, s, A, X, ld, o, trailing, inverse ? 1 : 0, leafinv,
                     logdet, info);
  GPK_LAUNCH_CHECK();
  return GPK_OK;
}

template int launch_leaf<double>(double*, double*, int64_t, int64_t, double*, double*, int*,
                                 const double*, hipStream_t, const Batch&);
template int launch_leaf<float>(float*, float*, int64_t, int64_t, double*, double*, int*,
                                const double*, hipStream_t, const Batch&);

}  // namespace gpk
