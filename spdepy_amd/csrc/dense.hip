// Dense FP64 kernels for the multifrontal factorisation, written for CDNA4
// (gfx950): batched tile-list GEMM on v_mfma_f64_16x16x4f64 and the
// bandwidth-bound products of one right-hand side.
#include <hip/hip_runtime.h>

#include "internal.hpp"

#include <vector>

namespace spde {

typedef double d4 __attribute__((ext_vector_type(4)));

// ----------------------------------------------------------------- GEMM
// C(M x N) = alpha op(A) op(B) + beta C, column-major, FP64 MFMA over a list of
// tiles: register-fed (gemm_reg_body), but for 64x64 tiles of A^T B
// (gemm_tn_body).  The MFMA computes the transposed tile (B-fragment as the matrix
// "A" input) so that the 16 lanes of a row group own 16 consecutive rows of one
// column of C: stores are 128-byte coalesced in column-major memory.  Accumulator
// layout of v_mfma_f64_16x16x4f64 (measured): lane l, register v holds
// D[l/16 + 4v][l%16].
// SPLIT: the block computes the chunk t.pad of `split` chunks of the tile's
// K range (each a multiple of 16 deep) and writes the raw 64x64 partial tile
// to ws + blockIdx.x * 4096 (column-major, ld 64); split_reduce_kernel then
// applies alpha, beta and the lower-triangle rule.
// List entry of block b: the dispatcher hands blocks to the eight XCDs in
// turn (b and b + 8 share an XCD and its L2).  Inside every full group of 64
// blocks, XCD x takes the eight consecutive entries 8x .. 8x + 7, which share
// operand panels (a tile row of a problem is consecutive in the list); the
// list order, deepest tiles first, holds at the granularity of a group.
__device__ __forceinline__ int xcd_tile(int b, int nb) {
  const int g = b >> 6;
  if ((g + 1) * 64 > nb) return b;
  const int r = b & 63;
  return (g << 6) + ((r & 7) << 3) + (r >> 3);
}

// A^T B in 64x64 tiles, both operands with contiguous k, staged in LDS: four waves in
// a 2x2 arrangement, each 32 x 32.  LDS is double buffered and the next 16-deep
// K-slice is prefetched into registers while the current one feeds the MFMAs; the
// tiles are m-major (n-major), as they come from memory, with pitch 17.
template <bool SPLIT>
__device__ __forceinline__ void gemm_tn_body(const GemmProb* __restrict__ probs, const GemmTile* __restrict__ tiles,
                                             const Bases& bases, int split = 1, double* __restrict__ ws = nullptr) {
  constexpr int BM = 64, BN = 64, BK = 16, PITCH = BK + 1, TM = 2, TN = 2, LOADS = BM * BK / 256, STEP = 256 / BK;
  __shared__ double As[2][BM * PITCH];
  __shared__ double Bs[2][BN * PITCH];
  const GemmTile t = tiles[SPLIT ? (int)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x)];
  const GemmProb P = probs[t.prob];
  const double* __restrict__ A = bases.p[P.a_base] + P.a_off;
  const double* __restrict__ B = bases.p[P.b_base] + P.b_off;
  double* __restrict__ C = bases.p[P.c_base] + P.c_off;
  const int M = P.M, N = P.N;
  const int m0 = t.tm * BM, n0 = t.tn * BN;
  int kb = 0, K = P.K;  // this block's K range [kb, K): the zeros of a triangular operand are skipped
  if (P.kmode == 1)
    kb = min(K, n0);
  else if (P.kmode == 2)
    kb = min(K, m0);
  else if (P.kmode == 3)
    K = min(K, m0 + BM);
  if constexpr (SPLIT) {
    const int kc = ((K - kb + split - 1) / split + 15) / 16 * 16;
    const int k0 = min(K, kb + t.pad * kc);
    K = min(K, k0 + kc);
    kb = k0;
  }
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = (wave & 1) * 32, wn = (wave >> 1) * 32;
  const int lr = lane & 15, lk = lane >> 4;
  const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
  const int row = tid / BK, col = tid % BK;  // a thread's rows row + q STEP of both tiles, k = col
  auto at = [](int k, int m) { return m * PITCH + k; };
  d4 acc[TN][TM];
#pragma unroll
  for (int x = 0; x < TN; ++x)
#pragma unroll
    for (int y = 0; y < TM; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
  double ra[LOADS], rb[LOADS];
  auto load = [&](int k0) {
    k0 += kb;
    const bool full = interior && (k0 + BK <= K);
    const int gk = k0 + col;
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int gm = m0 + row + q * STEP;
      ra[q] = (full || (gm < M && gk < K)) ? A[gk + (int64_t)gm * P.lda] : 0.0;
    }
#pragma unroll
    for (int q = 0; q < LOADS; ++q) {
      const int gn = n0 + row + q * STEP;
      rb[q] = (full || (gn < N && gk < K)) ? B[gk + (int64_t)gn * P.ldb] : 0.0;
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int q = 0; q < LOADS; ++q) As[buf][at(col, row + q * STEP)] = ra[q];
#pragma unroll
    for (int q = 0; q < LOADS; ++q) Bs[buf][at(col, row + q * STEP)] = rb[q];
  };
  const int nk = (K - kb + BK - 1) / BK;
  if (nk > 0) {
    load(0);
    store(0);
  }
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1;
    if (kt + 1 < nk) load((kt + 1) * BK);
    double fa[2][TM], fb[2][TN];
#pragma unroll
    for (int mi = 0; mi < TM; ++mi) fa[0][mi] = As[cur][at(lk, wm + mi * 16 + lr)];
#pragma unroll
    for (int ni = 0; ni < TN; ++ni) fb[0][ni] = Bs[cur][at(lk, wn + ni * 16 + lr)];
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int f = s & 1;
      if (s < 3) {
#pragma unroll
        for (int mi = 0; mi < TM; ++mi) fa[f ^ 1][mi] = As[cur][at(4 * (s + 1) + lk, wm + mi * 16 + lr)];
#pragma unroll
        for (int ni = 0; ni < TN; ++ni) fb[f ^ 1][ni] = Bs[cur][at(4 * (s + 1) + lk, wn + ni * 16 + lr)];
      }
#pragma unroll
      for (int ni = 0; ni < TN; ++ni)
#pragma unroll
        for (int mi = 0; mi < TM; ++mi)
          acc[ni][mi] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[f][ni], fa[f][mi], acc[ni][mi], 0, 0, 0);
    }
    if (kt + 1 < nk) store(cur ^ 1);
    __syncthreads();
  }
  if constexpr (SPLIT) {
    double* w = ws + (int64_t)blockIdx.x * (BM * BN);
#pragma unroll
    for (int ni = 0; ni < TN; ++ni)
#pragma unroll
      for (int mi = 0; mi < TM; ++mi)
#pragma unroll
        for (int v = 0; v < 4; ++v)
          w[(wm + mi * 16 + lr) + (wn + ni * 16 + lk + 4 * v) * BM] = acc[ni][mi][v];
    return;
  }
  const double alpha = P.alpha, beta = P.beta;
  // lower problems: the part of a diagonal tile above the diagonal is left
  // untouched (it is never read, and stays as initialised)
  const bool diag_tile = P.lower && t.tm == t.tn;
#pragma unroll
  for (int ni = 0; ni < TN; ++ni)
#pragma unroll
    for (int mi = 0; mi < TM; ++mi)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int m = m0 + wm + mi * 16 + lr;
        const int n = n0 + wn + ni * 16 + lk + 4 * v;
        if ((interior || (m < M && n < N)) && !(diag_tile && m < n)) {
          double* c = C + m + (int64_t)n * P.ldc;
          const double r = alpha * acc[ni][mi][v];
          *c = (beta == 0.0) ? r : r + beta * (*c);
        }
      }
}

// The product without LDS.  An FP64 MFMA keeps its SIMD busy for 64
// cycles and consumes two 512-byte fragments, so the matrix cores are fed
// from L1/L2 directly and no wave ever waits at a barrier.  Each lane loads
// its own fragment elements: lane (lr, lk) = (lane % 16, lane / 16) holds, for
// the sub-steps s = 0..3 of a 16-deep slab, k = 4 lk + s of row lr of each
// 16-row fragment.  The order of k inside a slab is free as long as both
// operands use it, and this one lets an operand whose k is contiguous (op(A) =
// A^T, op(B) = B) be read 16 bytes at a time (VEC: its offset and leading
// dimension are even); an operand with contiguous rows reads 128-byte segments.
// A half of the slab (two sub-steps) is reloaded for the next slab as soon as
// its MFMAs are issued, two to four thousand cycles before its use.  Rows past
// the edge are clamped (their results are not stored); the last, partial
// slab loads zeros past K.
// Alone on the chip (TFLOP/s; LDS kernels before -> this one, 78.6 peak):
// 4096^3 NT 58 -> 65, NN 58 -> 67, TN 51 -> 64; 4096 x 1920 x 4096 NT 53 -> 59,
// NN 54 -> 60, TN 47 -> 66; 64x64 tiles NT 46 -> 56.  With 64x64 tiles and k
// contiguous in both operands the 16-line loads bound it (38 against 52
// TFLOP/s), so that form is staged (gemm_tn_body).
template <bool KC, bool VEC, int T>
__device__ __forceinline__ void load_half(double (&f)[T][4], const uint32_t (&off)[T], const char* base, int64_t ldb,
                                          int h) {
  if constexpr (KC) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      if constexpr (VEC) {
        const double2 x = *(const double2*)(base + off[t] + h * 16);
        f[t][2 * h] = x.x;
        f[t][2 * h + 1] = x.y;
      } else {
        f[t][2 * h] = *(const double*)(base + off[t] + h * 16);
        f[t][2 * h + 1] = *(const double*)(base + off[t] + h * 16 + 8);
      }
    }
  } else {
#pragma unroll
    for (int u = 0; u < 2; ++u) {
      const char* b = base + (2 * h + u) * ldb;
#pragma unroll
      for (int t = 0; t < T; ++t) f[t][2 * h + u] = *(const double*)(b + off[t]);
    }
  }
}
// The partial slab: k = 4 lk + s < rem.
template <bool KC, int T>
__device__ __forceinline__ void load_tail(double (&f)[T][4], const uint32_t (&off)[T], const char* base, int64_t ldb,
                                          int lk, int rem) {
#pragma unroll
  for (int s = 0; s < 4; ++s) {
    const bool in = 4 * lk + s < rem;
#pragma unroll
    for (int t = 0; t < T; ++t) f[t][s] = in ? *(const double*)(base + off[t] + (KC ? (int64_t)s * 8 : s * ldb)) : 0.0;
  }
}

// PULL: C = alpha op(A) op(B) + the children's update blocks (the extend-add
// of the multifrontal method, read once in place of a read-modify-write of C).
template <bool TA, bool TB, bool VEC, int TM, int TN, bool SPLIT = false, bool PULL = false>
__device__ __forceinline__ void gemm_reg_body(const GemmProb* __restrict__ probs, const GemmTile* __restrict__ tiles,
                                              const Bases& bases, int split = 1, double* __restrict__ ws = nullptr) {
  constexpr int BM = 32 * TM, BN = 32 * TN;  // four waves, 2 x 2
  constexpr bool AKC = TA, BKC = !TB;        // k contiguous
  const GemmTile t = tiles[SPLIT ? (int)blockIdx.x : xcd_tile(blockIdx.x, gridDim.x)];
  const GemmProb P = probs[t.prob];
  const int M = P.M, N = P.N;
  const int m0 = t.tm * BM, n0 = t.tn * BN;
  int kb = 0, K = P.K;  // this block's K range [kb, K): the zeros of a triangular operand are skipped
  if (P.kmode == 1)
    kb = min(K, n0);
  else if (P.kmode == 2)
    kb = min(K, m0);
  else if (P.kmode == 3)
    K = min(K, m0 + BM);
  if constexpr (SPLIT) {
    const int kc = ((K - kb + split - 1) / split + 15) / 16 * 16;
    const int k0 = min(K, kb + t.pad * kc);
    K = min(K, k0 + kc);
    kb = k0;
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int wm = (wave & 1) * 16 * TM, wn = (wave >> 1) * 16 * TN;
  // wave-uniform bases at the tile's first row and column and at kb; the lane
  // offsets stay below 2^32 (128 rows or 12 columns of one front, 64 columns of a
  // solution: checked when the launch is made)
  const int64_t lda = (int64_t)P.lda * 8, ldb = (int64_t)P.ldb * 8;
  const char* pa = (const char*)(bases.p[P.a_base] + P.a_off) + (AKC ? m0 * lda + kb * 8ll : m0 * 8ll + kb * lda);
  const char* pb = (const char*)(bases.p[P.b_base] + P.b_off) + (BKC ? n0 * ldb + kb * 8ll : n0 * 8ll + kb * ldb);
  uint32_t oa[TM], ob[TN];
#pragma unroll
  for (int y = 0; y < TM; ++y) {
    const int r = min(wm + y * 16 + lr, M - 1 - m0);
    oa[y] = AKC ? (uint32_t)(r * (uint32_t)lda + lk * 32) : (uint32_t)(r * 8 + lk * 4 * (uint32_t)lda);
  }
#pragma unroll
  for (int x = 0; x < TN; ++x) {
    const int c = min(wn + x * 16 + lr, N - 1 - n0);
    ob[x] = BKC ? (uint32_t)(c * (uint32_t)ldb + lk * 32) : (uint32_t)(c * 8 + lk * 4 * (uint32_t)ldb);
  }
  const int64_t sa = AKC ? 128 : 16 * lda, sb = BKC ? 128 : 16 * ldb;
  d4 acc[TN][TM];
#pragma unroll
  for (int x = 0; x < TN; ++x)
#pragma unroll
    for (int y = 0; y < TM; ++y) acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
  double fa[TM][4], fb[TN][4];
  auto mul = [&](int h) {
#pragma unroll
    for (int s = 2 * h; s < 2 * h + 2; ++s)
#pragma unroll
      for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < TM; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[x][s], fa[y][s], acc[x][y], 0, 0, 0);
  };
  const int nk = max(K - kb, 0) >> 4, rem = max(K - kb, 0) & 15;
  if (nk > 0) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      load_half<AKC, VEC, TM>(fa, oa, pa, lda, h);
      load_half<BKC, VEC, TN>(fb, ob, pb, ldb, h);
    }
    for (int kt = 1; kt < nk; ++kt) {
      pa += sa;
      pb += sb;
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        mul(h);
        __builtin_amdgcn_sched_barrier(0);
        load_half<AKC, VEC, TM>(fa, oa, pa, lda, h);
        load_half<BKC, VEC, TN>(fb, ob, pb, ldb, h);
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    mul(0);
    mul(1);
    pa += sa;
    pb += sb;
  }
  if (rem) {
    load_tail<AKC, TM>(fa, oa, pa, lda, lk, rem);
    load_tail<BKC, TN>(fb, ob, pb, ldb, lk, rem);
    mul(0);
    mul(1);
  }
  if constexpr (SPLIT) {
    double* w = ws + (int64_t)blockIdx.x * (BM * BN);
#pragma unroll
    for (int x = 0; x < TN; ++x)
#pragma unroll
      for (int y = 0; y < TM; ++y)
#pragma unroll
        for (int v = 0; v < 4; ++v) w[(wm + y * 16 + lr) + (wn + x * 16 + lk + 4 * v) * BM] = acc[x][y][v];
    return;
  }
  double* C = bases.p[P.c_base] + P.c_off;
  const double alpha = P.alpha, beta = P.beta;
  const bool interior = (m0 + BM <= M) && (n0 + BN <= N);
  // lower problems: the part of a tile above the diagonal is left
  // untouched (it is never read, and stays as initialised)
  const bool straddles = P.lower && m0 < n0 + BN;
  Pull q{};
  int im[TM][2];
  if constexpr (PULL) {
    q = bases.pulls[P.pull];
#pragma unroll
    for (int y = 0; y < TM; ++y)
#pragma unroll
      for (int c = 0; c < 2; ++c)
        im[y][c] = child_row(bases.inv, q, c, P.pull_row + min(m0 + wm + y * 16 + lr, M - 1));
  }
#pragma unroll
  for (int x = 0; x < TN; ++x)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int n = n0 + wn + x * 16 + lk + 4 * v;
      int jn[2];
      if constexpr (PULL) {
#pragma unroll
        for (int c = 0; c < 2; ++c) jn[c] = child_row(bases.inv, q, c, P.pull_row + min(n, N - 1));
      }
#pragma unroll
      for (int y = 0; y < TM; ++y) {
        const int m = m0 + wm + y * 16 + lr;
        if ((interior || (m < M && n < N)) && !(straddles && m < n)) {
          double* c = C + m + (int64_t)n * P.ldc;
          const double r = alpha * acc[x][y][v];
          if constexpr (PULL)
            *c = assembled(bases.p[kFront], r, q, im[y][0], im[y][1], jn[0], jn[1]);
          else
            *c = (beta == 0.0) ? r : r + beta * (*c);
        }
      }
    }
}

// 64x64 tiles.
template <bool TA, bool TB, bool VEC>
__global__ __launch_bounds__(256) void gemm64_kernel(const GemmProb* __restrict__ probs,
                                                     const GemmTile* __restrict__ tiles, Bases bases) {
  if constexpr (TA && !TB)
    gemm_tn_body<false>(probs, tiles, bases);
  else
    gemm_reg_body<TA, TB, VEC, 2, 2>(probs, tiles, bases);
}

// The level SYRK with the children's update blocks.
template <int TM>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TM == 4 ? 3 : 4, TM == 4 ? 3 : 8))) void
syrk_pull_kernel(const GemmProb* __restrict__ probs, const GemmTile* __restrict__ tiles, Bases bases) {
  gemm_reg_body<false, true, true, TM, 2, false, true>(probs, tiles, bases);
}

// Split-K partial tiles (64x64) and their ordered sum.
template <bool TA, bool TB, bool VEC>
__global__ __launch_bounds__(256) void gemm64_split_kernel(const GemmProb* __restrict__ probs,
                                                           const GemmTile* __restrict__ tiles, Bases bases, int split,
                                                           double* __restrict__ ws) {
  if constexpr (TA && !TB)
    gemm_tn_body<true>(probs, tiles, bases, split, ws);
  else
    gemm_reg_body<TA, TB, VEC, 2, 2, true>(probs, tiles, bases, split, ws);
}

// Block (b, y): quarter y of the C tile of tiles[b * split] = alpha * sum_q
// partial[b * split + q] (q ascending) + beta C, inside the problem and, for lower
// problems, on or below the diagonal.  PULL: plus the children's update blocks
// (beta not used).  Four entries a thread, the partials of four chunks in
// flight: bound by the latency of its loads (a block per tile with sixteen entries
// a thread one after another took 10-38 us, more than the chunks it summed).
template <bool PULL>
__global__ __launch_bounds__(256) void split_reduce_kernel(const GemmProb* __restrict__ probs,
                                                           const GemmTile* __restrict__ tiles, Bases bases, int split,
                                                           const double* __restrict__ ws) {
  const GemmTile t = tiles[(int64_t)blockIdx.x * split];
  const GemmProb P = probs[t.prob];
  double* C = bases.p[P.c_base] + P.c_off;
  const int m0 = t.tm * 64, n0 = t.tn * 64;
  const bool diag_tile = P.lower && t.tm == t.tn;
  const int e0 = blockIdx.y * 1024 + threadIdx.x;
  const double* w = ws + (int64_t)blockIdx.x * split * 4096 + e0;
  double acc[4] = {0.0, 0.0, 0.0, 0.0}, old[4];
  const int m = m0 + (e0 & 63);
  bool in[4];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int n = n0 + (e0 >> 6) + 4 * u;
    in[u] = m < P.M && n < P.N && !(diag_tile && m < n);
    old[u] = !PULL && in[u] && P.beta != 0.0 ? C[m + (int64_t)n * P.ldc] : 0.0;
  }
  int q = 0;
  for (; q + 4 <= split; q += 4) {
    double v[4][4];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u) v[c][u] = w[(q + c) * 4096 + u * 256];
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int u = 0; u < 4; ++u) acc[u] += v[c][u];
  }
  for (; q < split; ++q)
#pragma unroll
    for (int u = 0; u < 4; ++u) acc[u] += w[q * 4096 + u * 256];
#pragma unroll
  for (int u = 0; u < 4; ++u) {
    const int n = n0 + (e0 >> 6) + 4 * u;
    if (!in[u]) continue;
    double* c = C + m + (int64_t)n * P.ldc;
    const double r = P.alpha * acc[u];
    if constexpr (PULL) {
      const Pull pq = bases.pulls[P.pull];
      const int i = P.pull_row + m, j = P.pull_row + n;
      *c = assembled(bases.p[kFront], r, pq, child_row(bases.inv, pq, 0, i), child_row(bases.inv, pq, 1, i),
                     child_row(bases.inv, pq, 0, j), child_row(bases.inv, pq, 1, j));
    } else {
      *c = P.beta == 0.0 ? r : r + P.beta * old[u];
    }
  }
}

// Large tiles: 128x64 at three waves per SIMD (64x128 where op(A) = A^T and
// op(B) = B^T: the operand with contiguous k takes the short edge, 67 against 59
// TFLOP/s at 4096^3), and 128x128 at two waves where k is contiguous in both
// operands (their 16-line loads want the larger tile: 64 against 50; elsewhere
// 128x64 leads 128x128, 65 against 61 NT and 67 against 63 NN).
template <bool TA, bool TB, bool VEC>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(TA && !TB ? 2 : 3, TA && !TB ? 2 : 3))) void
gemm128_kernel(const GemmProb* __restrict__ probs, const GemmTile* __restrict__ tiles, Bases bases) {
  gemm_reg_body<TA, TB, VEC, (TA && TB) ? 2 : 4, TA ? 4 : 2>(probs, tiles, bases);
}

// y = alpha op(A) x + beta y for N <= kGemvMaxN columns (solves with few
// right-hand sides).  Bandwidth-bound: A is read once, coalesced.
// A not transposed (M x K): block = 64 rows (lane = row), the four waves take
// quarters of K, partial sums combined in LDS in wave order.
// A transposed (K x M stored): one wave per output row m (a column of A),
// lanes stride over k, butterfly sum across the wave.
// loads each lane issues before their products in the GEMV's inner loop
constexpr int kGemvDepth = 16;
template <bool TA, int NW = 4>
__global__ __launch_bounds__(NW * 64) void gemv_kernel(const GemmProb* __restrict__ probs,
                                                       const GemmTile* __restrict__ tiles, Bases bases) {
  const GemmTile t = tiles[blockIdx.x];
  const GemmProb P = probs[t.prob];
  const double* __restrict__ A = bases.p[P.a_base] + P.a_off;
  const double* __restrict__ X = bases.p[P.b_base] + P.b_off;
  double* __restrict__ Y = bases.p[P.c_base] + P.c_off;
  const int N = P.N, K = P.K;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  double acc[kGemvMaxN];
#pragma unroll
  for (int c = 0; c < kGemvMaxN; ++c) acc[c] = 0.0;
  if constexpr (!TA) {
    __shared__ double red[NW][kGemvMaxN][64];
    const int m = t.tm * 64 + lane;
    const int q = (K + NW - 1) / NW, k0 = wave * q, k1 = min(K, k0 + q);
    if (m < P.M) {
      // batches of kGemvDepth loads issued before their products, so that
      // many columns' worth of A are in flight per lane; the sums still run
      // in ascending k
      const double* __restrict__ a = A + m + (int64_t)k0 * P.lda;
      int k = k0;
      for (; k + kGemvDepth <= k1; k += kGemvDepth, a += (int64_t)kGemvDepth * P.lda) {
        double av[kGemvDepth];
#pragma unroll
        for (int u = 0; u < kGemvDepth; ++u) av[u] = a[(int64_t)u * P.lda];
#pragma unroll
        for (int u = 0; u < kGemvDepth; ++u)
#pragma unroll
          for (int c = 0; c < kGemvMaxN; ++c)
            if (c < N) acc[c] += av[u] * X[k + u + (int64_t)c * P.ldb];
      }
      for (; k < k1; ++k, a += P.lda) {
        const double av = *a;
#pragma unroll
        for (int c = 0; c < kGemvMaxN; ++c)
          if (c < N) acc[c] += av * X[k + (int64_t)c * P.ldb];
      }
    }
#pragma unroll
    for (int c = 0; c < kGemvMaxN; ++c) red[wave][c][lane] = acc[c];
    __syncthreads();
    if (wave == 0 && m < P.M)
      for (int c = 0; c < N; ++c) {
        double v = red[0][c][lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) v += red[w][c][lane];
        double* y = Y + m + (int64_t)c * P.ldc;
        const double r = P.alpha * v;
        *y = (P.beta == 0.0) ? r : r + P.beta * (*y);
      }
  } else {
    const int m = t.tm * 4 + wave;
    if (m >= P.M) return;
    const double* a = A + (int64_t)m * P.lda;
#pragma unroll 8
    for (int k = lane; k < K; k += 64) {
      const double av = a[k];
#pragma unroll
      for (int c = 0; c < kGemvMaxN; ++c)
        if (c < N) acc[c] += av * X[k + (int64_t)c * P.ldb];
    }
#pragma unroll
    for (int c = 0; c < kGemvMaxN; ++c)
      for (int o = 32; o > 0; o >>= 1) acc[c] += __shfl_xor(acc[c], o, 64);
    if (lane == 0)
      for (int c = 0; c < N; ++c) {
        double* y = Y + m + (int64_t)c * P.ldc;
        const double r = P.alpha * acc[c];
        *y = (P.beta == 0.0) ? r : r + P.beta * (*y);
      }
  }
}

void launch_gemm(const GemmLaunch& g, const Bases& b, hipStream_t s, unsigned lds) {
  if (g.ntiles == 0) return;
  dim3 grid(g.ntiles), block(256);
  if (g.gemv) {
    if (g.ta)
      hipLaunchKernelGGL(gemv_kernel<true>, grid, block, 0, s, g.d_probs, g.d_tiles, b);
    else if (g.gemv_wide)
      hipLaunchKernelGGL((gemv_kernel<false, 16>), grid, dim3(1024), 0, s, g.d_probs, g.d_tiles, b);
    else
      hipLaunchKernelGGL(gemv_kernel<false>, grid, block, 0, s, g.d_probs, g.d_tiles, b);
    return;
  }
  // VEC matters only where k is contiguous in an operand
#define SPDE_GEMM_FORM(K, ...)                                        \
  do {                                                                \
    const bool vec = g.vec;                                           \
    if (!g.ta && g.tb)                                                \
      hipLaunchKernelGGL((K<false, true, true>), __VA_ARGS__);        \
    else if (!g.ta && vec)                                            \
      hipLaunchKernelGGL((K<false, false, true>), __VA_ARGS__);       \
    else if (!g.ta)                                                   \
      hipLaunchKernelGGL((K<false, false, false>), __VA_ARGS__);      \
    else if (!g.tb && vec)                                            \
      hipLaunchKernelGGL((K<true, false, true>), __VA_ARGS__);        \
    else if (!g.tb)                                                   \
      hipLaunchKernelGGL((K<true, false, false>), __VA_ARGS__);       \
    else if (vec)                                                     \
      hipLaunchKernelGGL((K<true, true, true>), __VA_ARGS__);         \
    else                                                              \
      hipLaunchKernelGGL((K<true, true, false>), __VA_ARGS__);        \
  } while (0)
  if (g.split > 1) {
    double* ws = b.ws + g.ws_off;
    SPDE_GEMM_FORM(gemm64_split_kernel, grid, block, 0, s, g.d_probs, g.d_tiles, b, g.split, ws);
    if (g.pull)
      hipLaunchKernelGGL(split_reduce_kernel<true>, dim3(g.ntiles / g.split, 4), block, 0, s, g.d_probs, g.d_tiles, b,
                         g.split, ws);
    else
      hipLaunchKernelGGL(split_reduce_kernel<false>, dim3(g.ntiles / g.split, 4), block, 0, s, g.d_probs, g.d_tiles, b,
                         g.split, ws);
    return;
  }
  if (g.pull) {
    if (g.tile == 128)
      hipLaunchKernelGGL(syrk_pull_kernel<4>, grid, block, lds, s, g.d_probs, g.d_tiles, b);
    else
      hipLaunchKernelGGL(syrk_pull_kernel<2>, grid, block, lds, s, g.d_probs, g.d_tiles, b);
    return;
  }
  if (g.tile == 128)
    SPDE_GEMM_FORM(gemm128_kernel, grid, block, lds, s, g.d_probs, g.d_tiles, b);
  else
    SPDE_GEMM_FORM(gemm64_kernel, grid, block, lds, s, g.d_probs, g.d_tiles, b);
#undef SPDE_GEMM_FORM
}

__global__ void fill_kernel(double* __restrict__ p, int64_t n, double v) {
  for (int64_t i = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

// Lane-layout probe of v_mfma_f64_16x16x4f64 (64 lanes, 4 outputs each).
// which=0: a = 1 on lanes 0..15, b = lane+1 on lanes 0..15;
// which=1: a = lane+1 on lanes 0..15, b = 1 on lanes 0..15.
__global__ __launch_bounds__(64) void mfma_probe_kernel(int which, double* __restrict__ out) {
  const int l = threadIdx.x;
  double a = 0.0, b = 0.0;
  if (l < 16) {
    a = which == 0 ? 1.0 : (double)(l + 1);
    b = which == 0 ? (double)(l + 1) : 1.0;
  }
  d4 acc = {0.0, 0.0, 0.0, 0.0};
  acc = __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, acc, 0, 0, 0);
  for (int v = 0; v < 4; ++v) out[4 * l + v] = acc[v];
}

void launch_fill(double* p, int64_t n, double v, hipStream_t s) {
  if (n <= 0) return;
  int64_t blocks = (n + 255) / 256;
  if (blocks > 65536) blocks = 65536;
  hipLaunchKernelGGL(fill_kernel, dim3((unsigned)blocks), dim3(256), 0, s, p, n, v);
}

}  // namespace spde

using namespace spde;

extern "C" int spde_debug_mfma_probe(int which, double* out, void* stream) {
  if (!out || which < 0 || which > 1) {
    set_error("spde_debug_mfma_probe: invalid argument");
    return SPDE_ERR_ARG;
  }
  hipLaunchKernelGGL(mfma_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, which, out);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

extern "C" int spde_debug_gemm(int ta, int tb, int M, int N, int K, double alpha, const double* A, int lda,
                               const double* B, int ldb, double beta, double* C, int ldc, int tile, void* stream) {
  if (M <= 0 || N <= 0 || K < 0 || !A || !B || !C || lda < (ta ? K : M) || ldb < (tb ? N : K) || ldc < M ||
      (tile != 64 && tile != 128)) {
    set_error("spde_debug_gemm: invalid argument");
    return SPDE_ERR_ARG;
  }
  GemmProb P{};  // every field zero (kmode 0: no triangular operand)
  P.a_off = P.b_off = P.c_off = 0;
  P.lda = lda;
  P.ldb = ldb;
  P.ldc = ldc;
  P.M = M;
  P.N = N;
  P.K = K;
  P.a_base = 0;
  P.b_base = 1;
  P.c_base = 2;
  P.lower = 0;
  P.alpha = alpha;
  P.beta = beta;
  std::vector<GemmTile> tiles;
  GemmLaunch g;
  g.tile = tile;
  g.ta = ta != 0;
  g.tb = tb != 0;
  g.vec = !((uintptr_t)A & 15) && !((uintptr_t)B & 15) && !(lda & 1) && !(ldb & 1);
  for (int a = 0; a < (M + g.tile_m() - 1) / g.tile_m(); ++a)
    for (int b = 0; b < (N + g.tile_n() - 1) / g.tile_n(); ++b) tiles.push_back({0, a, b, 0});
  g.ntiles = (int)tiles.size();
  SPDE_HIP(hipMalloc((void**)&g.d_probs, sizeof(GemmProb)));
  SPDE_HIP(hipMalloc((void**)&g.d_tiles, sizeof(GemmTile) * tiles.size()));
  SPDE_HIP(hipMemcpy(g.d_probs, &P, sizeof(GemmProb), hipMemcpyHostToDevice));
  SPDE_HIP(hipMemcpy(g.d_tiles, tiles.data(), sizeof(GemmTile) * tiles.size(), hipMemcpyHostToDevice));
  Bases bs;
  for (int q = 0; q < kNumBases; ++q) bs.p[q] = nullptr;
  bs.p[0] = const_cast<double*>(A);
  bs.p[1] = const_cast<double*>(B);
  bs.p[2] = C;
  bs.ws = nullptr;
  bs.pulls = nullptr;
  bs.inv = nullptr;
  launch_gemm(g, bs, (hipStream_t)stream, 0);
  SPDE_HIP(hipStreamSynchronize((hipStream_t)stream));
  hipFree(g.d_probs);
  hipFree(g.d_tiles);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}
