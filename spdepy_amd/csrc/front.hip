// Dense partial factorisation of a level's fronts: the own columns of every
// front in one launch.  A task list is worked through by resident blocks that
// take tickets in order; 64x64 tiles of L are published by flags.
#include <hip/hip_runtime.h>

#include "internal.hpp"
#include "wait.hpp"

namespace spde {

typedef double d4 __attribute__((ext_vector_type(4)));

struct Piv4 {
  double i0, i1, i2, i3, l10, l20, l30, l21, l31, l32, d0, d1, d2, d3;
};

// Keeps an updated register value where it is computed: without it the
// compiler defers the rank-4 updates of later columns to their first use and
// keeps every step's operands live (hundreds of registers, spilled).
__device__ inline void pin(double& v) { asm volatile("" : "+v"(v)); }

// 1/sqrt(x) for x > 0 (hardware estimate refined twice), x for the factor.
__device__ inline double pivot_rsq(double x, bool& bad) {
  if (!(x > 0.0)) {
    bad = true;
    x = 1.0;
  }
  double y = __builtin_amdgcn_rsq(x);
  const double hx = 0.5 * x;
  y = y * (1.5 - hx * y * y);
  y = y * (1.5 - hx * y * y);
  return y;
}

// 4x4 Cholesky factor of D(i, j) = D[i * P + j] (lower part read).
template <int P>
__device__ inline void chol4(const double* D, Piv4& c, int& badcol) {
  bool b0 = false, b1 = false, b2 = false, b3 = false;
  double x = D[0];
  c.i0 = pivot_rsq(x, b0);
  c.d0 = b0 ? 1.0 : x * c.i0;
  c.l10 = D[P] * c.i0;
  c.l20 = D[2 * P] * c.i0;
  c.l30 = D[3 * P] * c.i0;
  x = D[P + 1] - c.l10 * c.l10;
  c.i1 = pivot_rsq(x, b1);
  c.d1 = b1 ? 1.0 : x * c.i1;
  c.l21 = (D[2 * P + 1] - c.l20 * c.l10) * c.i1;
  c.l31 = (D[3 * P + 1] - c.l30 * c.l10) * c.i1;
  x = D[2 * P + 2] - c.l20 * c.l20 - c.l21 * c.l21;
  c.i2 = pivot_rsq(x, b2);
  c.d2 = b2 ? 1.0 : x * c.i2;
  c.l32 = (D[3 * P + 2] - c.l30 * c.l20 - c.l31 * c.l21) * c.i2;
  x = D[3 * P + 3] - c.l30 * c.l30 - c.l31 * c.l31 - c.l32 * c.l32;
  c.i3 = pivot_rsq(x, b3);
  c.d3 = b3 ? 1.0 : x * c.i3;
  badcol = b0 ? 0 : (b1 ? 1 : (b2 ? 2 : (b3 ? 3 : -1)));
}

constexpr int kYP = 66;  // pitch of Y (16-byte aligned rows)
constexpr int kWP = 65;  // pitch of W and X
struct DiagLds {
  double pub[2][64 * 4];  // pivot columns, row-major [r][0..3]
  double Y[64 * kYP];     // diagonal tile on entry, then the finished L (zeros right of the diagonal)
  double Wl[64 * kWP];    // X of the tile left of the diagonal, then W = L^-1
  double Xs[32 * 33];
  double idg[64];         // 1 / L(k, k)
  int ticket;
};

// Cholesky factor and inverse of one 64x64 diagonal block by a 256-thread
// block.  Thread (r, g) (lane r of
// wave g) keeps row r, columns c = 4q + g (q = 0..15), in registers, so each
// step of four pivot columns j0..j0+3 has exactly one of them in every
// thread.  Step: the threads publish their pivot-column entry (one LDS write
// each, double buffered), every thread forms the 4x4 pivot block's factor
// itself, finishes its row's four entries, writes its own one to the L copy
// Y in LDS, and the rank-4 update of its columns right of the pivot block,
// with the finished rows read back from Y (broadcast reads, no
// recomputation), follows in the next step.  Entries right of the diagonal are
// never read, so the update runs unconditionally over them.  W = L^-1 is
// then built by recursive blocking in LDS (below).  Pivots use v_rsq_f64 with
// two Newton steps (relative error below 2^-52) instead of a square root and
// a division.  Blocks narrower than 64 are padded with the identity.  A
// non-positive pivot is recorded in *status as (global elimination column
// + 1) and replaced by 1 so the sweep completes.  a: the block's entries; Fb:
// where L goes; W is left in S.Wl.
__device__ __forceinline__ void diag_factor(DiagLds& S, double (&a)[16], int kb, double* Fb, int64_t ld, int colbase,
                                            int* __restrict__ status, int tid) {
  double(&pub)[2][64 * 4] = S.pub;
  double(&Y)[64 * kYP] = S.Y;
  double(&Wl)[64 * kWP] = S.Wl;
  double(&Xs)[32 * 33] = S.Xs;
  double(&idg)[64] = S.idg;
  constexpr int YP = kYP, WP = kWP;
  const int r = tid & 63, g = tid >> 6;
  // The rank-4 update of step s - 1 is applied to the next pivot column
  // first and to the later columns during step s, beside its serial 4x4
  // factor and row solve (same operations in the same order per entry).
  double p0 = 0.0, p1 = 0.0, p2 = 0.0, p3 = 0.0;
#pragma unroll
  for (int s = 0; s < 16; ++s) {
    const int j0 = 4 * s, buf = s & 1, jp = j0 - 4;
    if (s > 0) {
      const double* yc = &Y[(4 * s + g) * YP + jp];
      a[s] -= p0 * yc[0] + p1 * yc[1] + p2 * yc[2] + p3 * yc[3];
    }
    pub[buf][4 * r + g] = a[s];
    __syncthreads();
    Piv4 c;
    int bad;
    chol4<4>(&pub[buf][4 * j0], c, bad);
    if (bad >= 0 && tid == 0 && j0 + bad < kb) atomicCAS(status, 0, colbase + j0 + bad + 1);
    if (s > 0) {
#pragma unroll
      for (int q = s + 1; q < 16; ++q) {
        const double* yc = &Y[(4 * q + g) * YP + jp];
        a[q] -= p0 * yc[0] + p1 * yc[1] + p2 * yc[2] + p3 * yc[3];
      }
    }
    // row r's four entries; on the pivot rows this yields the factor's
    // entries left of and on the diagonal, the rest (and all of the rows
    // above) are cleared
    const double* pr = &pub[buf][4 * r];
    double y0 = pr[0] * c.i0;
    double y1 = (pr[1] - y0 * c.l10) * c.i1;
    double y2 = (pr[2] - y0 * c.l20 - y1 * c.l21) * c.i2;
    double y3 = (pr[3] - y0 * c.l30 - y1 * c.l31 - y2 * c.l32) * c.i3;
    y0 = (r >= j0) ? y0 : 0.0;
    y1 = (r >= j0 + 1) ? y1 : 0.0;
    y2 = (r >= j0 + 2) ? y2 : 0.0;
    y3 = (r >= j0 + 3) ? y3 : 0.0;
    const double mine = (g == 0) ? y0 : (g == 1 ? y1 : (g == 2 ? y2 : y3));
    a[s] = mine;
    Y[r * YP + j0 + g] = mine;
    if (tid < 4) idg[j0 + tid] = (tid == 0) ? c.i0 : (tid == 1 ? c.i1 : (tid == 2 ? c.i2 : c.i3));
    __syncthreads();
    p0 = y0;
    p1 = y1;
    p2 = y2;
    p3 = y3;
#pragma unroll
    for (int q = s + 1; q < 16; ++q) pin(a[q]);
  }
  if (r < kb) {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int c = 4 * q + g;
      if (c < kb && c <= r) Fb[r + (int64_t)c * ld] = a[q];
    }
  }
  // W = L^-1 by recursive blocking: the four 16x16 diagonal blocks are
  // inverted by column-oriented forward substitution (wave g, lane j < 16:
  // column j of block g), then W21 = -W22 (L21 W11) for the two 32x32 and
  // the 64x64 block rows, the products spread over the block.  Wl is
  // row-major with zeros above the diagonal; blocks beyond kb hold the
  // identity padding of L, so W is the identity there too.
  for (int e = tid; e < 64 * WP; e += 256) Wl[e] = 0.0;
  __syncthreads();
  if (r < 16) {
    const int o = 16 * g, j = r;
    double x[16];
#pragma unroll
    for (int i = 0; i < 16; ++i) x[i] = (i == j) ? 1.0 : 0.0;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      x[kk] *= idg[o + kk];
#pragma unroll
      for (int i = kk + 1; i < 16; ++i) x[i] -= Y[(o + i) * YP + o + kk] * x[kk];
    }
#pragma unroll
    for (int i = 0; i < 16; ++i) Wl[(o + i) * WP + o + j] = x[i];
  }
  __syncthreads();
  {
    // 32 level, pair P = rows/cols 32P .. 32P + 31: X = L(o+16.., o..) W00,
    // W10 = -W11 X; thread: pair tid >> 7, row i, columns j0, j0 + 1
    const int P = tid >> 7, t = tid & 127, i = t >> 3, j0 = (t & 7) * 2, o = 32 * P;
    double x0 = 0.0, x1 = 0.0;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const double l = Y[(o + 16 + i) * YP + o + kk];
      x0 += l * Wl[(o + kk) * WP + o + j0];
      x1 += l * Wl[(o + kk) * WP + o + j0 + 1];
    }
    Xs[(P * 16 + i) * 33 + j0] = x0;
    Xs[(P * 16 + i) * 33 + j0 + 1] = x1;
    __syncthreads();
    double w0 = 0.0, w1 = 0.0;
#pragma unroll
    for (int kk = 0; kk < 16; ++kk) {
      const double v = Wl[(o + 16 + i) * WP + o + 16 + kk];
      w0 += v * Xs[(P * 16 + kk) * 33 + j0];
      w1 += v * Xs[(P * 16 + kk) * 33 + j0 + 1];
    }
    Wl[(o + 16 + i) * WP + o + j0] = -w0;
    Wl[(o + 16 + i) * WP + o + j0 + 1] = -w1;
  }
  __syncthreads();
  {
    // 64 level: X = L(32.., 0..31) W_aa, W_ba = -W_bb X; thread: column
    // j = tid & 31, rows i0 + 8u
    const int j = tid & 31, i0 = tid >> 5;
    double x[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < 32; ++kk) {
      const double wv = Wl[kk * WP + j];
#pragma unroll
      for (int u = 0; u < 4; ++u) x[u] += Y[(32 + i0 + 8 * u) * YP + kk] * wv;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) Xs[(i0 + 8 * u) * 33 + j] = x[u];
    __syncthreads();
    double w[4] = {0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int kk = 0; kk < 32; ++kk) {
      const double xv = Xs[kk * 33 + j];
#pragma unroll
      for (int u = 0; u < 4; ++u) w[u] += Wl[(32 + i0 + 8 * u) * WP + 32 + kk] * xv;
    }
#pragma unroll
    for (int u = 0; u < 4; ++u) Wl[(32 + i0 + 8 * u) * WP + j] = -w[u];
  }
  __syncthreads();
}

// ------------------------------------------------------- tile exchange
// Tiles are exchanged inside one launch between blocks on different XCDs,
// whose L2 caches are not coherent.  The writer stores with agent scope
// (written through), waits for the stores and then adds to the tile's counter;
// the reader polls the counter with agent scope and then reads the tile
// through its caches.  No cache can hold an old copy: a tile's lines belong to it
// alone (FrontLay), before it is published only its owner reads them, and a
// launch starts with clean caches.
__device__ __forceinline__ void put(double* p, double v) {
  __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
// Element at a wave-uniform base plus a lane's byte offset (one 32-bit
// register per lane offset instead of a 64-bit address per element).
__device__ __forceinline__ double* at(const double* base, uint32_t off) { return (double*)((char*)base + off); }
__device__ __forceinline__ void publish(int* flag, int add) {
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if ((threadIdx.x & 63) == 0) __hip_atomic_fetch_add(flag, add, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ int peek(const int* p) {
  return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
constexpr int kTileDone = 4;
// The tickets make every wait end: a task waits only for tasks with lower
// tickets (checked when the plan is made), which blocks already run.  A wait that
// passes kSpinLimit polls all the same raises the stop flag and sets *status to
// kStalled, every later wait gives up at once, and the factorisation reports an
// error.
struct Waiter : WaitBudget {
  int* stop;
  int* status;
  __device__ __forceinline__ Waiter(int* stop_, int* status_) : stop(stop_), status(status_) {}
  // false: keep waiting
  __device__ __forceinline__ bool over() {
    if (spent()) {
      if ((threadIdx.x & 63) == 0) {
        __hip_atomic_store(stop, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        __hip_atomic_store(status, kStalled, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      }
      return gave_up = true;
    }
    if ((spins & 1023) == 0 && peek(stop)) return gave_up = true;
    __builtin_amdgcn_s_sleep(1);
    return false;
  }
};
__device__ __forceinline__ void wait_tile(const int* flag, Waiter& w) {
  w.begin();
  while (peek(flag) < kTileDone)
    if (w.gave_up || w.over()) break;
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  asm volatile("" ::: "memory");
}
// Number of columns k0, k0 + 1, .. < k1 (at most 32) whose tiles in rows ia
// and ib are all published; waits for the first.
__device__ __forceinline__ int wait_columns(const int* fl, int R, int k0, int k1, int ia, int ib, Waiter& w) {
  const int lane = threadIdx.x & 63;
  const int k = k0 + (lane & 31), row = lane < 32 ? ia : ib;
  int n;
  w.begin();
  for (;;) {
    const bool ok = k < k1 && peek(fl + (int64_t)k * R + row) >= kTileDone;
    const unsigned long long m = __ballot(ok);
    const unsigned both = (unsigned)m & (unsigned)(m >> 32);
    n = both == 0xffffffffu ? 32 : __builtin_ctz(~both);
    if (n > 0) break;
    if (w.gave_up || w.over()) {
      n = 1;
      break;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
  asm volatile("" ::: "memory");
  return __builtin_amdgcn_readfirstlane(n);
}

// acc[x][y] += (rows of fragment y) (rows of fragment x)^T over the columns
// [64 k0, 64 k1) of one front: base at the front, oa / ob the byte offsets of the
// lanes' rows (plus 4 lk columns), in 16-deep slabs as the register GEMM.
template <int TM, int TN>
__device__ __forceinline__ void strip_product(d4 (&acc)[TN][TM], const uint32_t (&oa)[TM], const uint32_t (&ob)[TN],
                                              const char* base, int64_t ldb, int k0, int k1) {
  const char* p = base + (int64_t)k0 * 64 * ldb;
  double fa[TM][4], fb[TN][4];
  auto load = [&](int h) {
#pragma unroll
    for (int u = 2 * h; u < 2 * h + 2; ++u) {
      const char* q = p + u * ldb;
#pragma unroll
      for (int y = 0; y < TM; ++y) fa[y][u] = *(const double*)(q + oa[y]);
#pragma unroll
      for (int x = 0; x < TN; ++x) fb[x][u] = *(const double*)(q + ob[x]);
    }
  };
  auto mul = [&](int h) {
#pragma unroll
    for (int u = 2 * h; u < 2 * h + 2; ++u)
#pragma unroll
      for (int x = 0; x < TN; ++x)
#pragma unroll
        for (int y = 0; y < TM; ++y)
          acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(fb[x][u], fa[y][u], acc[x][y], 0, 0, 0);
  };
  load(0);
  load(1);
  const int nk = (k1 - k0) * 4;
  for (int kt = 1; kt < nk; ++kt) {
    p += 16 * ldb;
    mul(0);
    __builtin_amdgcn_sched_barrier(0);
    load(0);
    __builtin_amdgcn_sched_barrier(0);
    mul(1);
    __builtin_amdgcn_sched_barrier(0);
    load(1);
    __builtin_amdgcn_sched_barrier(0);
  }
  mul(0);
  mul(1);
}

// X = -acc W^T for TM fragments of 16 rows and 64 columns.  The accumulator
// layout (lane (lr, lk), element v: row lr, column lk + 4v) is the fragment layout
// of the next product with k = 16 g + lk + 4 v, so acc is its operand as it is.
// W (lower triangular, column-major at zoff) is read in the same order.
template <int TM, class Out>
__device__ __forceinline__ void times_wt(const d4 (&acc)[4][TM], const double* W, int64_t zld, int lr, int lk,
                                         Out&& out) {
  const uint32_t ow = (uint32_t)lr * 8u + (uint32_t)lk * (uint32_t)zld * 8u;
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    d4 X[TM];
#pragma unroll
    for (int y = 0; y < TM; ++y) X[y] = d4{0.0, 0.0, 0.0, 0.0};
    double w[4][4];
#pragma unroll
    for (int g = 0; g <= x; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v) w[g][v] = *at(W + 16 * x + (16 * g + 4 * v) * zld, ow);
#pragma unroll
    for (int g = 0; g <= x; ++g)
#pragma unroll
      for (int v = 0; v < 4; ++v)
#pragma unroll
        for (int y = 0; y < TM; ++y)
          X[y] = __builtin_amdgcn_mfma_f64_16x16x4f64(w[g][v], acc[g][y][v], X[y], 0, 0, 0);
#pragma unroll
    for (int y = 0; y < TM; ++y) out(x, y, -X[y]);
  }
}

// Tiles (i, j) and (i + 1, j) below the diagonal block j: S - sum_k L_ik L_jk^T,
// then times W_j^T.  Each wave has a strip of 32 rows and works alone.
__device__ __forceinline__ void panel_task(const FrontDesc& f, int i, int j, double* F, const double* Z, int* fl,
                                           Waiter& wt, int tid) {
  const int lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int it = i + (wave >> 1);
  if (it >= f.R) return;
  const int64_t ld = f.ld, ldb = ld * 8;
  double* Ff = F + f.foff;
  const int r0 = 64 * it + 32 * (wave & 1);
  uint32_t oa[2], ob[4], oc[2];
  const uint32_t c1 = (uint32_t)lk * (uint32_t)ldb;
  bool in[2];
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int row = r0 + 16 * y + lr;
    in[y] = row < f.nrows;
    oc[y] = (uint32_t)min(row, f.nrows - 1) * 8u + c1;  // column lk
    oa[y] = oc[y] + 3u * c1;                            // column 4 lk
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) ob[x] = (uint32_t)(64 * j + 16 * x + lr) * 8u + (uint32_t)lk * 4u * (uint32_t)ldb;
  d4 acc[4][2];
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
      acc[x][y] = d4{0.0, 0.0, 0.0, 0.0};
  for (int k = 0; k < j;) {
    const int n = wait_columns(fl, f.R, k, j, it, j, wt);
    strip_product<2, 4>(acc, oa, ob, (const char*)Ff, ldb, k, k + n);
    k += n;
  }
  // S is subtracted from the finished sum (as the trailing update of a whole
  // column range would be), not accumulated upon
#pragma unroll
  for (int x = 0; x < 4; ++x)
#pragma unroll
    for (int y = 0; y < 2; ++y)
#pragma unroll
      for (int v = 0; v < 4; ++v) acc[x][y][v] -= *at(Ff + (64 * j + 16 * x + 4 * v) * ld, oc[y]);
  wait_tile(fl + (int64_t)j * f.R + j, wt);
  times_wt<2>(acc, Z + f.zoff + (int64_t)64 * j * (f.pp + 1), f.pp, lr, lk, [&](int x, int y, const d4& X) {
    if (in[y])
#pragma unroll
      for (int v = 0; v < 4; ++v) put(at(Ff + (64 * j + 16 * x + 4 * v) * ld, oc[y]), X[v]);
  });
  publish(fl + (int64_t)j * f.R + it, 2);
}

// Diagonal block j, and the tile (j, j - 1) left of it, whose solve the block
// does itself: one hand-over per 64 columns on the front's critical path.
// Each wave has 16 rows until the block is gathered in LDS.
__device__ __forceinline__ void diag_task(const FrontDesc& f, int j, double* F, double* Z, int* fl, int* status,
                                          DiagLds& S, Waiter& wt, int tid) {
  const int lane = tid & 63, wave = tid >> 6;
  const int lr = lane & 15, lk = lane >> 4;
  const int64_t ld = f.ld, ldb = ld * 8;
  double* Ff = F + f.foff;
  const int kb = min(64, f.p - 64 * j);
  double* Fb = Ff + 64 * j + (int64_t)64 * j * ld;
  double a[16];
  if (j > 0) {
    const int row = 64 * j + 16 * wave + lr;
    d4 acc[8][1];  // 0..3: columns of tile j - 1; 4..7: of tile j
    const uint32_t ck = (uint32_t)lk * 4u * (uint32_t)ldb, oc = (uint32_t)row * 8u + (uint32_t)lk * (uint32_t)ldb;
    uint32_t oa[1] = {(uint32_t)row * 8u + ck}, ob[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) {
      ob[x] = (uint32_t)(64 * (j - 1) + 16 * x + lr) * 8u + ck;
      acc[x][0] = d4{0.0, 0.0, 0.0, 0.0};
    }
    for (int k = 0; k < j - 1;) {
      const int n = wait_columns(fl, f.R, k, j - 1, j, j - 1, wt);
      strip_product<1, 8>(acc, oa, ob, (const char*)Ff, ldb, k, k + n);
      k += n;
    }
    // the tile left of the diagonal now, the diagonal tile after its last column
    double sjj[4][4];
#pragma unroll
    for (int x = 0; x < 4; ++x)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        acc[x][0][v] -= *at(Ff + (64 * (j - 1) + 16 * x + 4 * v) * ld, oc);
        sjj[x][v] = *at(Ff + (64 * j + 16 * x + 4 * v) * ld, oc);
      }
    wait_tile(fl + (int64_t)(j - 1) * f.R + j - 1, wt);
    d4 left[4][1], X[4][1];
#pragma unroll
    for (int x = 0; x < 4; ++x) left[x][0] = acc[x][0];
    times_wt<1>(left, Z + f.zoff + (int64_t)64 * (j - 1) * (f.pp + 1), f.pp, lr, lk, [&](int x, int, const d4& q) {
      X[x][0] = q;
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        put(at(Ff + (64 * (j - 1) + 16 * x + 4 * v) * ld, oc), q[v]);
        S.Wl[(16 * wave + lr) * kWP + 16 * x + lk + 4 * v] = q[v];
      }
    });
    __syncthreads();
    // S_jj - X X^T on and below the diagonal's 16-column groups
#pragma unroll
    for (int x = 0; x < 4; ++x)
      if (x <= wave) {
        d4 c = acc[4 + x][0];
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int v = 0; v < 4; ++v)
            c = __builtin_amdgcn_mfma_f64_16x16x4f64(S.Wl[(16 * x + lr) * kWP + 16 * g + lk + 4 * v], X[g][0][v], c, 0,
                                                     0, 0);
#pragma unroll
        for (int v = 0; v < 4; ++v) S.Y[(16 * wave + lr) * kYP + 16 * x + lk + 4 * v] = sjj[x][v] - c[v];
      }
    publish(fl + (int64_t)(j - 1) * f.R + j, 1);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int r = lane, c = 4 * q + wave;
      a[q] = (r < kb && c < kb) ? (c <= r ? S.Y[r * kYP + c] : 0.0) : (r == c ? 1.0 : 0.0);
    }
  } else {
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      const int r = lane, c = 4 * q + wave;
      a[q] = (r < kb && c < kb) ? (c <= r ? Fb[r + (int64_t)c * ld] : 0.0) : (r == c ? 1.0 : 0.0);
    }
  }
  diag_factor(S, a, kb, Fb, ld, f.colbase + 64 * j, status, tid);
  double* Zb = Z + f.zoff + (int64_t)64 * j * (f.pp + 1);
#pragma unroll
  for (int q = 0; q < 16; ++q) {
    const int c = 4 * q + wave;
    if (lane < kb && c < kb) put(at(Zb + (int64_t)c * f.pp, lane * 8u), S.Wl[lane * kWP + c]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  __syncthreads();
  if (tid < 64) publish(fl + (int64_t)j * f.R + j, kTileDone);
}

// One level.  Left-looking by 64-column blocks: a task keeps its tiles in
// registers over all earlier columns, waiting for each as it is published, and
// writes them once, so a front's chain (diagonal block, next tile, next
// diagonal block) runs ahead while the rest of the level fills the chip.
// 80 KB of LDS: two blocks per CU.
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) void front_factor_kernel(
    const FrontDesc* __restrict__ fronts, const FrontTask* __restrict__ tasks, int ntasks, double* F, double* Z,
    int* flags, int* ticket, int* stop, int* status) {
  __shared__ DiagLds S;
  Waiter wt{stop, status};
  for (;;) {
    // opaque here: the tasks' lane addresses are formed per task, not kept in
    // (spilled) registers across the ticket loop
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    if (threadIdx.x == 0) S.ticket = __hip_atomic_fetch_add(ticket, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    __syncthreads();
    const int t = __builtin_amdgcn_readfirstlane(S.ticket);
    if (t >= ntasks) return;
    const FrontTask T = tasks[t];
    const FrontDesc f = fronts[T.front];
    if (T.i == T.j)
      diag_task(f, T.j, F, Z, flags + f.flag0, status, S, wt, tid);
    else
      panel_task(f, T.i, T.j, F, Z, flags + f.flag0, wt, tid);
    __syncthreads();
  }
}

__global__ __launch_bounds__(256) void clear_flags_kernel(int* p, int n) {
  for (int i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) p[i] = 0;
}

void launch_front_factor(const FrontDesc* fronts, const FrontTask* tasks, int ntasks, double* F, double* Z, int* flags,
                         int* ticket, int* stop, int* status, hipStream_t s) {
  if (ntasks <= 0) return;
  hipLaunchKernelGGL(front_factor_kernel, dim3(ntasks < 512 ? ntasks : 512), dim3(256), 0, s, fronts, tasks, ntasks, F,
                     Z, flags, ticket, stop, status);
}
void launch_clear_flags(int* p, int n, hipStream_t s) {
  hipLaunchKernelGGL(clear_flags_kernel, dim3((n + 4095) / 4096), dim3(256), 0, s, p, n);
}

}  // namespace spde
