// Plan construction (device arenas, launch schedules) and the numeric
// multifrontal Cholesky, log-determinant, triangular solves and Takahashi
// selected inverse.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <functional>
#include <stdexcept>

#include "internal.hpp"

namespace spde {

void launch_gemm(const GemmLaunch& g, const Bases& b, hipStream_t s, unsigned lds = 0);
void launch_own_assemble(const NodeDev* nodes, const int4* tiles, int ntiles, const Pull* pulls, const int32_t* inv,
                         double* F, hipStream_t s);
void launch_front_factor(const FrontDesc* fronts, const FrontTask* tasks, int ntasks, double* F, double* Z, int* flags,
                         int* ticket, int* stop, int* status, hipStream_t s);
void launch_clear_flags(int* p, int n, hipStream_t s);
void launch_fill(double* p, int64_t n, double v, hipStream_t s);
void launch_scatter(const double* q, const int64_t* map, int64_t nnz, double* F, hipStream_t s);
void launch_diag_add(const double* add, const int64_t* diag, const int64_t* map, int64_t n, double* F, hipStream_t s);
int logdet_parts(int64_t n);
void launch_logdet(const int64_t* diag, const int64_t* map, int64_t n, const double* F, double* partial, double* out,
                   hipStream_t s);
void launch_permute_in(const double* B, int64_t ldb, const int32_t* perm, int64_t n, int nrhs, double* xy,
                       hipStream_t s);
void launch_permute_out(const double* xy, const int32_t* perm, int64_t n, int nrhs, double* B, int64_t ldb,
                        hipStream_t s);
void launch_fwd_gather(const int32_t* lvl_nodes, int nn, const NodeDev* nodes, const int32_t* children,
                       const int32_t* relpos, const double* xy, int64_t n, int nrhs, double* vec, hipStream_t s);
void launch_bwd_gather(const int32_t* lvl_nodes, int nn, const NodeDev* nodes, const int32_t* bnd, const double* xy,
                       int64_t n, int nrhs, double* vec, hipStream_t s);
void launch_sigma_gather(const int32_t* lvl_nodes, const NodeDev* nodes, const int32_t* relpos, double* S,
                         const int4* tiles, int ntiles, hipStream_t s);
void launch_gather_pattern(const double* S, const int64_t* mapsym, int64_t nnz, double* out, hipStream_t s);
void launch_zero_lower(const NodeDev* nodes, const int4* tiles, int ntiles, double* F, hipStream_t s);
void loglik_release(spde_plan* pl);  // loglik.hip

static thread_local std::string g_err;
void set_error(const std::string& m) { g_err = m; }

// Clears a factorisation's status word (a kernel rather than a memset node,
// so that a captured factorisation replays correctly).
__global__ void clear_status_kernel(int* status) {
  if (threadIdx.x == 0) status[threadIdx.x] = 0;
}

// Device layout of the fronts and Z blocks (FrontLay).
void build_layout(spde_plan* pl) {
  const Symbolic& sym = pl->sym;
  pl->lay.resize(sym.nodes.size());
  int64_t foff = 0, zoff = 0;
  for (size_t q = 0; q < sym.nodes.size(); ++q) {
    const Node& nd = sym.nodes[q];
    FrontLay& f = pl->lay[q];
    f.pp = (nd.p + kFrontPad - 1) / kFrontPad * kFrontPad;
    const int nf = f.pp + (int)nd.B.size();
    f.ld = (nf + 15) / 16 * 16;
    f.foff = foff;
    f.zoff = zoff;
    foff += (int64_t)f.ld * nf;
    zoff += (int64_t)f.pp * f.pp;
  }
  pl->lay_front = foff;
  pl->lay_z = zoff;
}

// Scatter map of the device layout from the compact one (an entry's column is its
// column variable's place in the node: no division per entry).
std::vector<int64_t> layout_map(const spde_plan* pl) {
  const Symbolic& sym = pl->sym;
  const Structure& st = pl->st;
  struct Place {
    int64_t from, to;  // of the node's front in either layout
    int32_t start, p, n, ld, pad;
  };
  std::vector<Place> place(sym.nodes.size());
  for (size_t q = 0; q < place.size(); ++q) {
    const Node& nd = sym.nodes[q];
    const FrontLay& f = pl->lay[q];
    place[q] = {nd.foff, f.foff, nd.start, nd.p, nd.n(), f.ld, f.pp - nd.p};
  }
  std::vector<int64_t> map(pl->map.size());
  for (size_t e = 0; e < map.size(); ++e) {
    if (pl->map[e] < 0) {
      map[e] = -1;
      continue;
    }
    const int pc = sym.iperm[st.indices[e]];
    const Place& f = place[sym.col_node[pc]];
    const int64_t col = pc - f.start, row = pl->map[e] - f.from - col * f.n;
    map[e] = f.to + (row < f.p ? row : row + f.pad) + col * f.ld;
  }
  return map;
}

// Device-side per-level index tables that are not part of LevelPlan.
struct LevelDev {
  int32_t* d_nodes = nullptr;
  int nn = 0;
  int4* d_gtiles = nullptr;
  int ngtiles = 0;
};

}  // namespace spde

using namespace spde;

namespace {

struct PlanExtra {            // kept beside the plan (not in the public struct)
  std::vector<LevelDev> lvl;
  int32_t* d_children = nullptr;
  int4* d_ztiles = nullptr;    // lower 64x64 tiles of every front (node, ti, tj)
  int nztiles = 0;
  // selected inverse: second stream for the products that need only the
  // factor, and its events (created at the first selected inverse)
  hipStream_t pre = nullptr;
  hipEvent_t ev_start = nullptr;
  std::vector<hipEvent_t> ev_pre;
};

PlanExtra* extra(spde_plan* p) { return static_cast<PlanExtra*>(p->extra); }

thread_local bool g_host_only_build = false;  // plan descriptors built for inspection only

template <class T>
int upload(T** dst, const std::vector<T>& src) {
  *dst = nullptr;
  if (src.empty() || g_host_only_build) return SPDE_OK;
  SPDE_HIP(hipMalloc((void**)dst, src.size() * sizeof(T)));
  SPDE_HIP(hipMemcpy(*dst, src.data(), src.size() * sizeof(T), hipMemcpyHostToDevice));
  return SPDE_OK;
}

// Arena sizes (doubles) per operand base, for the host-side bounds check.
struct ArenaSizes {
  int64_t sz[kNumBases];
};

bool operand_ok(int64_t off, int64_t ld, int64_t rows, int64_t cols, int64_t size) {
  if (rows <= 0 || cols <= 0) return true;
  if (off < 0 || ld < rows) return false;
  return off + (rows - 1) + (cols - 1) * ld < size;
}

// A lane's offsets inside a tile (register-fed products: tile rows or columns with
// contiguous k, else up to 12 k columns) must fit 32 bits.
bool lanes_ok(const GemmLaunch& g, const GemmProb& P) {
  if (g.gemv || (g.ta && !g.tb && g.tile == 64)) return true;  // 64-bit offsets
  auto span = [](bool kc, int64_t edge, int64_t rows, int64_t ld) {
    const int64_t last = std::max<int64_t>(std::min(edge, rows) - 1, 0);
    return kc ? last * ld * 8 + 96 : last * 8 + 12 * ld * 8;
  };
  const int64_t most = (int64_t)UINT32_MAX;
  return span(g.ta, g.tile_m(), P.M, P.lda) <= most && span(!g.tb, g.tile_n(), P.N, P.ldb) <= most;
}

// Every problem of a launch must touch only its operands' arenas.
int validate(const GemmLaunch& g, const ArenaSizes& a, const char* what) {
  for (const GemmProb& P : g.h_probs) {
    const int64_t ar = g.ta ? P.K : P.M, ac = g.ta ? P.M : P.K;
    const int64_t br = g.tb ? P.N : P.K, bc = g.tb ? P.K : P.N;
    const bool ok = operand_ok(P.a_off, P.lda, ar, ac, a.sz[P.a_base]) &&
                    operand_ok(P.b_off, P.ldb, br, bc, a.sz[P.b_base]) &&
                    operand_ok(P.c_off, P.ldc, P.M, P.N, a.sz[P.c_base]) && lanes_ok(g, P);
    if (!ok) {
      set_error(std::string("launch plan out of bounds in ") + what);
      return SPDE_ERR_STATE;
    }
  }
  for (const GemmTile& t : g.h_tiles)
    if (t.prob < 0 || t.prob >= (int)g.h_probs.size()) {
      set_error(std::string("tile list out of range in ") + what);
      return SPDE_ERR_STATE;
    }
  return SPDE_OK;
}

ArenaSizes arena_sizes(const spde_plan* pl, int nrhs) {
  ArenaSizes a;
  a.sz[kFront] = pl->lay_front;
  a.sz[kZ] = pl->lay_z;
  a.sz[kSigma] = pl->lay_front;
  a.sz[kWork] = pl->work_doubles;
  a.sz[kVec] = pl->sym.vec_doubles * nrhs;
  a.sz[kX] = pl->sym.n * nrhs;
  return a;
}

void make_tiles(GemmLaunch& g, int force_tile);

// Split-K for launches of 64-tiles that leave the chip's 1,024 block slots
// (four per CU) under-filled with deep problems: under 256 tiles and at least
// 512 deep, S = min(512 / tiles, K_max / 256, 64) chunks; under 1,024 tiles
// and at least 1,024 deep, S = min(round(2048 / tiles), K_max / 256) chunks
// (about two rounds of the chip).  Chunks are at least 256 deep; the partial
// tiles take S * tiles * 64 * 64 doubles of the workspace counted in *ws.
void plan_split(GemmLaunch& g, int64_t* ws) {
  if (!ws || g.gemv || g.tile != 64 || g.h_tiles.empty()) return;
  int kmax = 0;
  for (const GemmProb& P : g.h_probs) kmax = std::max(kmax, P.K);
  const int64_t nt = (int64_t)g.h_tiles.size();
  int S = 0;
  if (nt < 256 && kmax >= 512)
    S = (int)std::min<int64_t>(std::min<int64_t>(512 / nt, kmax / 256), 64);
  else if (nt < 1024 && kmax >= 1024)
    S = (int)std::min<int64_t>((2048 + nt / 2) / nt, kmax / 256);
  if (S < 2) return;
  std::vector<GemmTile> t;
  t.reserve(nt * S);
  for (const GemmTile& b : g.h_tiles)
    for (int q = 0; q < S; ++q) t.push_back({b.prob, b.tm, b.tn, q});
  g.h_tiles.swap(t);
  g.split = S;
  g.ws_off = *ws;
  *ws += (int64_t)g.h_tiles.size() * 64 * 64;
}

int finalize(GemmLaunch& g, int64_t* ws) {
  make_tiles(g, 0);
  plan_split(g, ws);
  g.nprobs = (int)g.h_probs.size();
  g.ntiles = (int)g.h_tiles.size();
  int rc = upload(&g.d_probs, g.h_probs);
  if (rc) return rc;
  return upload(&g.d_tiles, g.h_tiles);
}

// flop_scale: algorithmic share of 2MNK (0.5 for a triangular operand)
void add_prob(GemmLaunch& g, const GemmProb& P, bool lower, double flop_scale = 1.0) {
  if (P.M <= 0 || P.N <= 0) return;
  if (P.K <= 0 && P.beta == 1.0) return;
  GemmProb Q = P;
  Q.lower = lower ? 1 : 0;
  g.h_probs.push_back(Q);
  g.flops += 2.0 * P.M * (double)P.N * P.K * (lower ? 0.5 : 1.0) * flop_scale;
  const double cmn = P.M * (double)P.N * (lower ? 0.5 : 1.0);
  g.bytes += 8.0 * (P.M * (double)P.K + P.N * (double)P.K + cmn * (P.beta != 0.0 ? 2.0 : 1.0));
}

// A launch takes the large tiles when the mean depth K is at least 128 and
// they fill the chip's block slots once (768 of 128x64, three per CU;
// 512 of 128x128, two per CU); else 64 (more blocks in flight, less waste at
// the edges).  Then the tile list (tiles strictly above the diagonal of a lower problem
// are skipped).
void make_tiles(GemmLaunch& g, int force_tile) {
  // few right-hand sides: row blocks of 64 (A not transposed) or groups of 4
  // outputs (A transposed) for the bandwidth-bound kernel
  bool narrow = !g.h_probs.empty() && !g.tb && !force_tile;
  for (const GemmProb& P : g.h_probs) narrow = narrow && P.N <= kGemvMaxN && !P.lower;
  g.gemv = narrow;
  if (narrow) {
    g.tile = 0;
    g.h_tiles.clear();
    int kmax = 0;
    for (const GemmProb& P : g.h_probs) kmax = std::max(kmax, P.K);
    g.gemv_wide = !g.ta && kmax >= 1024;
    const int rows = g.ta ? 4 : 64;
    for (size_t i = 0; i < g.h_probs.size(); ++i)
      for (int a = 0; a < (g.h_probs[i].M + rows - 1) / rows; ++a) g.h_tiles.push_back({(int32_t)i, a, 0, 0});
    return;
  }
  // 16-byte loads of operands with contiguous k (op(A) = A^T, op(B) = B)
  g.vec = true;
  for (const GemmProb& P : g.h_probs) {
    if (g.ta) g.vec = g.vec && !(P.a_off & 1) && !(P.lda & 1);
    if (!g.tb) g.vec = g.vec && !(P.b_off & 1) && !(P.ldb & 1);
  }
  g.tile = 128;
  const int64_t BM = g.tile_m(), BN = g.tile_n();
  int64_t big = 0;  // large tiles that would be launched (on or below the diagonal of lower problems)
  double ksum = 0.0;
  for (const GemmProb& P : g.h_probs) {
    const int64_t tm = (P.M + BM - 1) / BM, tn = (P.N + BN - 1) / BN;
    for (int64_t a = 0; a < tm; ++a) big += P.lower ? std::min(tn, ((a + 1) * BM + BN - 1) / BN) : tn;
    ksum += P.K;
  }
  const bool deep = !g.h_probs.empty() && ksum / g.h_probs.size() >= 128.0;
  g.tile = force_tile ? force_tile : (deep && big >= (BM * BN == 128 * 64 ? 768 : 512) ? 128 : 64);
  g.h_tiles.clear();
  const int T = g.tile_m(), TN = g.tile_n();
  for (size_t i = 0; i < g.h_probs.size(); ++i) {
    const GemmProb& P = g.h_probs[i];
    const int tm = (P.M + T - 1) / T, tn = (P.N + TN - 1) / TN;
    for (int a = 0; a < tm; ++a)
      for (int b = 0; b < tn; ++b)
        if (!P.lower || (a + 1) * T > b * TN) g.h_tiles.push_back({(int32_t)i, a, b, 0});
  }
  // deepest tiles first: the blocks dispatched last are the shortest, which
  // shortens the launch's final, partly filled round
  auto depth = [&](const GemmTile& t) {
    const GemmProb& P = g.h_probs[t.prob];
    int kb = 0, ke = P.K;
    if (P.kmode == 1) kb = std::min(P.K, t.tn * TN);
    if (P.kmode == 2) kb = std::min(P.K, t.tm * T);
    if (P.kmode == 3) ke = std::min(P.K, (t.tm + 1) * T);
    return ke - kb;
  };
  std::stable_sort(g.h_tiles.begin(), g.h_tiles.end(),
                   [&](const GemmTile& x, const GemmTile& y) { return depth(x) > depth(y); });
}

// A problem with a triangular operand whose zeros the kernel skips (kmode).
GemmProb tri(GemmProb P, int kmode) {
  P.kmode = (int8_t)kmode;
  return P;
}

GemmProb prob(int8_t ab, int64_t ao, int lda, int8_t bb, int64_t bo, int ldb, int8_t cb, int64_t co, int ldc, int M,
              int N, int K, double alpha, double beta) {
  GemmProb P{};
  P.a_off = ao;
  P.b_off = bo;
  P.c_off = co;
  P.lda = lda;
  P.ldb = ldb;
  P.ldc = ldc;
  P.M = M;
  P.N = N;
  P.K = K;
  P.a_base = ab;
  P.b_base = bb;
  P.c_base = cb;
  P.lower = 0;
  P.kmode = 0;
  P.alpha = alpha;
  P.beta = beta;
  return P;
}

// Fronts and tasks of one level in ticket order: by column j over all fronts,
// diagonal j, then diagonal j + 1 ahead of the tiles below j (it waits for W_j
// only), then those tiles, two row tiles to a task.  Checked here: every tile
// that a task waits for is produced by a task with a lower ticket.
int build_front_tasks(spde_plan* pl, LevelPlan& L) {
  const Symbolic& sym = pl->sym;
  std::vector<FrontDesc> fd;
  int pmax = 0;
  for (int id : L.nodes) {
    const Node& nd = sym.nodes[id];
    const FrontLay& f = pl->lay[id];
    if (nd.p == 0) continue;
    FrontDesc d{};
    d.foff = f.foff;
    d.zoff = f.zoff;
    d.ld = f.ld;
    d.pp = f.pp;
    d.p = nd.p;
    d.nrows = f.pp + (int)nd.B.size();
    d.R = (d.nrows + 63) / 64;
    d.P = f.pp / 64;
    d.flag0 = pl->nflags;
    d.colbase = nd.start;
    if (f.pp != 64 * ((nd.p + 63) / 64) || f.foff + (int64_t)f.ld * d.nrows > pl->lay_front || f.ld < d.nrows ||
        f.zoff + (int64_t)f.pp * f.pp > pl->lay_z || (f.foff & 15) || (f.ld & 15) || (f.zoff & 15)) {
      set_error("front layout out of bounds");
      return SPDE_ERR_STATE;
    }
    pl->nflags += d.R * d.P;
    pmax = std::max(pmax, d.P);
    fd.push_back(d);
  }
  std::vector<FrontTask> tasks;
  for (size_t q = 0; q < fd.size(); ++q) tasks.push_back({(int32_t)q, 0, 0, 0});
  for (int j = 0; j < pmax; ++j) {
    for (size_t q = 0; q < fd.size(); ++q)
      if (j + 1 < fd[q].P) tasks.push_back({(int32_t)q, j + 1, j + 1, 0});
    for (size_t q = 0; q < fd.size(); ++q) {
      if (j >= fd[q].P) continue;
      for (int i = j + 1 < fd[q].P ? j + 2 : j + 1; i < fd[q].R; i += 2) tasks.push_back({(int32_t)q, j, i, 0});
    }
  }
  std::vector<std::vector<int>> made(fd.size());  // ticket of each tile
  for (size_t q = 0; q < fd.size(); ++q) made[q].assign((size_t)fd[q].R * fd[q].P, -1);
  auto at = [&](int q, int i, int k) -> int& { return made[q][(size_t)k * fd[q].R + i]; };
  for (size_t t = 0; t < tasks.size(); ++t) {
    const FrontTask& T = tasks[t];
    if (T.i == T.j) {
      at(T.front, T.j, T.j) = (int)t;
      if (T.j > 0) at(T.front, T.j, T.j - 1) = (int)t;
    } else {
      for (int i = T.i; i < std::min(T.i + 2, fd[T.front].R); ++i) at(T.front, i, T.j) = (int)t;
    }
  }
  bool ok = true;
  for (size_t t = 0; t < tasks.size(); ++t) {
    const FrontTask& T = tasks[t];
    auto before = [&](int i, int k) {
      const int m = at(T.front, i, k);
      ok = ok && m >= 0 && m < (int)t;
    };
    if (T.i == T.j) {
      for (int k = 0; k + 1 < T.j; ++k) before(T.j, k), before(T.j - 1, k);
      if (T.j > 0) before(T.j - 1, T.j - 1);
    } else {
      for (int k = 0; k < T.j; ++k) {
        before(T.j, k);
        for (int i = T.i; i < std::min(T.i + 2, fd[T.front].R); ++i) before(i, k);
      }
      before(T.j, T.j);
    }
  }
  if (!ok) {
    set_error("factorisation tasks out of order");
    return SPDE_ERR_STATE;
  }
  L.ntasks = (int)tasks.size();
  int rc = upload(&L.d_fronts, fd);
  if (rc) return rc;
  return upload(&L.d_tasks, tasks);
}

int build_factor_plan(spde_plan* pl) {
  const Symbolic& sym = pl->sym;
  pl->split_fs = 0;
  pl->levels.assign(sym.levels.size(), LevelPlan());
  for (size_t l = 0; l < sym.levels.size(); ++l) {
    LevelPlan& L = pl->levels[l];
    L.nodes = sym.levels[l];
    std::vector<int4> own;
    for (int id : L.nodes) {
      const Node& nd = sym.nodes[id];
      const FrontLay& f = pl->lay[id];
      if (nd.nchild == 0) continue;
      for (int ti = 0; ti * 64 < f.pp + (int)nd.B.size(); ++ti)
        for (int tj = 0; tj <= ti && tj * 64 < f.pp; ++tj) own.push_back(make_int4(id, ti, tj, 0));
    }
    L.nowntiles = (int)own.size();
    int rcf = upload(&L.d_owntiles, own);
    if (!rcf) rcf = build_front_tasks(pl, L);
    if (rcf) return rcf;
    L.syrk.ta = false;
    L.syrk.tb = true;
    L.syrk.pull = true;
    for (int id : L.nodes) {
      const Node& nd = sym.nodes[id];
      const FrontLay& f = pl->lay[id];
      const int n = f.ld, b = (int)nd.B.size();
      // the update block is written here together with the children's
      // contributions to it
      GemmProb P = prob(kFront, f.foff + f.pp, n, kFront, f.foff + f.pp, n, kFront,
                        f.foff + f.pp + (int64_t)f.pp * n, n, b, b, nd.p, -1.0, 0.0);
      P.pull = id;
      P.pull_row = f.pp;
      add_prob(L.syrk, P, true);
    }
    int rc = finalize(L.syrk, &pl->split_fs);
    if (rc) return rc;
  }
  // inverse of L11 for every node: recursive halving, batched by height
  struct Op {
    int node, a, m, b;
  };
  std::vector<std::vector<Op>> ops;
  std::function<int(int, int, int)> rec = [&](int node, int a, int b) -> int {
    if (b - a <= NB) return 0;
    int half = (b - a + 1) / 2;
    half = ((half + NB - 1) / NB) * NB;
    const int m = a + half;
    if (m >= b) return 0;
    const int h = 1 + std::max(rec(node, a, m), rec(node, m, b));
    if ((int)ops.size() <= h) ops.resize(h + 1);
    ops[h].push_back({node, a, m, b});
    return h;
  };
  for (size_t q = 0; q < sym.nodes.size(); ++q) rec((int)q, 0, sym.nodes[q].p);
  pl->trtri.clear();
  int64_t work = 0;
  for (size_t h = 1; h < ops.size(); ++h) {
    GemmLaunch gx, gz;
    int64_t woff = 0;
    for (const Op& o : ops[h]) {
      const FrontLay& f = pl->lay[o.node];
      const int n = f.ld, p = f.pp;
      const int r = o.b - o.m, c = o.m - o.a, rl = (r + 15) / 16 * 16;
      // X = L_ma Z_aa (Z_aa lower), Z_ma = -Z_mm X (Z_mm lower)
      add_prob(gx, tri(prob(kFront, f.foff + o.m + (int64_t)o.a * n, n, kZ, f.zoff + o.a + (int64_t)o.a * p, p,
                            kWork, woff, rl, r, c, c, 1.0, 0.0),
                       1),
               false, 0.5);
      add_prob(gz, tri(prob(kZ, f.zoff + o.m + (int64_t)o.m * p, p, kWork, woff, rl, kZ,
                            f.zoff + o.m + (int64_t)o.a * p, p, r, c, r, -1.0, 0.0),
                       3),
               false, 0.5);
      woff += (int64_t)rl * c;
    }
    work = std::max(work, woff);
    int rc = finalize(gx, &pl->split_fs);
    if (rc) return rc;
    rc = finalize(gz, &pl->split_fs);
    if (rc) return rc;
    pl->trtri.push_back(std::move(gx));
    pl->trtri.push_back(std::move(gz));
  }
  pl->trtri_heights = (int)(pl->trtri.size() / 2);
  pl->work_doubles = std::max<int64_t>(work, 1);
  const ArenaSizes as = arena_sizes(pl, 1);
  for (auto& L : pl->levels) {
    int rc = validate(L.syrk, as, "factor syrk");
    if (rc) return rc;
  }
  for (auto& g : pl->trtri) {
    int rc = validate(g, as, "inverse of L11");
    if (rc) return rc;
  }
  for (const Node& nd : sym.nodes)
    for (int rp : nd.relpos)
      if (nd.parent < 0 || rp < 0 || rp >= sym.nodes[nd.parent].n()) {
        set_error("relative position out of the parent front");
        return SPDE_ERR_STATE;
      }
  return SPDE_OK;
}

void free_launch(GemmLaunch& g);

int build_solve_plan(spde_plan* pl, int k) {
  auto hit = pl->solve_cache.find(k);
  if (hit != pl->solve_cache.end()) {
    const auto& v = hit->second.launches;
    for (size_t l = 0; l < pl->levels.size(); ++l) {
      LevelPlan& L = pl->levels[l];
      L.fwd_y = v[4 * l], L.fwd_u = v[4 * l + 1], L.bwd_t = v[4 * l + 2], L.bwd_x = v[4 * l + 3];
    }
    pl->split_solve = hit->second.split;
    pl->solve_nrhs = k;
    return SPDE_OK;
  }
  const Symbolic& sym = pl->sym;
  const int n = (int)sym.n;
  // solve launches take the split workspace after the factor and
  // selected-inverse regions (fixed when the plan is made)
  int64_t acc = pl->split_fs;
  spde_plan::SolveSet set;
  for (auto& L : pl->levels) {
    GemmLaunch fy, fu, bt, bx;
    fy.ta = false, fy.tb = false;
    fu.ta = false, fu.tb = false;
    bt.ta = true, bt.tb = false;
    bx.ta = true, bx.tb = false;
    for (int id : L.nodes) {
      const Node& nd = sym.nodes[id];
      const FrontLay& f = pl->lay[id];
      const int nf = nd.n(), p = nd.p, b = (int)nd.B.size();
      const int64_t v = nd.voff * k;
      add_prob(fy, prob(kZ, f.zoff, f.pp, kVec, v, nf, kX, nd.start, n, p, k, p, 1.0, 0.0), false);
      add_prob(fu, prob(kFront, f.foff + f.pp, f.ld, kX, nd.start, n, kVec, v + p, nf, b, k, p, -1.0, 1.0), false);
      add_prob(bt, prob(kFront, f.foff + f.pp, f.ld, kVec, v + p, nf, kVec, v, nf, p, k, b, -1.0, 1.0), false);
      add_prob(bx, prob(kZ, f.zoff, f.pp, kVec, v, nf, kX, nd.start, n, p, k, p, 1.0, 0.0), false);
    }
    const ArenaSizes as = arena_sizes(pl, k);
    for (GemmLaunch* g : {&fy, &fu, &bt, &bx}) {
      int rc = validate(*g, as, "solve");
      if (!rc) rc = finalize(*g, &acc);
      if (rc) {
        for (auto& q : set.launches) free_launch(q);
        for (GemmLaunch* h : {&fy, &fu, &bt, &bx}) free_launch(*h);
        return rc;
      }
    }
    set.launches.push_back(fy);
    set.launches.push_back(fu);
    set.launches.push_back(bt);
    set.launches.push_back(bx);
  }
  set.split = acc - pl->split_fs;
  pl->solve_cache[k] = set;
  return build_solve_plan(pl, k);
}

int build_selinv_plan(spde_plan* pl) {
  const Symbolic& sym = pl->sym;
  PlanExtra* ex = extra(pl);
  // X^T = Z^T L21^T (p x b) lives in its front's own block right of the own
  // columns (rows [0, p), columns from pp), which the selected inverse does not
  // use otherwise: the X products run ahead of the level chain on a second stream
  // without a workspace.  Stored transposed, Sigma21 = -Sigma22 X reads contiguous
  // rows of both operands and Sigma11 -= X^T Sigma21 of its first
  for (size_t l = 0; l < pl->levels.size(); ++l) {
    LevelPlan& L = pl->levels[l];
    L.si_x.ta = true, L.si_x.tb = true;
    L.si_s21.ta = false, L.si_s21.tb = true;
    L.si_s11a.ta = true, L.si_s11a.tb = false;
    L.si_s11b.ta = false, L.si_s11b.tb = false;
    std::vector<int4> gt;
    for (size_t q = 0; q < L.nodes.size(); ++q) {
      const Node& nd = sym.nodes[L.nodes[q]];
      const FrontLay& f = pl->lay[L.nodes[q]];
      const int p = nd.p, b = (int)nd.B.size();
      if (b > 0 && nd.parent >= 0)
        for (int ti = 0; ti < (b + 63) / 64; ++ti)
          for (int tj = 0; tj <= ti; ++tj) gt.push_back(make_int4((int)q, ti, tj, 0));
      const int64_t xo = f.foff + (int64_t)f.pp * f.ld;
      add_prob(L.si_x, tri(prob(kZ, f.zoff, f.pp, kFront, f.foff + f.pp, f.ld, kSigma, xo, f.ld, p, b, p, 1.0, 0.0), 2),
               false, 0.5);
      add_prob(L.si_s21, prob(kSigma, xo + f.pp, f.ld, kSigma, xo, f.ld, kSigma, f.foff + f.pp, f.ld, b, p, b, -1.0, 0.0),
               false);
      add_prob(L.si_s11a, tri(prob(kZ, f.zoff, f.pp, kZ, f.zoff, f.pp, kSigma, f.foff, f.ld, p, p, p, 1.0, 0.0), 2), true,
               1.0 / 3.0);
      add_prob(L.si_s11b, prob(kSigma, xo, f.ld, kSigma, f.foff + f.pp, f.ld, kSigma, f.foff, f.ld, p, p, b, -1.0, 1.0),
               true);
    }
    const ArenaSizes as = arena_sizes(pl, 1);
    for (GemmLaunch* g : {&L.si_x, &L.si_s21, &L.si_s11a, &L.si_s11b}) {
      int rc = validate(*g, as, "selected inverse");
      if (rc) return rc;
      rc = finalize(*g, &pl->split_fs);
      if (rc) return rc;
    }
    LevelDev& D = ex->lvl[l];
    D.ngtiles = (int)gt.size();
    int rc = upload(&D.d_gtiles, gt);
    if (rc) return rc;
  }
  pl->selinv_built = true;
  return SPDE_OK;
}

void free_launch(GemmLaunch& g) {
  hipFree(g.d_probs);
  hipFree(g.d_tiles);
  g.d_probs = nullptr;
  g.d_tiles = nullptr;
}

// LDS each 64-tile block of the selected inverse's second-stream products
// (X = L21 Z, Z^T Z, one level ahead of the chain) reserves, so that the chain's own
// products on the first stream keep most of the chip: 48 KB allows three such blocks
// of the register-fed forms per CU, one or two of the staged A^T B form.  Exact
// evaluation at 100x100x20 and 60x60x12, two alternating runs each on one card: 48 KB
// 60.7 and 61.0, 7.0 and 7.2 ms; none 61.2 and 61.5, 7.3 and 7.3; 32 KB 61.4 and
// 61.0, 7.3 and 7.0; 64 KB 60.8 and 61.4, 7.0 and 7.1.  (Capping the 128-tile launches
// too slowed each by a fifth on the staged products: they run at full width.)
constexpr unsigned kPreLds = 48 * 1024;
// GEMM launch, bracketed by HIP events when the plan's timing is enabled.
void run_gemm(spde_plan* pl, const GemmLaunch& g, const Bases& b, hipStream_t s, unsigned lds = 0) {
  if (g.ntiles == 0) return;
  const int kind = (g.tile == 128 ? 4 : 0) + (g.ta ? 2 : 0) + (g.tb ? 1 : 0);
  if (pl->prof_on && ((pl->prof_mask >> kind) & 1)) {
    while (pl->prof_ev.size() < 2 * (pl->prof_n + 1)) {
      hipEvent_t e;
      hipEventCreate(&e);
      pl->prof_ev.push_back(e);
    }
    hipEventRecord(pl->prof_ev[2 * pl->prof_n], s);
    launch_gemm(g, b, s, lds);
    hipEventRecord(pl->prof_ev[2 * pl->prof_n + 1], s);
    if (pl->prof_flops.size() <= pl->prof_n) {
      pl->prof_flops.resize(pl->prof_n + 1);
      pl->prof_bytes.resize(pl->prof_n + 1);
      pl->prof_tiles.resize(pl->prof_n + 1);
      pl->prof_kind.resize(pl->prof_n + 1);
    }
    pl->prof_flops[pl->prof_n] = g.flops;
    pl->prof_bytes[pl->prof_n] = g.bytes;
    pl->prof_tiles[pl->prof_n] = g.ntiles;
    pl->prof_kind[pl->prof_n] = kind;
    pl->prof_n++;
    pl->prof_stream = s;
    return;
  }
  launch_gemm(g, b, s, lds);
}

// The slot's split-K workspace covers the factor, selected-inverse and
// current solve regions (grows only when the solve plan grows, after the
// device has drained).
int ensure_splitws(spde_plan* pl, int slot) {
  Slot& sl = pl->slots[slot];
  const int64_t need = pl->split_fs + pl->split_solve;
  if (need <= sl.splitws_cap) return SPDE_OK;
  SPDE_HIP(hipDeviceSynchronize());
  hipFree(sl.splitws);
  sl.splitws = nullptr;
  sl.splitws_cap = 0;
  SPDE_HIP(hipMalloc((void**)&sl.splitws, sizeof(double) * need));
  sl.splitws_cap = need;
  return SPDE_OK;
}

Bases make_bases(spde_plan* pl, int slot, double* x) {
  Bases b;
  b.ws = pl->slots[slot].splitws;
  b.pulls = pl->d_pulls;
  b.inv = pl->d_inv;
  b.p[kFront] = pl->slots[slot].front;
  b.p[kZ] = pl->slots[slot].z;
  b.p[kSigma] = pl->slots[slot].sigma;
  b.p[kWork] = pl->slots[slot].work;
  b.p[kVec] = pl->slots[slot].vec;
  b.p[kX] = x;
  return b;
}

// Words of a slot's factorisation counters: stop flag, tickets, tiles.
int flag_words(const spde_plan* pl) { return 1 + (int)pl->levels.size() + pl->nflags; }

// Device arenas of a factor slot, allocated on its first factorisation.  The
// fronts and Z are cleared once (on the factorisation's stream): later
// factorisations clear only the lower triangles, and nothing writes above a
// front's diagonal.
int ensure_slot(spde_plan* pl, int slot, hipStream_t stream) {
  Slot& sl = pl->slots[slot];
  if (sl.front) return SPDE_OK;
  const Symbolic& sym = pl->sym;
  const size_t fb = sizeof(double) * std::max<int64_t>(pl->lay_front, 1);
  const size_t zb = sizeof(double) * std::max<int64_t>(pl->lay_z, 1);
  if (hipMalloc((void**)&sl.front, fb) != hipSuccess || hipMalloc((void**)&sl.z, zb) != hipSuccess ||
      hipMalloc((void**)&sl.work, sizeof(double) * pl->work_doubles) != hipSuccess ||
      hipMalloc((void**)&sl.partial, sizeof(double) * std::max(logdet_parts(sym.n), 1)) != hipSuccess ||
      hipMalloc((void**)&sl.ld, sizeof(double)) != hipSuccess ||
      hipMalloc((void**)&sl.flags, sizeof(int) * flag_words(pl)) != hipSuccess ||
      hipMalloc((void**)&sl.status, sizeof(int)) != hipSuccess) {
    for (void* p : {(void*)sl.front, (void*)sl.z, (void*)sl.work, (void*)sl.partial, (void*)sl.ld, (void*)sl.status,
                    (void*)sl.flags})
      if (p) hipFree(p);
    sl.front = sl.z = sl.work = sl.partial = sl.ld = nullptr;
    sl.status = sl.flags = nullptr;
    set_error("factor slot " + std::to_string(slot) + ": device allocation of " +
              std::to_string((fb + zb) >> 20) + " MiB failed");
    return SPDE_ERR_ALLOC;
  }
  // cleared on the stream of the factorisation that follows, so the clear is
  // ordered before it whatever stream the caller uses
  SPDE_HIP(hipMemsetAsync(sl.front, 0, fb, stream));
  SPDE_HIP(hipMemsetAsync(sl.z, 0, zb, stream));
  SPDE_HIP(hipMemsetAsync(sl.status, 0, sizeof(int), stream));
  return SPDE_OK;
}

int check_slot(spde_plan* pl, int slot) {
  if (!pl || pl->host_only) {
    set_error("plan has no device state");
    return SPDE_ERR_STATE;
  }
  if (slot < 0 || slot >= pl->nslots) {
    set_error("factor slot out of range");
    return SPDE_ERR_ARG;
  }
  return SPDE_OK;
}

}  // namespace

extern "C" {

const char* spde_last_error(void) { return g_err.c_str(); }

int spde_plan_create(int M, int N, int T, int bc, int leaf_max, int nslots, int flags, spde_plan** out) {
  if (!out || bc < 1 || bc > 3 || M < 2 || N < 2 || T < 1 || nslots < 0) {
    set_error("spde_plan_create: invalid argument");
    return SPDE_ERR_ARG;
  }
  *out = nullptr;
  spde_plan* pl = new spde_plan();
  pl->lat = Lattice{M, N, T, bc};
  pl->lat.wide = (flags & SPDE_PLAN_WIDE_TIME) ? 1 : 0;
  try {
    build_structure(pl->lat, pl->st);
    if (pl->lat.wide) check_wide_layout(pl->lat, pl->st);
    build_symbolic(pl->lat, pl->st, leaf_max > 0 ? leaf_max : 128, pl->sym);
    build_scatter_map(pl->st, pl->sym, pl->map);
  } catch (const std::exception& e) {
    set_error(std::string("spde_plan_create: ") + e.what());
    delete pl;
    return SPDE_ERR_ARG;
  }
  build_layout(pl);
  pl->host_only = (flags & SPDE_PLAN_HOST_ONLY) != 0;
  pl->nslots = nslots;
  PlanExtra* ex = new PlanExtra();
  pl->extra = ex;
  if (pl->host_only) {
    // build and bounds-check every launch schedule without touching the device
    g_host_only_build = true;
    ex->lvl.resize(pl->sym.levels.size());
    int rc = build_factor_plan(pl);
    if (!rc) rc = build_selinv_plan(pl);
    if (!rc) rc = build_solve_plan(pl, 3);
    g_host_only_build = false;
    if (rc) {
      spde_plan_destroy(pl);
      return rc;
    }
    *out = pl;
    return SPDE_OK;
  }
  const Symbolic& sym = pl->sym;
  std::vector<int64_t> dmap = layout_map(pl);
  int rc = SPDE_OK;
#define TRY(x)                   \
  do {                           \
    rc = (x);                    \
    if (rc) {                    \
      spde_plan_destroy(pl);     \
      return rc;                 \
    }                            \
  } while (0)
  TRY(upload(&pl->d_indptr, pl->st.indptr));
  TRY(upload(&pl->d_indices, pl->st.indices));
  TRY(upload(&pl->d_code, pl->st.code));
  // the diagonal add and the log-determinant read F[map[diag[i]]] for every variable
  if ((int64_t)pl->st.diag.size() != sym.n) TRY((set_error("diagonal positions do not match the order"), SPDE_ERR_STATE));
  for (int64_t i = 0; i < sym.n; ++i) {
    const int64_t e = pl->st.diag[i];
    if (e < 0 || e >= (int64_t)dmap.size() || dmap[e] < 0 || dmap[e] >= pl->lay_front)
      TRY((set_error("diagonal entry outside the fronts"), SPDE_ERR_STATE));
  }
  TRY(upload(&pl->d_diag, pl->st.diag));
  TRY(upload(&pl->d_map, dmap));
  // in place: the mirror of an upper entry is a lower one, which stays as it is
  for (size_t e = 0; e < dmap.size(); ++e)
    if (dmap[e] < 0) dmap[e] = dmap[pl->st.mirror[e]];
  TRY(upload(&pl->d_mapsym, dmap));
  TRY(upload(&pl->d_perm, sym.perm));
  std::vector<int32_t> relpos(std::max<int64_t>(sym.relpos_total, 1)), bnd(std::max<int64_t>(sym.relpos_total, 1));
  std::vector<NodeDev> nodes(sym.nodes.size());
  std::vector<int32_t> children(2 * sym.nodes.size(), -1);
  for (size_t q = 0; q < sym.nodes.size(); ++q) {
    const Node& nd = sym.nodes[q];
    for (size_t k = 0; k < nd.B.size(); ++k) {
      bnd[nd.relpos_off + k] = nd.B[k];
      // position in the parent's padded front
      int rp = nd.relpos.empty() ? 0 : nd.relpos[k];
      if (nd.parent >= 0 && rp >= sym.nodes[nd.parent].p) rp += pl->lay[nd.parent].pp - sym.nodes[nd.parent].p;
      relpos[nd.relpos_off + k] = rp;
    }
    nodes[q] = NodeDev{pl->lay[q].foff, pl->lay[q].zoff, nd.voff, nd.relpos_off, nd.start, nd.p, nd.n(), nd.parent,
                       (int32_t)nd.B.size(), nd.level, pl->lay[q].ld, pl->lay[q].pp};
    for (int c = 0; c < nd.nchild; ++c) children[2 * q + c] = nd.child[c];
  }
  TRY(upload(&pl->d_relpos, relpos));
  TRY(upload(&pl->d_bnd, bnd));
  TRY(upload(&pl->d_nodes, nodes));
  {
    // children's rows by row of the padded parent front
    std::vector<Pull> pulls(sym.nodes.size());
    int nfmax = 0;
    for (size_t q = 0; q < sym.nodes.size(); ++q)
      nfmax = std::max(nfmax, pl->lay[q].pp + (int)sym.nodes[q].B.size());
    std::vector<int32_t> inv(nfmax, -1);  // the rows of a missing child
    for (size_t q = 0; q < sym.nodes.size(); ++q) {
      const Node& nd = sym.nodes[q];
      Pull& P = pulls[q];
      for (int s = 0; s < 2; ++s) {
        P.u[s] = 0;
        P.inv[s] = 0;
        P.cld[s] = 0;
        if (s >= nd.nchild || sym.nodes[nd.child[s]].B.empty()) continue;
        const Node& c = sym.nodes[nd.child[s]];
        const FrontLay& cl = pl->lay[nd.child[s]];
        const int nf = pl->lay[q].pp + (int)nd.B.size();
        P.u[s] = cl.foff + cl.pp + (int64_t)cl.pp * cl.ld;
        P.cld[s] = cl.ld;
        P.inv[s] = (int64_t)inv.size();
        inv.resize(inv.size() + nf, -1);
        for (size_t k = 0; k < c.B.size(); ++k) {
          const int at = relpos[c.relpos_off + k];
          if (at < 0 || at >= nf || (k && at <= relpos[c.relpos_off + k - 1]) ||
              P.u[s] + (int64_t)(c.B.size() - 1) * (cl.ld + 1) >= pl->lay_front)
            TRY((set_error("child rows outside the parent front"), SPDE_ERR_STATE));
          inv[P.inv[s] + at] = (int32_t)k;
        }
      }
    }
    TRY(upload(&pl->d_pulls, pulls));
    TRY(upload(&pl->d_inv, inv));
  }
  TRY(upload(&ex->d_children, children));
  {
    std::vector<int4> zt;
    for (size_t q = 0; q < sym.nodes.size(); ++q) {
      // lower triangle of the own columns only (the update block is
      // written by the SYRK before anything adds to it)
      const int pp = pl->lay[q].pp, nt = (pp + (int)sym.nodes[q].B.size() + 63) / 64, pt = pp / 64;
      for (int a = 0; a < nt; ++a)
        for (int b = 0; b <= a && b < pt; ++b) zt.push_back(int4{(int)q, a, b, 0});
    }
    if (zt.size() > (size_t)INT32_MAX) TRY((set_error("front tile list too long"), SPDE_ERR_STATE));
    ex->nztiles = (int)zt.size();
    TRY(upload(&ex->d_ztiles, zt));
  }
  ex->lvl.resize(sym.levels.size());
  for (size_t l = 0; l < sym.levels.size(); ++l) {
    ex->lvl[l].nn = (int)sym.levels[l].size();
    TRY(upload(&ex->lvl[l].d_nodes, sym.levels[l]));
  }
  TRY(build_factor_plan(pl));
  TRY(build_selinv_plan(pl));  // fixes the split workspace of factor and selected inverse
  const int64_t Ns = pl->lat.Ns();
  SPDE_HIP(hipMalloc((void**)&pl->d_tmpl, sizeof(double) * Ns * kTmpl));
  SPDE_HIP(hipMalloc((void**)&pl->d_red, sizeof(double)));
  if (pl->lat.T == 1) {
    std::vector<int32_t> pos((size_t)Ns * 25, -1);
    for (int64_t r = 0; r < Ns; ++r)
      for (int64_t e = pl->st.indptr[r]; e < pl->st.indptr[r + 1]; ++e)
        if (pl->st.code[e] < 25) pos[(size_t)r * 25 + pl->st.code[e]] = (int32_t)e;
    TRY(upload(&pl->d_pos25, pos));
  }
  SPDE_HIP(hipMalloc((void**)&pl->d_acan, sizeof(double) * Ns * 9));
  SPDE_HIP(hipMalloc((void**)&pl->d_a0can, sizeof(double) * Ns * 9));
  SPDE_HIP(hipMalloc((void**)&pl->d_qdiag, sizeof(double) * Ns));
  // slot arenas are allocated by the slot's first factorisation (ensure_slot):
  // a plan with two slots of which one is used holds one slot's memory
  pl->slots.resize(nslots);
  SPDE_HIP(hipMalloc((void**)&pl->d_win, sizeof(double) * Ns * 60));
  *out = pl;
  return SPDE_OK;
#undef TRY
}

void spde_plan_destroy(spde_plan* pl) {
  if (!pl) return;
  if (!pl->host_only) spde::loglik_release(pl);
  if (pl->host_only) {
    delete extra(pl);
  } else {
    hipDeviceSynchronize();
    for (auto* p : {(void*)pl->d_indptr, (void*)pl->d_indices, (void*)pl->d_code, (void*)pl->d_diag,
                    (void*)pl->d_map, (void*)pl->d_mapsym, (void*)pl->d_perm, (void*)pl->d_relpos,
                    (void*)pl->d_bnd, (void*)pl->d_nodes, (void*)pl->d_pulls, (void*)pl->d_inv, (void*)pl->d_tmpl, (void*)pl->d_acan,
                    (void*)pl->d_a0can, (void*)pl->d_qdiag, (void*)pl->d_win, (void*)pl->d_red, (void*)pl->d_pos25,
                    (void*)pl->d_sprow, (void*)pl->d_spcol, (void*)pl->d_gpart, (void*)pl->d_tan})
      hipFree(p);
    for (auto& s : pl->slots) {
      hipFree(s.front);
      hipFree(s.z);
      hipFree(s.sigma);
      hipFree(s.work);
      hipFree(s.partial);
      hipFree(s.ld);
      hipFree(s.status);
      hipFree(s.flags);
      hipFree(s.vec);
      hipFree(s.xy);
      hipFree(s.splitws);
    }
    for (auto& L : pl->levels) {
      hipFree(L.d_fronts);
      hipFree(L.d_tasks);
      hipFree(L.d_owntiles);
      for (GemmLaunch* g : {&L.syrk, &L.si_x, &L.si_s21, &L.si_s11a, &L.si_s11b}) free_launch(*g);
    }
    for (auto& g : pl->trtri) free_launch(g);
    for (auto& kv : pl->solve_cache)
      for (auto& g : kv.second.launches) free_launch(g);
    for (auto e : pl->prof_ev) hipEventDestroy(e);
    if (pl->prof_base) hipEventDestroy(pl->prof_base);
    if (PlanExtra* ex = extra(pl)) {
      for (auto& d : ex->lvl) {
        hipFree(d.d_nodes);
        hipFree(d.d_gtiles);
      }
      hipFree(ex->d_children);
      hipFree(ex->d_ztiles);
      for (auto e : ex->ev_pre) hipEventDestroy(e);
      if (ex->ev_start) hipEventDestroy(ex->ev_start);
      if (ex->pre) hipStreamDestroy(ex->pre);
      delete ex;
    }
  }
  delete pl;
}

int spde_plan_get_info(const spde_plan* pl, spde_plan_info* info) {
  if (!pl || !info) {
    set_error("spde_plan_get_info: null argument");
    return SPDE_ERR_ARG;
  }
  info->n = pl->sym.n;
  info->nnz_struct = (int64_t)pl->st.indices.size();
  info->nnz_L = pl->sym.nnz_L;
  info->front_doubles = pl->lay_front;
  info->z_doubles = pl->lay_z;
  info->nnodes = (int64_t)pl->sym.nodes.size();
  info->nlevels = (int64_t)pl->sym.levels.size();
  info->max_front = pl->sym.max_front;
  info->max_p = pl->sym.max_p;
  info->flops_factor = pl->sym.flops_factor;
  info->flops_selinv = pl->sym.flops_selinv;
  info->split_doubles = pl->split_fs + pl->split_solve;
  return SPDE_OK;
}

int spde_plan_export(const spde_plan* pl, int64_t* indptr, int32_t* indices, uint8_t* code, int32_t* perm,
                     int32_t* nodes, int64_t* foff, int32_t* bnd, int32_t* relpos, int64_t* map) {
  if (!pl) {
    set_error("spde_plan_export: null plan");
    return SPDE_ERR_ARG;
  }
  const auto& st = pl->st;
  const auto& sym = pl->sym;
  if (indptr) std::memcpy(indptr, st.indptr.data(), st.indptr.size() * sizeof(int64_t));
  if (indices) std::memcpy(indices, st.indices.data(), st.indices.size() * sizeof(int32_t));
  if (code) std::memcpy(code, st.code.data(), st.code.size());
  if (perm) std::memcpy(perm, sym.perm.data(), sym.perm.size() * sizeof(int32_t));
  if (map) std::memcpy(map, pl->map.data(), pl->map.size() * sizeof(int64_t));
  for (size_t q = 0; q < sym.nodes.size(); ++q) {
    const Node& nd = sym.nodes[q];
    if (nodes) {
      int32_t* r = nodes + 8 * q;
      r[0] = nd.start;
      r[1] = nd.p;
      r[2] = nd.n();
      r[3] = nd.parent;
      r[4] = nd.child[0];
      r[5] = nd.child[1];
      r[6] = nd.level;
      r[7] = (int32_t)nd.B.size();
    }
    if (foff) foff[q] = nd.foff;
    for (size_t k = 0; k < nd.B.size(); ++k) {
      if (bnd) bnd[nd.relpos_off + k] = nd.B[k];
      if (relpos) relpos[nd.relpos_off + k] = nd.relpos.empty() ? -1 : nd.relpos[k];
    }
  }
  return SPDE_OK;
}

int spde_factor_async(spde_plan* pl, int slot, const double* qval, const double* diag_add, void* stream) {
  int rc = check_slot(pl, slot);
  if (rc) return rc;
  if (!qval) {
    set_error("spde_factor_async: null values");
    return SPDE_ERR_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  rc = ensure_slot(pl, slot, s);
  if (rc) return rc;
  Slot& sl = pl->slots[slot];
  const Symbolic& sym = pl->sym;
  PlanExtra* ex = extra(pl);
  rc = ensure_splitws(pl, slot);
  if (rc) return rc;
  hipLaunchKernelGGL(clear_status_kernel, dim3(1), dim3(64), 0, s, sl.status);
  launch_clear_flags(sl.flags, flag_words(pl), s);
  launch_zero_lower(pl->d_nodes, ex->d_ztiles, ex->nztiles, sl.front, s);
  launch_scatter(qval, pl->d_map, (int64_t)pl->st.indices.size(), sl.front, s);
  if (diag_add) launch_diag_add(diag_add, pl->d_diag, pl->d_map, sym.n, sl.front, s);
  Bases b = make_bases(pl, slot, nullptr);
  for (size_t l = 0; l < pl->levels.size(); ++l) {
    LevelPlan& L = pl->levels[l];
    launch_own_assemble(pl->d_nodes, L.d_owntiles, L.nowntiles, pl->d_pulls, pl->d_inv, sl.front, s);
    launch_front_factor(L.d_fronts, L.d_tasks, L.ntasks, sl.front, sl.z, sl.flags + 1 + pl->levels.size(),
                        sl.flags + 1 + l, sl.flags, sl.status, s);
    run_gemm(pl, L.syrk, b, s);
  }
  for (auto& g : pl->trtri) run_gemm(pl, g, b, s);
  launch_logdet(pl->d_diag, pl->d_map, sym.n, sl.front, sl.partial, sl.ld, s);
  SPDE_HIP(hipGetLastError());
  sl.stream = s;
  sl.factored = true;  // a non-positive pivot is reported by spde_factor_finish
  return SPDE_OK;
}

int spde_factor_finish(spde_plan* pl, int slot, double* logdet) {
  int rc = check_slot(pl, slot);
  if (rc) return rc;
  Slot& sl = pl->slots[slot];
  if (!sl.front) {  // (the stream may be the null stream)
    set_error("spde_factor_finish: no factorisation was enqueued in this slot");
    return SPDE_ERR_STATE;
  }
  int status = 0;
  double ld = 0.0;
  SPDE_HIP(hipMemcpyAsync(&status, sl.status, sizeof(int), hipMemcpyDeviceToHost, sl.stream));
  SPDE_HIP(hipMemcpyAsync(&ld, sl.ld, sizeof(double), hipMemcpyDeviceToHost, sl.stream));
  SPDE_HIP(hipStreamSynchronize(sl.stream));
  if (status != 0) {
    sl.factored = false;
    if (status == kStalled) {
      set_error("spde_factor: the factorisation stalled");
      return SPDE_ERR_HIP;
    }
    const int col = status - 1;
    set_error("spde_factor: matrix is not positive definite (pivot at lattice index " +
              std::to_string(pl->sym.perm[col]) + ")");
    return SPDE_ERR_NOT_SPD;
  }
  if (logdet) *logdet = ld;
  return SPDE_OK;
}

int spde_factor(spde_plan* pl, int slot, const double* qval, const double* diag_add, double* logdet, void* stream) {
  int rc = spde_factor_async(pl, slot, qval, diag_add, stream);
  if (rc) return rc;
  return spde_factor_finish(pl, slot, logdet);
}

int spde_solve(spde_plan* pl, int slot, int mode, double* B, int nrhs, int64_t ldb, void* stream) {
  int rc = check_slot(pl, slot);
  if (rc) return rc;
  if (!B || nrhs <= 0 || ldb < pl->sym.n || mode < 0 || mode > SPDE_SOLVE_LT_NOPERM) {
    set_error("spde_solve: invalid argument");
    return SPDE_ERR_ARG;
  }
  if (mode == SPDE_SOLVE_P || mode == SPDE_SOLVE_PT) {
    // the permutation alone: no factor needed, the slot's staging buffer only
    Slot& sl = pl->slots[slot];
    const int64_t n = pl->sym.n;
    if (sl.xy_cap < n * nrhs) {
      SPDE_HIP(hipDeviceSynchronize());
      hipFree(sl.xy);
      sl.xy = nullptr;
      sl.xy_cap = 0;
      SPDE_HIP(hipMalloc((void**)&sl.xy, sizeof(double) * n * nrhs));
      sl.xy_cap = n * nrhs;
    }
    hipStream_t s = (hipStream_t)stream;
    if (mode == SPDE_SOLVE_P) {
      launch_permute_in(B, ldb, pl->d_perm, n, nrhs, sl.xy, s);
      SPDE_HIP(hipMemcpy2DAsync(B, ldb * sizeof(double), sl.xy, n * sizeof(double), n * sizeof(double), nrhs,
                                hipMemcpyDeviceToDevice, s));
    } else {
      SPDE_HIP(hipMemcpy2DAsync(sl.xy, n * sizeof(double), B, ldb * sizeof(double), n * sizeof(double), nrhs,
                                hipMemcpyDeviceToDevice, s));
      launch_permute_out(sl.xy, pl->d_perm, n, nrhs, B, ldb, s);
    }
    return SPDE_OK;
  }
  if (!pl->slots[slot].factored) {
    set_error("spde_solve: slot not factored");
    return SPDE_ERR_STATE;
  }
  const int most = solve_columns(pl->sym.n);
  if (nrhs > most) {
    for (int c = 0; c < nrhs; c += most)
      if ((rc = spde_solve(pl, slot, mode, B + c * ldb, std::min(most, nrhs - c), ldb, stream))) return rc;
    return SPDE_OK;
  }
  hipStream_t s = (hipStream_t)stream;
  PlanExtra* ex = extra(pl);
  const Symbolic& sym = pl->sym;
  const int64_t n = sym.n;
  Slot& sl = pl->slots[slot];
  if (pl->solve_nrhs != nrhs && pl->solve_cache.count(nrhs)) {
    // launch lists of this nrhs exist (their descriptors never change): swap them in
    rc = build_solve_plan(pl, nrhs);
    if (rc) return rc;
  }
  if (sl.vec_cap < sym.vec_doubles * nrhs || sl.xy_cap < n * nrhs || pl->solve_nrhs != nrhs) {
    // buffers change or new launch lists are built: let every stream drain first
    SPDE_HIP(hipDeviceSynchronize());
    if (sl.vec_cap < sym.vec_doubles * nrhs) {
      hipFree(sl.vec);
      sl.vec = nullptr;
      sl.vec_cap = 0;
      SPDE_HIP(hipMalloc((void**)&sl.vec, sizeof(double) * sym.vec_doubles * nrhs));
      sl.vec_cap = sym.vec_doubles * nrhs;
    }
    if (sl.xy_cap < n * nrhs) {
      hipFree(sl.xy);
      sl.xy = nullptr;
      sl.xy_cap = 0;
      SPDE_HIP(hipMalloc((void**)&sl.xy, sizeof(double) * n * nrhs));
      sl.xy_cap = n * nrhs;
    }
    if (pl->solve_nrhs != nrhs) {
      rc = build_solve_plan(pl, nrhs);
      if (rc) return rc;
    }
  }
  rc = ensure_splitws(pl, slot);
  if (rc) return rc;
  Bases b = make_bases(pl, slot, sl.xy);
  const int nl = (int)pl->levels.size();
  // in: P B for modes A and L; B as it is (already in elimination order) for the others
  const bool perm_in = mode == SPDE_SOLVE_A || mode == SPDE_SOLVE_L;
  // out: P^T X for modes A and LT; X in elimination order for L and the unpermuted modes
  const bool perm_out = mode == SPDE_SOLVE_A || mode == SPDE_SOLVE_LT;
  const bool fwd = mode == SPDE_SOLVE_A || mode == SPDE_SOLVE_L || mode == SPDE_SOLVE_L_NOPERM;
  const bool bwd = mode == SPDE_SOLVE_A || mode == SPDE_SOLVE_LT || mode == SPDE_SOLVE_LT_NOPERM;
  if (perm_in) {
    launch_permute_in(B, ldb, pl->d_perm, n, nrhs, sl.xy, s);
  } else {
    SPDE_HIP(hipMemcpy2DAsync(sl.xy, n * sizeof(double), B, ldb * sizeof(double), n * sizeof(double), nrhs,
                              hipMemcpyDeviceToDevice, s));
  }
  if (fwd) {
    for (int l = 0; l < nl; ++l) {
      LevelPlan& L = pl->levels[l];
      launch_fwd_gather(ex->lvl[l].d_nodes, ex->lvl[l].nn, pl->d_nodes, ex->d_children, pl->d_relpos, sl.xy, n,
                        nrhs, sl.vec, s);
      run_gemm(pl, L.fwd_y, b, s);
      run_gemm(pl, L.fwd_u, b, s);
    }
  }
  if (bwd) {
    for (int l = nl - 1; l >= 0; --l) {
      LevelPlan& L = pl->levels[l];
      launch_bwd_gather(ex->lvl[l].d_nodes, ex->lvl[l].nn, pl->d_nodes, pl->d_bnd, sl.xy, n, nrhs, sl.vec, s);
      run_gemm(pl, L.bwd_t, b, s);
      run_gemm(pl, L.bwd_x, b, s);
    }
  }
  if (perm_out) {
    launch_permute_out(sl.xy, pl->d_perm, n, nrhs, B, ldb, s);
  } else {
    SPDE_HIP(hipMemcpy2DAsync(B, ldb * sizeof(double), sl.xy, n * sizeof(double), n * sizeof(double), nrhs,
                              hipMemcpyDeviceToDevice, s));
  }
  return SPDE_OK;
}

int spde_prof_begin(spde_plan* pl) { return spde_prof_begin_kinds(pl, 0xff); }

int spde_prof_begin_kinds(spde_plan* pl, int kind_mask) {
  if (!pl || pl->host_only || kind_mask <= 0 || kind_mask > 0xff) {
    set_error("spde_prof_begin: no device plan or empty kind mask");
    return SPDE_ERR_ARG;
  }
  pl->prof_mask = kind_mask;
  if (!pl->prof_base) SPDE_HIP(hipEventCreate(&pl->prof_base));
  SPDE_HIP(hipDeviceSynchronize());
  SPDE_HIP(hipEventRecord(pl->prof_base, nullptr));
  SPDE_HIP(hipEventSynchronize(pl->prof_base));
  pl->prof_on = true;
  pl->prof_n = 0;
  return SPDE_OK;
}

int spde_prof_dump(spde_plan* pl, double* ms, double* flops, double* bytes, int32_t* kind, int32_t* tiles, int64_t cap,
                   int64_t* count) {
  if (!pl || pl->host_only) {
    set_error("spde_prof_dump: no device plan");
    return SPDE_ERR_ARG;
  }
  if (pl->prof_n) SPDE_HIP(hipDeviceSynchronize());  // launches may sit on several streams
  const int64_t n = std::min<int64_t>(cap, (int64_t)pl->prof_n);
  for (int64_t i = 0; i < n; ++i) {
    float t = 0.0f;
    SPDE_HIP(hipEventElapsedTime(&t, pl->prof_ev[2 * i], pl->prof_ev[2 * i + 1]));
    if (ms) ms[i] = t;
    if (flops) flops[i] = pl->prof_flops[i];
    if (bytes) bytes[i] = pl->prof_bytes[i];
    if (kind) kind[i] = pl->prof_kind[i];
    if (tiles) tiles[i] = pl->prof_tiles[i];
  }
  if (count) *count = (int64_t)pl->prof_n;
  return SPDE_OK;
}

int spde_prof_end(spde_plan* pl, double* gemm_ms, double* gemm_flops, int64_t* launches, double* busy_ms,
                  double* gemm_bytes) {
  if (!pl || pl->host_only) {
    set_error("spde_prof_end: no device plan");
    return SPDE_ERR_ARG;
  }
  pl->prof_on = false;
  double ms = 0.0, fl = 0.0, by = 0.0;
  if (pl->prof_n) SPDE_HIP(hipDeviceSynchronize());  // launches may sit on several streams
  std::vector<std::pair<float, float>> iv(pl->prof_n);
  for (size_t i = 0; i < pl->prof_n; ++i) {
    float t = 0.0f, a = 0.0f, b = 0.0f;
    SPDE_HIP(hipEventElapsedTime(&t, pl->prof_ev[2 * i], pl->prof_ev[2 * i + 1]));
    SPDE_HIP(hipEventElapsedTime(&a, pl->prof_base, pl->prof_ev[2 * i]));
    SPDE_HIP(hipEventElapsedTime(&b, pl->prof_base, pl->prof_ev[2 * i + 1]));
    iv[i] = {a, b};
    ms += t;
    fl += pl->prof_flops[i];
    by += pl->prof_bytes[i];
  }
  // time during which at least one GEMM launch was in flight (launches on
  // different streams overlap)
  std::sort(iv.begin(), iv.end());
  double busy = 0.0, cur_a = 0.0, cur_b = -1.0;
  for (auto& p : iv) {
    if (p.first > cur_b) {
      if (cur_b > cur_a) busy += cur_b - cur_a;
      cur_a = p.first;
      cur_b = p.second;
    } else if (p.second > cur_b) {
      cur_b = p.second;
    }
  }
  if (cur_b > cur_a) busy += cur_b - cur_a;
  if (gemm_ms) *gemm_ms = ms;
  if (gemm_flops) *gemm_flops = fl;
  if (launches) *launches = (int64_t)pl->prof_n;
  if (busy_ms) *busy_ms = busy;
  if (gemm_bytes) *gemm_bytes = by;
  pl->prof_n = 0;
  return SPDE_OK;
}

int spde_selinv(spde_plan* pl, int slot, double* sigma, void* stream) {
  int rc = check_slot(pl, slot);
  if (rc) return rc;
  if (!pl->slots[slot].factored) {
    set_error("spde_selinv: slot not factored");
    return SPDE_ERR_STATE;
  }
  hipStream_t s = (hipStream_t)stream;
  PlanExtra* ex = extra(pl);
  const Symbolic& sym = pl->sym;
  Slot& sl = pl->slots[slot];
  if (!sl.sigma) {
    SPDE_HIP(hipStreamSynchronize(s));
    SPDE_HIP(hipMalloc((void**)&sl.sigma, sizeof(double) * std::max<int64_t>(pl->lay_front, 1)));
  }
  if (!pl->selinv_built) {
    rc = build_selinv_plan(pl);
    if (rc) return rc;
  }
  rc = ensure_splitws(pl, slot);
  if (rc) return rc;
  if (!ex->pre) {
    SPDE_HIP(hipStreamCreateWithFlags(&ex->pre, hipStreamNonBlocking));  // default priority
    SPDE_HIP(hipEventCreateWithFlags(&ex->ev_start, hipEventDisableTiming));
    ex->ev_pre.resize(pl->levels.size());
    for (auto& e : ex->ev_pre) SPDE_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  }
  Bases b = make_bases(pl, slot, nullptr);
  // Top-down over the levels.  X = L21 Z and Sigma11 = Z^T Z need only the
  // factor: they run on the second stream, one level ahead of the chain
  // gather -> Sigma21 = -Sigma22 X -> Sigma11 -= X^T Sigma21 on this one,
  // which waits for its level's event.  Every wait is enqueued right after
  // the record it waits on.
  SPDE_HIP(hipEventRecord(ex->ev_start, s));
  SPDE_HIP(hipStreamWaitEvent(ex->pre, ex->ev_start, 0));
  for (int l = (int)pl->levels.size() - 1; l >= 0; --l) {
    LevelPlan& L = pl->levels[l];
    LevelDev& D = ex->lvl[l];
    for (const GemmLaunch* g : {&L.si_x, &L.si_s11a}) run_gemm(pl, *g, b, ex->pre, g->tile == 128 ? 0 : kPreLds);
    SPDE_HIP(hipEventRecord(ex->ev_pre[l], ex->pre));
    launch_sigma_gather(D.d_nodes, pl->d_nodes, pl->d_relpos, sl.sigma, D.d_gtiles, D.ngtiles, s);
    SPDE_HIP(hipStreamWaitEvent(s, ex->ev_pre[l], 0));
    run_gemm(pl, L.si_s21, b, s);
    run_gemm(pl, L.si_s11b, b, s);
  }
  if (sigma) launch_gather_pattern(sl.sigma, pl->d_mapsym, (int64_t)pl->st.indices.size(), sigma, s);
  return SPDE_OK;
}

}  // extern "C"
