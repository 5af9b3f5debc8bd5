// Internal plan object shared by the HIP translation units.
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <map>
#include <vector>

#include "../../include/spdepy_amd.h"
#include "plan.hpp"

namespace spde {

void set_error(const std::string& msg);

#define SPDE_HIP(call)                                                        \
  do {                                                                        \
    hipError_t e_ = (call);                                                   \
    if (e_ != hipSuccess) {                                                   \
      ::spde::set_error(std::string(#call) + ": " + hipGetErrorString(e_));   \
      return SPDE_ERR_HIP;                                                    \
    }                                                                         \
  } while (0)

constexpr int NB = 64;  // diagonal block width of the dense partial factorisation
constexpr int kTmpl = 143;  // per-cell assembly template (doubles)

// Operand base pointers of a batched launch (selected per operand by id).
enum Base : int8_t { kFront = 0, kZ = 1, kSigma = 2, kWork = 3, kVec = 4, kX = 5, kNumBases = 6 };
// Update blocks of a front's children, read where the front's entries are
// formed: u: offset of child s's update block, inv + i: row of that block which is
// row i of this (padded) front, -1 if none (a missing child has -1 throughout).
struct Pull {
  int64_t u[2], inv[2];
  int32_t cld[2];
};
// Entry (i, j), i >= j, of a front: s plus the children's update blocks (the
// extend-add), first child first, formed where it is used.  i0, i1 and j0, j1: its
// row and column in the children (child_row); relpos increases, so the child's
// entry is in its lower triangle too.
// Without branches, so that the loads of many entries are in flight together:
// an entry that a child does not have reads F[0] and adds zero.
__device__ __forceinline__ double assembled(const double* F, double s, const Pull& q, int i0, int i1, int j0, int j1) {
  const bool h0 = (i0 | j0) >= 0, h1 = (i1 | j1) >= 0;
  const double u0 = F[h0 ? q.u[0] + i0 + (int64_t)j0 * q.cld[0] : 0];
  const double u1 = F[h1 ? q.u[1] + i1 + (int64_t)j1 * q.cld[1] : 0];
  s = h0 ? s + u0 : s;
  return h1 ? s + u1 : s;
}
__device__ __forceinline__ int child_row(const int32_t* inv, const Pull& q, int s, int i) { return inv[q.inv[s] + i]; }
struct Bases {
  double* p[kNumBases];
  double* ws;  // split-K partial tiles of the slot
  const Pull* pulls;
  const int32_t* inv;
};

// One GEMM problem: C = alpha op(A) op(B) + beta C, column-major.
struct GemmProb {
  int64_t a_off, b_off, c_off;
  int32_t lda, ldb, ldc;
  int32_t M, N, K;
  int8_t a_base, b_base, c_base, lower;
  // triangular operand, zeros skipped: 1 op(B) lower (k >= first column of
  // the tile), 2 op(A) upper (k >= first row), 3 op(A) lower (k < last row + 1)
  int8_t kmode;
  int32_t pull;     // launches with `pull`: entry of Bases::pulls added to C
  int32_t pull_row; // front row of C's first row and column
  double alpha, beta;
};
struct GemmTile {
  int32_t prob, tm, tn, pad;
};

// A batched GEMM launch: problems + tile list (device), transposition flags.
struct GemmLaunch {
  bool ta = false, tb = false;
  int tile = 64;                 // longer edge of a block tile (64 or 128), chosen when finalised
  int tile_m() const { return tile == 128 && ta && tb ? 64 : tile; }  // rows and columns of a tile
  int tile_n() const { return tile == 128 && !ta ? 64 : tile; }
  bool vec = false;              // operands with contiguous k: even offsets and leading dimensions (16-byte loads)
  int ntiles = 0, nprobs = 0;
  GemmProb* d_probs = nullptr;
  GemmTile* d_tiles = nullptr;
  std::vector<GemmProb> h_probs;
  std::vector<GemmTile> h_tiles;
  double flops = 0;
  double bytes = 0;   // algorithmic HBM bytes: A, B, C read once (C only if beta != 0), C written once
  // split-K (few tiles, deep K): each tile's K range is cut into `split`
  // chunks computed by separate blocks into partial tiles at ws + ws_off (in
  // the slot's split workspace), summed in chunk order by a second kernel
  int split = 1;
  int64_t ws_off = 0;
  // few right-hand sides (N <= kGemvMaxN, op(B) = B, general C): a
  // bandwidth-bound kernel reading A once instead of 64-wide MFMA tiles
  bool pull = false;             // the children's update blocks are added to C (level SYRK)
  bool gemv = false;
  bool gemv_wide = false;        // narrow launch with deep K: sixteen waves share each row block's K range
};
// One column only: at 100x100x20 a full solve takes 2.5 ms with the
// bandwidth-bound kernel for one right-hand side, but from two right-hand
// sides on the MFMA tiles are faster (3.2 ms for two, 4.9 ms for eight,
// against 3.8 and 10.6 ms with the per-column kernel).
constexpr int kGemvMaxN = 1;

struct FrontDesc {      // one front of a level's factorisation
  int64_t foff, zoff;
  int32_t ld, pp, p, nrows;  // nrows = pp + boundary rows
  int32_t R, P;         // row tiles and own column tiles of 64
  int32_t flag0;        // counter of tile (i, k): flag0 + k R + i
  int32_t colbase;      // elimination column of the first own column
};
constexpr int kStalled = -1;  // status of a factorisation whose waits gave up
struct FrontTask {      // i = j: the diagonal block j; else tiles (i, j), (i + 1, j)
  int32_t front, j, i, pad;
};
struct LevelPlan {
  std::vector<int> nodes;
  // lower 64x64 tiles (node, ti, tj) of the own columns of fronts with children
  int4* d_owntiles = nullptr;
  int nowntiles = 0;
  // factorisation of the own columns: fronts and tasks in ticket order
  FrontDesc* d_fronts = nullptr;
  FrontTask* d_tasks = nullptr;
  int ntasks = 0;
  GemmLaunch syrk;
  // solves / selinv
  GemmLaunch fwd_y, fwd_u, bwd_t, bwd_x;   // the current nrhs' launches (owned by solve_cache)
  GemmLaunch si_x, si_s21, si_s11a, si_s11b;
};

struct Slot {
  double* front = nullptr;  // factor fronts
  double* z = nullptr;      // inverses of the diagonal blocks of L
  double* sigma = nullptr;  // selected-inverse fronts (allocated on first use)
  double* work = nullptr;   // inverse-of-L11 temporaries
  double* partial = nullptr;  // log-det partial sums per 256 variables
  double* ld = nullptr;     // device log-det
  int* status = nullptr;    // first non-positive pivot (elimination column + 1)
  int* flags = nullptr;     // factorisation: stop flag, a ticket counter per level, tile counters
  double* vec = nullptr;    // solve front vectors
  int64_t vec_cap = 0;      // in doubles
  double* xy = nullptr;     // elimination-ordered solve buffer
  int64_t xy_cap = 0;
  hipStream_t stream = nullptr;  // stream of the last factorisation
  bool factored = false;
  double* splitws = nullptr;  // split-K partial tiles: [factor + selected inverse | solve] regions
  int64_t splitws_cap = 0;
};

struct NodeDev {            // per-node table on the device
  int64_t foff, zoff, voff, relpos_off;  // foff, zoff: device layout
  int32_t start, p, n, parent, nb, level, ld, pp;
};

// Device layout of one front and its Z: the own columns are padded to pp (a
// multiple of kFrontPad), the boundary rows and columns follow at pp, and the
// leading dimension is a multiple of 16 doubles, so that every block of a
// front starts on a 128-byte line: fragment loads touch whole lines, operands
// with contiguous k are read 16 bytes at a time, and no two 64-row tiles
// share a line.  The symbolic analysis and the exported plan keep the compact
// n x n fronts.  (The pad rows and columns hold zeros or values nothing reads.)
struct FrontLay {
  int64_t foff, zoff;
  int32_t ld, pp;
};
constexpr int kFrontPad = 64;

}  // namespace spde

struct spde_plan {
  spde::Lattice lat;
  spde::Structure st;
  spde::Symbolic sym;
  std::vector<int64_t> map;      // scatter map (front offsets, -1 upper)

  bool host_only = true;
  int nslots = 0;
  // device structure
  int64_t* d_indptr = nullptr;
  int32_t* d_indices = nullptr;
  uint8_t* d_code = nullptr;
  int64_t* d_diag = nullptr;
  int64_t* d_map = nullptr;
  int64_t* d_mapsym = nullptr;
  int32_t* d_perm = nullptr;
  int32_t* d_relpos = nullptr;
  int32_t* d_bnd = nullptr;       // concatenated boundary lists (elimination indices)
  spde::NodeDev* d_nodes = nullptr;
  spde::Pull* d_pulls = nullptr;  // per node
  int32_t* d_inv = nullptr;
  double* d_tmpl = nullptr;       // per-cell value templates of the blocks of Q
  double* d_acan = nullptr;       // canonical 9-point spatial operator A
  double* d_a0can = nullptr;      // canonical 9-point initial-state operator A0
  double* d_qdiag = nullptr;      // diagonal of Qs per cell
  double* d_win = nullptr;        // per-cell gradient windows
  double* d_red = nullptr;        // one device scalar (reductions)
  int32_t* d_pos25 = nullptr;     // one-slice plans: entry index of (cell, 5x5 code), -1 if absent
  int64_t split_fs = 0;           // split-K workspace (doubles) of the factor and selected-inverse launches
  int64_t split_solve = 0;        // ... of the solve launches (current nrhs)
  double* d_gpart = nullptr;      // per (cell, slice) partial windows of the gradient reduction
  void* llws = nullptr;           // buffers and side stream of spde_loglik_grad (loglik.hip)
  void* extra = nullptr;          // device launch lists of the factor and selected inverse (numeric.hip)
  double* d_tan = nullptr;        // tangent assembly: templates + dA, dA0, dq of one direction
  int32_t* d_sprow = nullptr;     // one-slice plans: row and column of each entry (Kronecker kernels)
  int32_t* d_spcol = nullptr;
  int64_t work_doubles = 0;       // per-slot workspace size
  std::vector<spde::FrontLay> lay;  // device layout per node
  int nflags = 0;                   // tile counters of the factorisation (all levels)
  int64_t lay_front = 0, lay_z = 0;  // arena sizes (doubles) of that layout
  std::vector<spde::Slot> slots;
  std::vector<spde::LevelPlan> levels;
  std::vector<spde::GemmLaunch> trtri;  // per recursion height: pairs (X, Z2)
  int trtri_heights = 0;
  int solve_nrhs = -1;            // nrhs the solve launches are built for
  // solve launches per nrhs (four per level), built once each and swapped in
  // by value; their device descriptor arrays are freed with the plan
  struct SolveSet {
    std::vector<spde::GemmLaunch> launches;
    int64_t split = 0;
  };
  std::map<int, SolveSet> solve_cache;
  bool selinv_built = false;
  // optional event timing of the GEMM launches (measurement only)
  bool prof_on = false;
  int prof_mask = 0xff;           // kinds of GEMM launch timed (bit = kind code)
  std::vector<hipEvent_t> prof_ev;
  hipEvent_t prof_base = nullptr;
  std::vector<double> prof_flops;
  std::vector<double> prof_bytes;
  std::vector<int> prof_tiles;
  std::vector<int> prof_kind;
  size_t prof_n = 0;
  hipStream_t prof_stream = nullptr;
};
