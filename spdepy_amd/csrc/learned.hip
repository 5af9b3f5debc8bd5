// Learned preconditioner network: a 4-layer 3x3 convolutional network over
// the time slices of the lattice (input 8 channels = 7 stencil coefficients +
// 0, hidden 32 channels, output 32 channels of which 22 are the correction of
// the incomplete Cholesky factor), BF16 operands with FP32 accumulation on
// the CDNA matrix cores (v_mfma_f32_16x16x16_bf16), and its training
// kernels: backward data, weight and bias gradients, Adam.  No reference
// counterpart (the reference has no iterative solver); the correction it
// produces is applied by spde_ic_correct.
//
// Layouts.  Activations: pixel-major (NHWC), pixel p = x + M (y + N t), the
// channels of a pixel contiguous (FP32).  Master weights per layer: W[k][co]
// FP32 row-major with k = tap * cin + ci, tap = 3 (dy + 1) + (dx + 1), and
// bias[32].  The matrix-core operand of a layer is packed once per update as
// BF16 fragments: frag[((kc * 2 + h) * 64 + lane) * 4 + j] =
// W[16 kc + 4 (lane / 16) + j][16 h + lane % 16] (zero for k >= 9 cin), the B
// operand of the 16x16x16 instruction for k-chunk kc and output half h.
//
// A wave's tiles are 16 pixels x 32 channels: A rows are pixels (lane % 16), A
// k-columns 4 (lane / 16) + j; D rows 4 (lane / 16) + j, columns lane % 16.
#include <hip/hip_runtime.h>

#include <cmath>
#include <string>

#include "internal.hpp"

namespace spde {

typedef short bf16x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kCh = 32;  // hidden and padded output channels

// float -> bf16, round to nearest even (finite inputs)
__device__ __host__ inline unsigned short to_bf16(float f) {
  unsigned u;
  __builtin_memcpy(&u, &f, 4);
  u += 0x7FFFu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}

// A block works on patches of one time slice, kTx x TY pixels; the patch and its
// one-pixel border are staged in LDS once as BF16 (masked on the way), so that
// an activation is read from memory about 1.4 times instead of nine and converted
// as often.  Pixel-major, the channels of a pixel contiguous, 8 bytes of padding a
// pixel (the sixteen pixels of a fragment fall on different banks).
constexpr int kTx = 16;
typedef float f4u __attribute__((ext_vector_type(4), aligned(4)));

template <int CIN>
constexpr int patch_pitch = CIN + 4;  // halves per pixel

// Loads rows [y0 - B, y0 + TY + B) and columns [x0 - B, x0 + kTx + B) of slice t,
// zero outside, masked by mask > 0.  SUM: adds the thread's values to sum (its
// channels 4 (thread % (CIN / 4)) .. + 3).
template <int CIN, int TY, int B, int NT, bool SUM>
__device__ __forceinline__ void load_patch(unsigned short* __restrict__ lds, const float* __restrict__ in,
                                           const float* __restrict__ mask, int M, int N, int64_t t, int x0, int y0,
                                           float (&sum)[4]) {
  constexpr int W = kTx + 2 * B, H = TY + 2 * B, C4 = CIN / 4, total = W * H * C4;
#pragma unroll 4
  for (int c = threadIdx.x; c < total; c += NT) {
    const int pix = c / C4, part = c - pix * C4;
    const int py = pix / W, px = pix - py * W;
    const int x = x0 - B + px, y = y0 - B + py;
    f4u v = {0.f, 0.f, 0.f, 0.f};
    if (x >= 0 && x < M && y >= 0 && y < N) {
      const int64_t q = ((t * N + y) * (int64_t)M + x) * CIN + 4 * part;
      v = *(const f4u*)(in + q);
      if (mask) {
        const f4u k = *(const f4u*)(mask + q);
#pragma unroll
        for (int j = 0; j < 4; ++j) v[j] = k[j] > 0.f ? v[j] : 0.f;
      }
    }
    bf16x4 h;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      h[j] = (short)to_bf16(v[j]);
      if (SUM) sum[j] += v[j];
    }
    *(bf16x4*)(lds + pix * patch_pitch<CIN> + 4 * part) = h;
  }
}

// Convolution of one layer.  in: P x CIN; mask (optional, P x CIN): the input
// is in * (mask > 0) (backward data through a ReLU); out: P x 32, out = act(D +
// bias) with act ReLU when relu, bias optional.  Each of the four waves takes two
// rows of the 16 x 8 patch, 16 pixels x 32 channels per row.  HBM-bound (77 MB for
// 200,000 pixels and 32 channels with a mask): per-lane gathers of the fragments from
// memory took 186 us for it.
template <int CIN>
__global__ __launch_bounds__(256) void conv_kernel(int M, int N, int nx, int ny, const float* __restrict__ in,
                                                   const float* __restrict__ mask,
                                                   const unsigned short* __restrict__ frag,
                                                   const float* __restrict__ bias, int relu, float* __restrict__ out) {
  constexpr int TY = 8, W = kTx + 2, PP = patch_pitch<CIN>, nk = (9 * CIN + 15) / 16;
  __shared__ __align__(16) unsigned short patch[W * (TY + 2) * PP];
  const int64_t t = blockIdx.x / (nx * ny);
  const int r = (int)(blockIdx.x - t * (nx * ny));
  const int x0 = (r % nx) * kTx, y0 = (r / nx) * TY;
  float none[4];
  load_patch<CIN, TY, 1, 256, false>(patch, in, mask, M, N, t, x0, y0, none);
  __syncthreads();
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int px = lane & 15, kq = lane >> 4;
  f32x4 acc[2][2];
#pragma unroll
  for (int y = 0; y < 2; ++y)
#pragma unroll
    for (int h = 0; h < 2; ++h) acc[y][h] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int kc = 0; kc < nk; ++kc) {
    const int k0 = 16 * kc + 4 * kq;
    const int tap = k0 / CIN, ci = k0 - tap * CIN;
    const int dx = tap % 3, dy = tap / 3;
    const bf16x4 b0 = *(const bf16x4*)(frag + ((int64_t)(kc * 2 + 0) * 64 + lane) * 4);
    const bf16x4 b1 = *(const bf16x4*)(frag + ((int64_t)(kc * 2 + 1) * 64 + lane) * 4);
#pragma unroll
    for (int y = 0; y < 2; ++y) {
      bf16x4 a = {0, 0, 0, 0};
      if (tap < 9) a = *(const bf16x4*)(patch + ((2 * wave + y + dy) * W + px + dx) * PP + ci);
      acc[y][0] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b0, acc[y][0], 0, 0, 0);
      acc[y][1] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b1, acc[y][1], 0, 0, 0);
    }
  }
  const int co = lane & 15;
#pragma unroll
  for (int y = 0; y < 2; ++y) {
    const int gy = y0 + 2 * wave + y;
    if (gy >= N) continue;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int gx = x0 + 4 * kq + j;
      if (gx >= M) continue;
      float v0 = acc[y][0][j] + (bias ? bias[co] : 0.f), v1 = acc[y][1][j] + (bias ? bias[co + 16] : 0.f);
      if (relu) {
        v0 = v0 > 0.f ? v0 : 0.f;
        v1 = v1 > 0.f ? v1 : 0.f;
      }
      float* o = out + ((t * N + gy) * (int64_t)M + gx) * kCh;
      o[co] = v0;
      o[co + 16] = v1;
    }
  }
}

// Partial weight and bias gradients of a block's patches (patch b, b + blocks,
// .. in order): wpart[block][k][co] = sum_p X[p + off(tap)][ci] dZ[p][co] and
// bpart[block][co] = sum_p dZ[p][co] with dZ = G (G * (Y > 0) when Y), the operands
// of the product rounded to BF16 as in the forward pass, the bias in FP32.  The
// contraction runs over pixels: both fragments are gathered from the staged
// patches, four pixels of a row to a lane; the 2 * 18 tiles of 16 x 16 weights are
// spread over the eight waves and stay in registers.  (One wave per chunk and tile,
// gathering from memory, took 301 us and the bias another 308.)
template <int CIN>
__global__ __launch_bounds__(512) void conv_wgrad_kernel(int M, int N, int nx, int ny, int npatch,
                                                         const float* __restrict__ X, const float* __restrict__ G,
                                                         const float* __restrict__ Y, float* __restrict__ wpart,
                                                         float* __restrict__ bpart) {
  constexpr int TY = 8, W = kTx + 2, PP = patch_pitch<CIN>, PG = patch_pitch<kCh>, nkt = (9 * CIN + 15) / 16;
  constexpr int NTILE = 2 * nkt, PER = (NTILE + 7) / 8;
  __shared__ __align__(16) unsigned short xs[W * (TY + 2) * PP];
  __shared__ __align__(16) unsigned short gs[kTx * TY * PG];
  __shared__ float bs[512 * 4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int lr = lane & 15, kq = lane >> 4;
  f32x4 acc[PER];
#pragma unroll
  for (int q = 0; q < PER; ++q) acc[q] = f32x4{0.f, 0.f, 0.f, 0.f};
  float bsum[4] = {0.f, 0.f, 0.f, 0.f}, none[4];
  for (int b = blockIdx.x; b < npatch; b += gridDim.x) {
    const int64_t t = b / (nx * ny);
    const int r = (int)(b - t * (nx * ny));
    const int x0 = (r % nx) * kTx, y0 = (r / nx) * TY;
    __syncthreads();
    load_patch<CIN, TY, 1, 512, false>(xs, X, nullptr, M, N, t, x0, y0, none);
    load_patch<kCh, TY, 0, 512, true>(gs, G, Y, M, N, t, x0, y0, bsum);
    __syncthreads();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int tile = wave + 8 * q;  // k-tile * 2 + column half
      if (tile >= NTILE) break;
      const int krow = 16 * (tile >> 1) + lr, h = tile & 1;
      const int tap = krow / CIN, ci = krow - tap * CIN;
      const bool in = tap < 9;
      const unsigned short* xp = xs + (in ? ((tap / 3) * W + tap % 3) * PP + ci : 0);
      const unsigned short* gp = gs + 16 * h + lr;
#pragma unroll
      for (int y = 0; y < TY; ++y) {
        bf16x4 a, c;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          a[j] = in ? (short)xp[(y * W + 4 * kq + j) * PP] : (short)0;
          c[j] = (short)gp[(y * kTx + 4 * kq + j) * PG];
        }
        acc[q] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, c, acc[q], 0, 0, 0);
      }
    }
  }
  // D rows (k) 4 kq + j, column lane & 15
#pragma unroll
  for (int q = 0; q < PER; ++q) {
    const int tile = wave + 8 * q;
    if (tile >= NTILE) break;
    float* dst = wpart + ((int64_t)blockIdx.x * (nkt * 16) + 16 * (tile >> 1) + 4 * kq) * kCh + 16 * (tile & 1) + lr;
#pragma unroll
    for (int j = 0; j < 4; ++j) dst[j * kCh] = acc[q][j];
  }
  // thread's channels 4 (thread % 8) .. + 3: summed over the threads in order
#pragma unroll
  for (int j = 0; j < 4; ++j) bs[threadIdx.x * 4 + j] = bsum[j];
  __syncthreads();
  if (threadIdx.x < kCh) {
    float v = 0.f;
    for (int q = 0; q < 64; ++q) v += bs[q * 32 + threadIdx.x];
    bpart[(int64_t)blockIdx.x * kCh + threadIdx.x] = v;
  }
}

// dW[e] = sum over chunks of wpart[c][e], db likewise, in a fixed order: four
// threads take a quarter of the chunks each, 64 entries to a block.
__global__ __launch_bounds__(256) void chunk_sum_kernel(int nchunk, int64_t width, int64_t wstride,
                                                        const float* __restrict__ wpart,
                                                        const float* __restrict__ bpart, float* __restrict__ dW,
                                                        float* __restrict__ db) {
  __shared__ float red[4][64];
  const int l = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int64_t e = blockIdx.x * 64ll + l;
  const int q = (nchunk + 3) / 4, c0 = g * q, c1 = min(nchunk, c0 + q);
  const bool w = e < width, in = e < width + kCh;
  const float* src = w ? wpart + e : bpart + (e - width);
  const int64_t stride = w ? wstride : kCh;
  float s = 0.f;
  if (in) {
#pragma unroll 8
    for (int c = c0; c < c1; ++c) s += src[c * stride];
  }
  red[g][l] = s;
  __syncthreads();
  if (g == 0 && in) {
    const float v = ((red[0][l] + red[1][l]) + red[2][l]) + red[3][l];
    if (w)
      dW[e] = v;
    else
      db[e - width] = v;
  }
}

// BF16 fragments of the forward operand (transposed = 0) or of the
// backward-data operand (transposed = 1: W'[tap' * 32 + co][ci] =
// W[(8 - tap') * cin + ci][co], output channels ci, padded to 32).
__global__ void pack_kernel(int cin, int transposed, const float* __restrict__ W, unsigned short* __restrict__ frag) {
  const int kin = transposed ? 9 * kCh : 9 * cin;  // k extent of the packed operand
  const int nk = (kin + 15) / 16;
  const int e = blockIdx.x * blockDim.x + threadIdx.x;
  if (e >= nk * 2 * 64 * 4) return;
  const int j = e & 3, lane = (e >> 2) & 63, h = (e >> 8) & 1, kc = e >> 9;
  const int k = 16 * kc + 4 * (lane >> 4) + j;
  const int col = 16 * h + (lane & 15);
  float v = 0.f;
  if (k < kin) {
    if (!transposed) {
      v = W[(int64_t)k * kCh + col];
    } else {
      const int tp = k / kCh, co = k - tp * kCh;  // packed row = (tap', co); packed column = ci
      if (col < cin) v = W[(int64_t)((8 - tp) * cin + col) * kCh + co];
    }
  }
  frag[e] = to_bf16(v);
}

// Adam on FP32 parameters: m = b1 m + (1 - b1) g; v = b2 v + (1 - b2) g^2;
// theta -= lr (m / (1 - b1^t)) / (sqrt(v / (1 - b2^t)) + eps); entries with
// mask[e] == 0 stay fixed.
__global__ void adam_kernel(int64_t n, const float* __restrict__ g, const unsigned char* __restrict__ mask, float lr,
                            float b1, float b2, float eps, float c1, float c2, float* __restrict__ th,
                            float* __restrict__ m, float* __restrict__ v) {
  const int64_t e = blockIdx.x * (int64_t)blockDim.x + threadIdx.x;
  if (e >= n || (mask && !mask[e])) return;
  const float ge = g[e];
  const float me = b1 * m[e] + (1.f - b1) * ge, ve = b2 * v[e] + (1.f - b2) * ge * ge;
  m[e] = me;
  v[e] = ve;
  th[e] -= lr * (me / c1) / (sqrtf(ve / c2) + eps);
}

// Lane layout check of the BF16 matrix instruction: A[i][k] = 16 i + k,
// B = identity, so D = A; out[lane * 4 + j] = D fragment element j of lane.
__global__ void bf16_probe_kernel(float* out) {
  const int lane = threadIdx.x;
  bf16x4 a, b;
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int k = 4 * (lane >> 4) + j;
    a[j] = (short)to_bf16((float)(16 * (lane & 15) + k));
    b[j] = (short)to_bf16(k == (lane & 15) ? 1.f : 0.f);
  }
  f32x4 d = {0.f, 0.f, 0.f, 0.f};
  d = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, d, 0, 0, 0);
#pragma unroll
  for (int j = 0; j < 4; ++j) out[lane * 4 + j] = d[j];
}

inline unsigned nblk(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

}  // namespace spde

using namespace spde;

extern "C" {

int spde_conv_packed_size(int cin, int transposed, int64_t* halves) {
  if ((cin != 8 && cin != 32) || !halves) {
    set_error("spde_conv_packed_size: cin must be 8 or 32");
    return SPDE_ERR_ARG;
  }
  const int kin = transposed ? 9 * kCh : 9 * cin;
  *halves = (int64_t)((kin + 15) / 16) * 2 * 64 * 4;
  return SPDE_OK;
}

int spde_conv_pack(int cin, int transposed, const float* W, unsigned short* frag, void* stream) {
  int64_t sz = 0;
  int rc = spde_conv_packed_size(cin, transposed, &sz);
  if (rc) return rc;
  if (!W || !frag) {
    set_error("spde_conv_pack: invalid argument");
    return SPDE_ERR_ARG;
  }
  hipLaunchKernelGGL(pack_kernel, dim3(nblk(sz, 256)), dim3(256), 0, (hipStream_t)stream, cin, transposed, W, frag);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

int spde_conv_forward(int M, int N, int T, int cin, const float* in, const float* mask, const unsigned short* frag,
                      const float* bias, int relu, float* out, void* stream) {
  if (M < 1 || N < 1 || T < 1 || (cin != 8 && cin != 32) || !in || !frag || !out) {
    set_error("spde_conv_forward: invalid argument");
    return SPDE_ERR_ARG;
  }
  const int nx = (M + kTx - 1) / kTx, ny = (N + 7) / 8;
  if ((int64_t)nx * ny * T > INT32_MAX) {
    set_error("spde_conv_forward: lattice too large");
    return SPDE_ERR_ARG;
  }
  const dim3 grid((unsigned)(nx * ny * T));
  if (cin == 32)
    hipLaunchKernelGGL(conv_kernel<32>, grid, dim3(256), 0, (hipStream_t)stream, M, N, nx, ny, in, mask, frag, bias,
                       relu, out);
  else
    hipLaunchKernelGGL(conv_kernel<8>, grid, dim3(256), 0, (hipStream_t)stream, M, N, nx, ny, in, mask, frag, bias,
                       relu, out);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

int spde_conv_wgrad_workspace(int64_t P, int cin, int64_t* floats) {
  if (P < 1 || (cin != 8 && cin != 32) || !floats) {
    set_error("spde_conv_wgrad_workspace: invalid argument");
    return SPDE_ERR_ARG;
  }
  const int64_t nchunk = P / 1024 + 1 < 256 ? P / 1024 + 1 : 256;
  const int nkt = (9 * cin + 15) / 16;
  *floats = nchunk * (int64_t)nkt * 16 * kCh + nchunk * kCh;
  return SPDE_OK;
}

int spde_conv_backward(int M, int N, int T, int cin, const float* X, const float* G, const float* Y, float* dW,
                       float* db, float* work, void* stream) {
  if (M < 1 || N < 1 || T < 1 || (cin != 8 && cin != 32) || !X || !G || !dW || !db || !work) {
    set_error("spde_conv_backward: invalid argument");
    return SPDE_ERR_ARG;
  }
  hipStream_t s = (hipStream_t)stream;
  const int64_t P = (int64_t)M * N * T;
  const int64_t nchunk = P / 1024 + 1 < 256 ? P / 1024 + 1 : 256;
  const int nkt = (9 * cin + 15) / 16;
  float* wpart = work;
  float* bpart = work + nchunk * (int64_t)nkt * 16 * kCh;
  const int nx = (M + kTx - 1) / kTx, ny = (N + 7) / 8;
  if ((int64_t)nx * ny * T > INT32_MAX) {
    set_error("spde_conv_backward: lattice too large");
    return SPDE_ERR_ARG;
  }
  if (cin == 32)
    hipLaunchKernelGGL(conv_wgrad_kernel<32>, dim3((unsigned)nchunk), dim3(512), 0, s, M, N, nx, ny, nx * ny * T, X, G,
                       Y, wpart, bpart);
  else
    hipLaunchKernelGGL(conv_wgrad_kernel<8>, dim3((unsigned)nchunk), dim3(512), 0, s, M, N, nx, ny, nx * ny * T, X, G,
                       Y, wpart, bpart);
  // only k < 9 cin rows are real weights
  const int64_t width = 9ll * cin * kCh;
  hipLaunchKernelGGL(chunk_sum_kernel, dim3(nblk(width + kCh, 64)), dim3(256), 0, s, (int)nchunk, width,
                     (int64_t)nkt * 16 * kCh, wpart, bpart, dW, db);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

int spde_adam(int64_t n, const float* g, const unsigned char* mask, float lr, float b1, float b2, float eps, int step,
              float* theta, float* m, float* v, void* stream) {
  if (n < 1 || !g || !theta || !m || !v || step < 1) {
    set_error("spde_adam: invalid argument");
    return SPDE_ERR_ARG;
  }
  const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
  hipLaunchKernelGGL(adam_kernel, dim3(nblk(n, 256)), dim3(256), 0, (hipStream_t)stream, n, g, mask, lr, b1, b2, eps, c1,
                     c2, theta, m, v);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

int spde_debug_bf16_probe(float* out, void* stream) {
  if (!out) {
    set_error("spde_debug_bf16_probe: invalid argument");
    return SPDE_ERR_ARG;
  }
  hipLaunchKernelGGL(bf16_probe_kernel, dim3(1), dim3(64), 0, (hipStream_t)stream, out);
  SPDE_HIP(hipGetLastError());
  return SPDE_OK;
}

}  // extern "C"
