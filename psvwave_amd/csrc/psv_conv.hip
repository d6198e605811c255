// psv_conv.hip -- bfloat16 MFMA kernels that run and train the learned
// gradient preconditioner (a U-Net over the velocity kernels).
//
// Activations are NHWC bfloat16 bit patterns, images stacked along the rows
// (rows = batch * H).  A convolution is an implicit GEMM
//   out[m][n] = sum_k A[m][k] * B[k][n],   B[k][n] = w[n * K + k],
// with m = output pixel and A gathered from the input by one of three modes:
//   kConv       ks x ks "same" convolution, k = tap * cin + ci;
//   kScatter    2x2 stride-2 transposed convolution: K = cin, n = q * cout + co,
//               result written to pixel (2y + q / 2, 2x + q % 2);
//   kGather2x2  space-to-depth gather (the input gradient of the transposed
//               convolution): the input has 2H x 2W pixels,
//               k = q * cin + ci reads pixel (2y + q / 2, 2x + q % 2).
// One wavefront computes a 64 x 64 (or 128 x 32) tile of out with
// v_mfma_f32_32x32x16_bf16 (fp32 accumulation); bias, the erf GELU (optionally storing the
// pre-activation) and the GELU derivative of a stored pre-activation (the
// backward pass) are fused into the epilogue.
//
// The weight gradient dW[i][j] = sum_p L[p][i] R[p][j] is a second MFMA
// kernel whose reduction runs over pixels, split across wavefronts into
// fp32 partial sums that a fixed-order pass adds up (deterministic).
#include <hip/hip_runtime.h>

#include <cstdint>

#include "psv_kernels.h"

namespace psv {

namespace {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef float f32x4 __attribute__((ext_vector_type(4)));

__device__ inline uint16_t to_bf16(float v) {
  uint32_t u = __float_as_uint(v);
  if ((u & 0x7f800000u) == 0x7f800000u) return (uint16_t)((u >> 16) | ((u & 0xffff) ? 0x40 : 0));
  u += 0x7fffu + ((u >> 16) & 1u);  // round to nearest even
  return (uint16_t)(u >> 16);
}
// The same of two values by the device's conversion instruction (which gives
// every value the same bits, NaN payloads aside).
__device__ inline uint32_t to_bf16x2(float lo, float hi) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{lo, hi}, bf16x2));
}

__device__ inline float from_bf16(uint16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ inline float gelu(float v) { return 0.5f * v * (1.0f + erff(v * 0.70710678118654752f)); }

// d/dv [v Phi(v)] = Phi(v) + v phi(v)
__device__ inline float gelu_grad(float v) {
  return 0.5f * (1.0f + erff(v * 0.70710678118654752f)) +
         v * 0.39894228040143268f * __expf(-0.5f * v * v);
}

// Accumulator r of lane (half, l32) of v_mfma_f32_32x32x8_bf16 holds row
// 8 (r / 4) + 4 half + r % 4, column l32 of the 32 x 32 tile.
__device__ inline int acc_row(int r, int half) { return 8 * (r >> 2) + 4 * half + (r & 3); }

// A lane's 8 values of K (k = k0 + 8 half ... + 7) lie in one tap because
// cin and in_stride are multiples of 8, so they are one aligned 16-byte load.
// Source element offset of pixel (yg, x) (yi = row within its image) for a
// tap, or -1 outside the image.
__device__ inline long long conv_src(const ConvGemm &a, int tap, int yg, int x, int yi) {
  if (a.mode == kGather2x2)
    return ((long long)(2 * yg + (tap >> 1)) * (2 * a.W) + 2 * x + (tap & 1)) * a.in_stride;
  const int pad = a.ks / 2, dy = tap / a.ks - pad, dx = tap % a.ks - pad;
  if (yi + dy < 0 || yi + dy >= a.H || x + dx < 0 || x + dx >= a.W) return -1;
  return ((long long)(yg + dy) * a.W + x + dx) * a.in_stride;
}

// Epilogue of one output value (bias already added): keep the rounded
// pre-activation (training), GELU, times the GELU derivative of a stored
// pre-activation (backward), store.
__device__ inline void conv_store(const ConvGemm &a, long long pix, int co, float v) {
  if (a.pre16) {
    const uint16_t h = to_bf16(v);
    a.pre16[pix * a.cout + co] = h;
    v = from_bf16(h);
  }
  if (a.gelu) v = gelu(v);
  if (a.dz) v *= gelu_grad(from_bf16(a.dz[pix * a.dz_stride + co]));
  const long long o = pix * a.out_stride + a.out_off + co;
  if (a.out32)
    a.out32[o] = v;
  else
    a.out16[o] = to_bf16(v);
}

// The same of 8 consecutive channels, in 16-byte accesses.
__device__ inline void conv_store8(const ConvGemm &a, long long pix, int co, float v[8]) {
  if (a.pre16) {
    u32x4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = to_bf16x2(v[2 * e], v[2 * e + 1]);
    *(u32x4 *)(a.pre16 + pix * a.cout + co) = h;
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = from_bf16((uint16_t)(h[e >> 1] >> (16 * (e & 1))));
  }
  if (a.gelu) {
#pragma unroll
    for (int e = 0; e < 8; ++e) v[e] = gelu(v[e]);
  }
  if (a.dz) {
    const u32x4 z = *(const u32x4 *)(a.dz + pix * a.dz_stride + co);
#pragma unroll
    for (int e = 0; e < 8; ++e)
      v[e] *= gelu_grad(from_bf16((uint16_t)(z[e >> 1] >> (16 * (e & 1)))));
  }
  const long long o = pix * a.out_stride + a.out_off + co;
  if (a.out32) {
    *(f32x4 *)(a.out32 + o) = f32x4{v[0], v[1], v[2], v[3]};
    *(f32x4 *)(a.out32 + o + 4) = f32x4{v[4], v[5], v[6], v[7]};
  } else {
    u32x4 h;
#pragma unroll
    for (int e = 0; e < 4; ++e) h[e] = to_bf16x2(v[2 * e], v[2 * e + 1]);
    *(u32x4 *)(a.out16 + o) = h;
  }
}
// Whether every 8 channels that start at a multiple of 8 lie in aligned 16
// bytes of each tensor (two of a 32-bit one).
bool conv_stores8(const ConvGemm &a) {
  const uintptr_t p = (uintptr_t)a.out16 | (uintptr_t)a.out32 | (uintptr_t)a.pre16 |
                      (uintptr_t)a.dz;
  return (p & 15) == 0 && a.cout % 8 == 0 && a.out_stride % 8 == 0 && a.out_off % 8 == 0 &&
         (!a.dz || a.dz_stride % 8 == 0);
}

// A wavefront holds a 32 x 32 tile with a channel per lane, so stores from the
// accumulators are of 2 bytes, and each value costs an address and a
// conversion of its own, which with the activation was most of a 3 x 3 layer of
// 32 channels.  The tile is turned over in LDS instead (kTurnPitch: rows of 32
// values, 16-byte aligned, on shifted banks), and each lane takes 8 channels of
// a pixel twice: f(pixel row of the tile, first channel, values).  A training
// step on 16 images: 3 x 3 layers 1.36 -> 0.92 ms, with the pooling in such
// accesses 4.18 -> 3.24 ms in all.
constexpr int kTurnPitch = 36;
template <class F>
__device__ inline void turn_tile(float *s, const f32x16 &acc, float bias, int lane, F f) {
  const int half = lane >> 5, l32 = lane & 31;
#pragma unroll
  for (int r = 0; r < 16; ++r) s[acc_row(r, half) * kTurnPitch + l32] = acc[r] + bias;
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const int row = 16 * q + (lane >> 2), c = 8 * (lane & 3);
    const f32x4 lo = *(const f32x4 *)(s + row * kTurnPitch + c);
    const f32x4 hi = *(const f32x4 *)(s + row * kTurnPitch + c + 4);
    float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    f(row, c, v);
  }
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();  // the next tile overwrites this one
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Blocks go to the device's 8 dies (XCDs) in turn, each with an L2 of its own.
// A kernel numbers its blocks so that those which read the same data follow
// each other, and this number gives them to one die (3 x 3 layers of a
// training step 1.43 -> 1.36 ms): launched with a multiple of 8 blocks, those
// beyond the last exit.
__device__ inline int xcd_block() { return (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3); }
unsigned xcd_grid(long long blocks) { return (unsigned)((blocks + 7) / 8 * 8); }

// One wavefront computes a (32 WM) x (32 WN) tile of out with
// v_mfma_f32_32x32x16_bf16: per step of 16 along K each lane loads 16 bytes
// per 32-row slice of A and of B, and issues WM x WN matrix instructions.  A
// small image is bound by the latency of those loads: 2 x 2 scatter of 24 x 40
// pixels, 128 -> 64 channels: 37 us in 64 x 64 tiles of 15 blocks, 9.5 us in
// 32 x 32 tiles of 60.
template <int WM, int WN, bool STORE8>
__global__ void __launch_bounds__(256) conv_mfma_kernel(ConvGemm a) {
  __shared__ __attribute__((aligned(16))) float s_turn[STORE8 ? 4 * 32 * kTurnPitch : 1];
  const int lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
  const int M = a.rows * a.W, N = a.mode == kScatter ? 4 * a.cout : a.cout;
  const int ntaps = a.mode == kGather2x2 ? 4 : a.ks * a.ks, K = ntaps * a.cin;
  const int ntm = (M + 32 * WM - 1) / (32 * WM), ntn = (N + 32 * WN - 1) / (32 * WN);
  const int tile = xcd_block() * 4 + (threadIdx.x >> 6);
  if (tile >= ntm * ntn) return;  // whole wavefronts exit together
  const int tn = tile % ntn, tm = tile / ntn;
  int yg[WM], xx[WM], yi[WM];
  bool mok[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) {
    const int m = (tm * WM + i) * 32 + l32;
    mok[i] = m < M;
    yg[i] = m / a.W;
    xx[i] = m - yg[i] * a.W;
    yi[i] = yg[i] % a.H;
  }
  const uint16_t *bp[WN];
  bool nok[WN];
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    const int n = (tn * WN + j) * 32 + l32;
    nok[j] = n < N;
    bp[j] = a.w + (nok[j] ? (long long)n * K : 0) + 8 * half;
  }
  // this lane's position along K: tap and channel of k0 + 8 half
  int tap = (8 * half) / a.cin, ci = 8 * half - tap * a.cin;
  long long src[WM];
#pragma unroll
  for (int i = 0; i < WM; ++i) src[i] = mok[i] ? conv_src(a, tap, yg[i], xx[i], yi[i]) : -1;
  f32x16 acc[WM][WN];
#pragma unroll
  for (int i = 0; i < WM; ++i)
#pragma unroll
    for (int j = 0; j < WN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
  const bf16x8 zero = {};
  // A step's loads are issued kAhead steps before its matrix instructions:
  // far ahead in the small tiles, which few wavefronts run; the large ones
  // need their registers for wavefronts that hide the latency instead (with
  // 4 steps 128 x 32 tiles took 480 us a training step, with one 378)
  constexpr int kAhead = WM * WN == 1 ? 4 : 1;
  bf16x8 av[kAhead][WM], bv[kAhead][WN];
  auto load = [&](int s, int k0) {
    const bool kok = tap < ntaps;
#pragma unroll
    for (int i = 0; i < WM; ++i)
      av[s][i] = kok && src[i] >= 0 ? *(const bf16x8 *)(a.in + src[i] + ci) : zero;
#pragma unroll
    for (int j = 0; j < WN; ++j)
      bv[s][j] = kok && nok[j] ? *(const bf16x8 *)(bp[j] + k0) : zero;
    ci += 16;
    if (ci >= a.cin) {
      do {
        ci -= a.cin;
        ++tap;
      } while (ci >= a.cin);
      if (tap < ntaps) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
          src[i] = mok[i] ? conv_src(a, tap, yg[i], xx[i], yi[i]) : -1;
      }
    }
  };
#pragma unroll
  for (int s = 0; s < kAhead; ++s) load(s, 16 * s);  // past K: zeros
  for (int k0 = 0; k0 < K; k0 += 16 * kAhead) {
#pragma unroll
    for (int s = 0; s < kAhead; ++s) {
      if (k0 + 16 * s < K) {
#pragma unroll
        for (int i = 0; i < WM; ++i)
#pragma unroll
          for (int j = 0; j < WN; ++j)
            acc[i][j] =
                __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[s][i], bv[s][j], acc[i][j], 0, 0, 0);
        load(s, k0 + 16 * (s + kAhead));
      }
    }
  }
  if (STORE8) {
#pragma unroll
    for (int j = 0; j < WN; ++j) {
      const int nj = (tn * WN + j) * 32;
      const float b = a.bias && nok[j] ? a.bias[a.mode == kScatter ? (nj + l32) % a.cout : nj + l32] : 0.f;
#pragma unroll
      for (int i = 0; i < WM; ++i)
        turn_tile(s_turn + (threadIdx.x >> 6) * 32 * kTurnPitch, acc[i][j], b, lane,
                  [&](int row, int c, float *v) {
                    const int mm = (tm * WM + i) * 32 + row, n = nj + c;
                    if (mm >= M || n >= N) return;
                    long long pix = mm;
                    int co = n;
                    if (a.mode == kScatter) {
                      const int q = n / a.cout, py = mm / a.W, px = mm - py * a.W;
                      co = n - q * a.cout;
                      pix = (long long)(2 * py + (q >> 1)) * (2 * a.W) + (2 * px + (q & 1));
                    }
                    conv_store8(a, pix, co, v);
                  });
    }
    return;
  }
#pragma unroll
  for (int j = 0; j < WN; ++j) {
    if (!nok[j]) continue;
    const int n = (tn * WN + j) * 32 + l32;
    const int co = a.mode == kScatter ? n % a.cout : n;
    const float b = a.bias ? a.bias[co] : 0.f;
#pragma unroll
    for (int i = 0; i < WM; ++i) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int mm = (tm * WM + i) * 32 + acc_row(r, half);
        if (mm >= M) continue;
        long long pix = mm;
        if (a.mode == kScatter) {
          const int q = n / a.cout, py = mm / a.W, px = mm - py * a.W;
          pix = (long long)(2 * py + (q >> 1)) * (2 * a.W) + (2 * px + (q & 1));
        }
        conv_store(a, pix, co, acc[i][j][r] + b);
      }
    }
  }
}

// 3 x 3 convolution (mode 0, cin a multiple of 16, H a multiple of 4) with
// the operands staged in LDS.  A block computes 4 output rows x 32 columns
// x 32 channels; each wavefront one row.  Per 16 input channels the
// block loads the input tile with its halo (6 x 34 pixels, zero outside the
// image) and the weights of all 9 taps for its channels into LDS; the 9
// taps then read their A fragments from the same tile shifted by (dy, dx),
// so every input value is fetched from L2 once per block instead of 9 times.
// What bounds a small image is the chain of load latencies, a large one the
// LDS traffic: a chunk's loads are all issued together, during the matrix
// instructions of the chunk before (3 x 3 layers of one 316 x 188 image: 12 to
// 31 us each before, 10 to 15 so).  32 channels a block, not 64: twice the
// blocks and half the registers (all 26 layers of a training step on 16 images
// 1.39 ms against 1.49, inference on one 224 us against 296).
// With R = 2 rows a wavefront a value read from LDS serves two products more
// often (21 fragments for 18 instead of 36) and a block loads half the weights
// per row: 928 -> 893 us for the 26 layers of a training step, together with
// the operands' places free of bank conflicts.  What is left is vector issue,
// three quarters of the time: the activation, its derivative and the stores.
constexpr int kC3Cols = 32, kC3TileW = kC3Cols + 2, kC3Chan = 32;
template <bool STORE8, int R>
__global__ void __launch_bounds__(256) conv3_lds_kernel(ConvGemm a) {
  // the input tile and the weights, then the tiles of the four wavefronts
  constexpr int kC3Rows = 4 * R, kC3TileP = (kC3Rows + 2) * kC3TileW;
  // (each of channels 0 .. 7 of all pixels, then 8 .. 15, so that neighbouring
  // lanes read and write neighbouring 16 bytes)
  constexpr int kInHalf = kC3TileP * 8, kWHalf = 9 * kC3Chan * 8 + 32;
  constexpr int kIn = 2 * kInHalf, kBytes = 2 * (kIn + 2 * kWHalf);
  constexpr int kTurnBytes = STORE8 ? 4 * 4 * 32 * kTurnPitch : 0;
  __shared__ __attribute__((aligned(16))) char s_mem[kBytes > kTurnBytes ? kBytes : kTurnBytes];
  uint16_t *const s_in = (uint16_t *)s_mem, *const s_w = s_in + kIn;
  const int t = threadIdx.x, wave = t >> 6, lane = t & 63, half = lane >> 5, l32 = lane & 31;
  const int N = a.cout, K = 9 * a.cin;
  const int ntn = (N + kC3Chan - 1) / kC3Chan, ncol = (a.W + kC3Cols - 1) / kC3Cols;
  const int block = xcd_block();
  if (block >= a.rows / kC3Rows * ncol * ntn) return;
  const int nt = block % ntn, rest = block / ntn;
  const int ct = rest % ncol, band = rest / ncol;
  const int y0 = band * kC3Rows, x0 = ct * kC3Cols, n0 = nt * kC3Chan;
  const int yi0 = y0 % a.H;  // image row of the band's first row (bands never straddle images)
  f32x16 acc[R];
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[j][r] = 0.f;
  // this thread's 16-byte pieces of a chunk: source (null: zero) and place
  constexpr int NI = (kC3TileP * 2 + 255) / 256, NW = (9 * kC3Chan * 2 + 255) / 256;
  const uint16_t *src_in[NI], *src_w[NW];
#pragma unroll
  for (int q = 0; q < NI; ++q) {
    const int item = t + 256 * q, p = item >> 1, r = p / kC3TileW, c = p - r * kC3TileW;
    const int yl = yi0 - 1 + r, x = x0 - 1 + c;
    const bool ok = item < kC3TileP * 2 && yl >= 0 && yl < a.H && x >= 0 && x < a.W;
    src_in[q] = ok ? a.in + ((long long)(y0 - 1 + r) * a.W + x) * a.in_stride + 8 * (item & 1)
                   : nullptr;
  }
#pragma unroll
  for (int q = 0; q < NW; ++q) {
    const int item = t + 256 * q, tn = item >> 1, tap = tn / kC3Chan, n = tn - tap * kC3Chan;
    const bool ok = item < 9 * kC3Chan * 2 && n0 + n < N;
    src_w[q] = ok ? a.w + (long long)(n0 + n) * K + tap * a.cin + 8 * (item & 1) : nullptr;
  }
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 vi[NI], vw[NW];
  auto load = [&](int c0) {
#pragma unroll
    for (int q = 0; q < NI; ++q) vi[q] = src_in[q] ? *(const u32x4 *)(src_in[q] + c0) : zero;
#pragma unroll
    for (int q = 0; q < NW; ++q) vw[q] = src_w[q] ? *(const u32x4 *)(src_w[q] + c0) : zero;
  };
  load(0);
  for (int c0 = 0; c0 < a.cin; c0 += 16) {
    __syncthreads();  // the previous chunk's fragments have been read
#pragma unroll
    for (int q = 0; q < NI; ++q)
      if (256 * (q + 1) <= kC3TileP * 2 || t + 256 * q < kC3TileP * 2)
        *(u32x4 *)(s_in + (t & 1) * kInHalf + ((t + 256 * q) >> 1) * 8) = vi[q];
#pragma unroll
    for (int q = 0; q < NW; ++q)
      if (256 * (q + 1) <= 9 * kC3Chan * 2 || t + 256 * q < 9 * kC3Chan * 2)
        *(u32x4 *)(s_w + (t & 1) * kWHalf + ((t + 256 * q) >> 1) * 8) = vw[q];
    __syncthreads();
    if (c0 + 16 < a.cin) load(c0 + 16);
    bf16x8 av[R + 2][3];
#pragma unroll
    for (int dy = 0; dy < 3; ++dy) {
#pragma unroll
      for (int j = dy == 0 ? 0 : R + dy - 1; j < R + dy; ++j)
#pragma unroll
        for (int dx = 0; dx < 3; ++dx)
          av[j][dx] = *(const bf16x8 *)(s_in + half * kInHalf + ((wave * R + j) * kC3TileW + l32 + dx) * 8);
#pragma unroll
      for (int dx = 0; dx < 3; ++dx) {
        const bf16x8 bv =
            *(const bf16x8 *)(s_w + half * kWHalf + ((3 * dy + dx) * kC3Chan + l32) * 8);
#pragma unroll
        for (int j = 0; j < R; ++j)
          acc[j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(av[j + dy][dx], bv, acc[j], 0, 0, 0);
      }
    }
  }
  const int y = y0 + wave * R, n = n0 + l32;
  if (STORE8) {
    __syncthreads();  // the operands have been read
#pragma unroll
    for (int j = 0; j < R; ++j)
      turn_tile((float *)s_mem + wave * 32 * kTurnPitch, acc[j], a.bias && n < N ? a.bias[n] : 0.f,
                lane, [&](int row, int c, float *v) {
                  if (x0 + row < a.W && n0 + c < N)
                    conv_store8(a, (long long)(y + j) * a.W + x0 + row, n0 + c, v);
                });
    return;
  }
  if (n >= N) return;
  const float b = a.bias ? a.bias[n] : 0.f;
#pragma unroll
  for (int j = 0; j < R; ++j)
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int x = x0 + acc_row(r, half);
      if (x < a.W) conv_store(a, (long long)(y + j) * a.W + x, n, acc[j][r] + b);
    }
}

// Weight gradient: out[s][i][j] = sum over pixels p of split s of
// L[p][i] R[p][j].  L: the output gradient at the output pixels
// (l_s2d = 0: L[p][i] = l[p * l_stride + i]; l_s2d = 1: i = q * lc + c reads
// fine pixel (2y + q / 2, 2x + q % 2)); R: the layer input gathered as the
// forward convolution gathers it (j = tap * rc + c, zero outside the image).
// A block computes a tile of out, 64 x 64 or 32 x 96, each of its wavefronts
// a quarter of the split's pixels, added up in LDS in the end (a fourth of the
// partial sums to write and read again).  Per step of 16 pixels each
// lane loads 16 bytes (8 consecutive channels) of four consecutive pixels, of
// one of the tile's 16 groups of 8 columns of L or R, transposes them in registers and
// writes them, four pixels of a channel at a time, into this wavefront's part
// of LDS ([column][pixel]); the MFMA fragments (8 consecutive pixels of one
// column) are then two 8-byte LDS reads, all free of bank conflicts.  The next
// step's loads are in flight meanwhile.  Where rows hold a multiple of 4 pixels
// (ROW4) a lane's four lie in one row and need one test and one address.
// 18 layers of a training step on 16 images: 1.70 ms with a pixel per lane,
// written to LDS value by value; 1.38 so without ROW4, 1.04 with it; 0.86 with
// the flat tile and conflict-free writes (before, LDS was busy 83 % of the time,
// most of it with conflicts), and 0.33 -> 0.20 ms for the partial sums' addition.
constexpr int kWgRow = 20;                   // LDS row pitch in bf16: 16 pixels + 4
typedef unsigned int u32x2 __attribute__((ext_vector_type(2)));
// LDS place of a column: in every other 16 columns the two halves of 8 change
// places, so that the 16 lanes whose writes go together (4 groups of 8 columns
// by 4 of pixels) reach all banks; reads of 16 columns do in any case.
__device__ inline int wgrad_row(int col) { return (col ^ ((col >> 2) & 4)) * kWgRow; }
__device__ inline bf16x8 wgrad_fragment(const uint16_t *p) {
  const u32x2 lo = *(const u32x2 *)p, hi = *(const u32x2 *)(p + 4);
  return __builtin_bit_cast(bf16x8, u32x4{lo.x, lo.y, hi.x, hi.y});
}
template <bool ROW4, int U, int V>
__global__ void __launch_bounds__(256, U == 2 ? 3 : 4) wgrad_mfma_kernel(Wgrad a) {
  static_assert(4 * (U + V) == 16, "a lane for every group of columns and pixels");
  constexpr int kPart = 32 * U * kWgRow, kWave = kPart + 32 * V * kWgRow;
  __shared__ __attribute__((aligned(16))) uint16_t lds[4 * kWave];
  __shared__ float s_bias[4][32 * U];
  static_assert(sizeof(lds) >= 3 * 64 * 16 * sizeof(float), "a 32 x 32 tile of three wavefronts");
  const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, half = lane >> 5, l32 = lane & 31;
  const int nti = (a.I + 32 * U - 1) / (32 * U), ntj = (a.J + 32 * V - 1) / (32 * V);
  // the tiles of a split, which read the same pixels, on one die
  const int tile = xcd_block();
  if (tile >= nti * ntj * a.nsplit) return;
  const int ti = tile % nti, tj = (tile / nti) % ntj, s = tile / (nti * ntj);
  const int i0 = ti * 32 * U, j0 = tj * 32 * V;
  const long long P = (long long)a.rows * a.W;
  const long long p_begin = (long long)s * a.chunk + wave * (a.chunk / 4);
  const long long p_stop = p_begin + a.chunk / 4;
  const long long p_end = p_stop < P ? p_stop : P;
  uint16_t *const mine = lds + wave * kWave;
  const uint16_t *const la = mine, *const lb = la + kPart;
  // loading role: pixels 4 g .. 4 g + 3 of each step and columns 8 c .. 8 c + 7
  // of L or R
  const bool of_r = lane >= 16 * U;
  const int li = of_r ? lane - 16 * U : lane;
  const int g = (li >> 2) & 3, c8 = 8 * ((li & 3) + 4 * (li >> 4));
  const bool fine = !of_r && a.l_s2d;  // reads fine pixels
  const int col = of_r ? j0 + c8 : i0 + c8;
  const bool cok = col < (of_r ? a.J : a.I);
  const int tap = of_r ? col / a.rc : 0, pad = a.ks / 2;
  const int q = fine ? col / a.lc : 0;
  const int dy = of_r ? tap / a.ks - pad : 0, dx = of_r ? tap % a.ks - pad : 0;
  const int stride = of_r ? a.r_stride : a.l_stride;
  // element of pixel p: base + p * stride (fine pixels: see load)
  const uint16_t *const base =
      of_r ? a.r + ((long long)dy * a.W + dx) * stride + (col - tap * a.rc)
           : a.l + (fine ? ((long long)(q >> 1) * (2 * a.W) + (q & 1)) * stride + (col - q * a.lc)
                         : col);
  // its columns 0 .. 3 and 4 .. 7 of the 8
  uint16_t *const at = mine + (of_r ? kPart : 0) + 4 * g;
  uint16_t *const to[2] = {at + wgrad_row(c8), at + wgrad_row(c8 + 4)};
  long long p = p_begin + 4 * g;
  int yg = (int)(p / a.W), x = (int)(p - (long long)yg * a.W), yi = yg % a.H;
  f32x16 acc[U][V];
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int v = 0; v < V; ++v)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[u][v][r] = 0.f;
  const bool bias_tile = a.bias_out && tj == 0;  // also sums L over the pixels
  float lsum = 0.f;
  const u32x4 zero = {0u, 0u, 0u, 0u};
  u32x4 v[4];  // 8 bf16 of a pixel each, element t in the (t & 1) half of word t / 2
  const uint16_t *next = base + p * stride;  // of pixel p (not of fine pixels)
  auto load = [&]() {
    int xe = x, ye = yi, row = yg;
    if (ROW4) {  // four pixels of one row
      const bool ok = cok && p < p_end && yi + dy >= 0 && yi + dy < a.H;
      const uint16_t *from = next;
      long long each = stride;
      if (fine) from = base + (2 * p + 2LL * yg * a.W) * stride, each = 2 * stride;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        v[e] = zero;
        if (ok && (e > 0 || x + dx >= 0) && (e < 3 || x + 3 + dx < a.W))
          v[e] = *(const u32x4 *)(from + e * each);
      }
      next += 16LL * stride;
    }
#pragma unroll
    for (int e = 0; !ROW4 && e < 4; ++e) {
      v[e] = zero;
      const int yy = ye + dy, xx = xe + dx;
      if (cok && p + e < p_end && yy >= 0 && yy < a.H && xx >= 0 && xx < a.W)
        v[e] = *(const u32x4 *)(base + (fine ? 2 * (p + e) + 2LL * row * a.W : p + e) * stride);
      if (++xe == a.W) {
        xe = 0;
        ++row;
        if (++ye == a.H) ye = 0;
      }
    }
    p += 16;
    x += 16;
    while (x >= a.W) {
      x -= a.W;
      ++yg;
      if (++yi == a.H) yi = 0;
    }
  };
  load();
  for (long long p0 = p_begin; p0 < p_end; p0 += 16) {
    // channel t of the four pixels
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      const unsigned sel = t & 1 ? 0x07060302u : 0x05040100u;  // high or low halves
      const u32x2 w = {__builtin_amdgcn_perm(v[1][t >> 1], v[0][t >> 1], sel),
                       __builtin_amdgcn_perm(v[3][t >> 1], v[2][t >> 1], sel)};
      *(u32x2 *)(to[t >> 2] + (t & 3) * kWgRow) = w;
    }
    load();
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    bf16x8 af[U], bf[V];
#pragma unroll
    for (int u = 0; u < U; ++u) af[u] = wgrad_fragment(la + wgrad_row(32 * u + l32) + 8 * half);
#pragma unroll
    for (int u = 0; u < V; ++u) bf[u] = wgrad_fragment(lb + wgrad_row(32 * u + l32) + 8 * half);
    if (bias_tile) {
      const bf16x8 r0 = wgrad_fragment(la + wgrad_row(lane & (32 * U - 1)));
      const bf16x8 r1 = wgrad_fragment(la + wgrad_row(lane & (32 * U - 1)) + 8);
      float t0 = 0.f;
#pragma unroll
      for (int t = 0; t < 8; ++t) t0 += (float)r0[t];
#pragma unroll
      for (int t = 0; t < 8; ++t) t0 += (float)r1[t];
      lsum += t0;
    }
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();  // the next step overwrites this wavefront's LDS rows
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int v = 0; v < V; ++v)
        acc[u][v] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[u], bf[v], acc[u][v], 0, 0, 0);
  }
  // the four wavefronts' sums, added in their order: each 32 x 32 part by one
  // of them, the others' values through LDS
  if (bias_tile && lane < 32 * U) s_bias[wave][lane] = lsum;
  float *out = a.out + (long long)s * a.I * a.J;
  float *const part = (float *)lds;
#pragma unroll
  for (int u = 0; u < U; ++u)
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const int owner = (u * V + v) & 3;
      __syncthreads();  // the operands, or the part before, have been read
      if (wave != owner) {
        float *const to = part + ((wave - owner - 1) & 3) * 1024 + lane;
#pragma unroll
        for (int r = 0; r < 16; ++r) to[64 * r] = acc[u][v][r];
      }
      __syncthreads();
      if (wave != owner) continue;
      const int j = j0 + 32 * v + l32;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float sum = 0.f;
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const float x =
              w == owner ? acc[u][v][r] : part[((w - owner - 1) & 3) * 1024 + 64 * r + lane];
          sum = w == 0 ? x : sum + x;
        }
        const int ii = i0 + 32 * u + acc_row(r, half);
        if (ii < a.I && j < a.J) out[(long long)ii * a.J + j] = sum;
      }
    }
  if (bias_tile && wave == 0 && lane < 32 * U && i0 + lane < a.I)
    a.bias_out[(long long)s * a.I + i0 + lane] =
        ((s_bias[0][lane] + s_bias[1][lane]) + s_bias[2][lane]) + s_bias[3][lane];
}

// out[e] = sum over s < nsplit of part[s * n + e]: `so` split lanes per
// output (a power of two dividing 256), each summing every so-th split, then
// a tree over the lanes -- a fixed order for a given (n, nsplit).  Two such
// sums of as many splits in one launch, since the second is mostly too small
// to pay for its own: the blocks beyond the first's belong to it.
struct SplitSum {
  const float *part;
  float *out;
  long long n;
};
__global__ void __launch_bounds__(256) reduce_splits_kernel(SplitSum first, SplitSum second,
                                                            int nsplit, int so) {
  __shared__ float red[256];
  const int eo = 256 / so, el = threadIdx.x % eo, sl = threadIdx.x / eo;
  const long long blocks = (first.n + eo - 1) / eo;
  const bool of_second = blockIdx.x >= blocks;
  const float *const part = of_second ? second.part : first.part;
  const long long n = of_second ? second.n : first.n;
  const long long e = (blockIdx.x - (of_second ? blocks : 0)) * eo + el;
  float v[8] = {};
  if (e < n) {
    int sp = sl;
    for (; sp + 7 * so < nsplit; sp += 8 * so)
#pragma unroll
      for (int k = 0; k < 8; ++k) v[k] += part[(long long)(sp + k * so) * n + e];
#pragma unroll
    for (int k = 0; k < 7; ++k)
      if (sp + k * so < nsplit) v[k] += part[(long long)(sp + k * so) * n + e];
  }
  red[threadIdx.x] = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  __syncthreads();
  for (int w = so / 2; w >= 1; w /= 2) {
    if (sl < w) red[sl * eo + el] += red[(sl + w) * eo + el];
    __syncthreads();
  }
  if (sl == 0 && e < n) (of_second ? second.out : first.out)[e] = red[el];
}

// part[s][c] = sum of src[p * stride + off + c] over the pixels of split s;
// block = 64 channels x 4 pixel lanes.
__global__ void __launch_bounds__(256) channel_sum_kernel(const uint16_t *__restrict__ src,
                                                          int stride, int off, int C,
                                                          long long P, long long chunk,
                                                          float *part) {
  __shared__ float red[4][64];
  const int c = blockIdx.x * 64 + (threadIdx.x & 63), r = threadIdx.x >> 6;
  const long long p_begin = (long long)blockIdx.y * chunk;
  const long long p_end = p_begin + chunk < P ? p_begin + chunk : P;
  float v0 = 0.f, v1 = 0.f;
  if (c < C) {
    long long p = p_begin + r;
    for (; p + 4 < p_end; p += 8) {
      v0 += from_bf16(src[p * stride + off + c]);
      v1 += from_bf16(src[(p + 4) * stride + off + c]);
    }
    if (p < p_end) v0 += from_bf16(src[p * stride + off + c]);
  }
  red[r][threadIdx.x & 63] = v0 + v1;
  __syncthreads();
  if (r == 0 && c < C)
    part[(long long)blockIdx.y * C + c] =
        ((red[0][threadIdx.x] + red[1][threadIdx.x]) + red[2][threadIdx.x]) + red[3][threadIdx.x];
}

__global__ void maxpool2_kernel(const uint16_t *__restrict__ in, uint16_t *out, int H,
                                int W, int C) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int Ho = H / 2, Wo = W / 2;
  if (i >= (long long)Ho * Wo * C) return;
  const int c = (int)(i % C);
  const long long p = i / C;
  const int y = (int)(p / Wo), x = (int)(p % Wo);
  float v = -INFINITY;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b)
      v = fmaxf(v, from_bf16(in[((long long)(2 * y + a) * W + (2 * x + b)) * C + c]));
  out[i] = to_bf16(v);
}

// The same, a thread 8 channels of a pixel in 16-byte accesses.
__global__ void maxpool2x8_kernel(const uint16_t *__restrict__ in, uint16_t *out, unsigned n,
                                  unsigned Wo, unsigned C8) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned p = i / C8, c = 8 * (i - p * C8), y = p / Wo, x = p - y * Wo;
  const long long C = 8LL * C8, W = 2LL * Wo;
  const uint16_t *const at = in + (2LL * y * W + 2 * x) * C + c;
  u32x4 v[4], m;
#pragma unroll
  for (int q = 0; q < 4; ++q) v[q] = *(const u32x4 *)(at + ((q >> 1) * W + (q & 1)) * C);
#pragma unroll
  for (int e = 0; e < 4; ++e) {
    float lo = -INFINITY, hi = -INFINITY;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      lo = fmaxf(lo, __uint_as_float(v[q][e] << 16));
      hi = fmaxf(hi, __uint_as_float(v[q][e] & 0xffff0000u));
    }
    m[e] = to_bf16x2(lo, hi);
  }
  *(u32x4 *)(out + (long long)p * C + c) = m;
}

// Gradient at a block output that feeds both a 2x2 max pooling and a skip
// connection, times the GELU derivative of the block's pre-activation:
//   out = (route(dpool) + dskip) * gelu'(z),
// route(dpool) sending each pooled gradient to the first maximum of its
// window in row-major order (the pooling's own choice).
__global__ void pool_backward_kernel(const uint16_t *__restrict__ act,
                                     const uint16_t *__restrict__ z,
                                     const float *__restrict__ dpool,
                                     const uint16_t *__restrict__ dskip, int skip_stride,
                                     int skip_off, uint16_t *out, int rows, int W, int C) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (long long)rows * W * C) return;
  const int c = (int)(i % C);
  const long long pix = i / C;
  const int yg = (int)(pix / W), x = (int)(pix - (long long)yg * W);
  float g = 0.f;
  if (dpool) {
    const int cy = yg >> 1, cx = x >> 1;
    int best = 0;
    float bv = -INFINITY;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      const float v =
          from_bf16(act[((long long)(2 * cy + (q >> 1)) * W + 2 * cx + (q & 1)) * C + c]);
      if (q == 0 || v > bv) {
        bv = v;
        best = q;
      }
    }
    if (best == ((yg & 1) << 1) + (x & 1)) g = dpool[((long long)cy * (W >> 1) + cx) * C + c];
  }
  if (dskip) g += from_bf16(dskip[pix * skip_stride + skip_off + c]);
  out[i] = to_bf16(g * gelu_grad(from_bf16(z[i])));
}

// The same, a thread the four pixels of a window and 8 channels of them: each
// window's values are read once and found by 32-bit divisions, in 16-byte
// accesses.
__global__ void __launch_bounds__(256)
    pool_backward8_kernel(const uint16_t *__restrict__ act, const uint16_t *__restrict__ z,
                          const float *__restrict__ dpool, const uint16_t *__restrict__ dskip,
                          int skip_stride, int skip_off, uint16_t *out, unsigned n, unsigned Wo,
                          unsigned C8) {
  const unsigned i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const unsigned p = i / C8, c = 8 * (i - p * C8), y = p / Wo, x = p - y * Wo;
  const long long C = 8LL * C8, W = 2LL * Wo, pix = 2LL * y * W + 2 * x;
  int best[8];
  float d[8];
  if (dpool) {
    u32x4 a[4];
#pragma unroll
    for (int q = 0; q < 4; ++q)
      a[q] = *(const u32x4 *)(act + (pix + (q >> 1) * W + (q & 1)) * C + c);
    const u32x4 d0 = *(const u32x4 *)(dpool + (long long)p * C + c);
    const u32x4 d1 = *(const u32x4 *)(dpool + (long long)p * C + c + 4);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      d[e] = __uint_as_float(e < 4 ? d0[e] : d1[e - 4]);
      float bv = 0.f;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const float v = from_bf16((uint16_t)(a[q][e >> 1] >> (16 * (e & 1))));
        if (q == 0 || v > bv) {
          bv = v;
          best[e] = q;
        }
      }
    }
  }
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const long long at = pix + (q >> 1) * W + (q & 1);
    const u32x4 zv = *(const u32x4 *)(z + at * C + c);
    u32x4 s = {0u, 0u, 0u, 0u}, o;
    if (dskip) s = *(const u32x4 *)(dskip + at * skip_stride + skip_off + c);
    float g[8];
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      g[e] = dpool && best[e] == q ? d[e] : 0.f;
      if (dskip) g[e] += from_bf16((uint16_t)(s[e >> 1] >> (16 * (e & 1))));
      g[e] *= gelu_grad(from_bf16((uint16_t)(zv[e >> 1] >> (16 * (e & 1)))));
    }
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = to_bf16x2(g[2 * e], g[2 * e + 1]);
    *(u32x4 *)(out + at * C + c) = o;
  }
}

constexpr long long kC3TwoRows = 1024;  // blocks of two rows a wavefront

// The layouts of all layers in one launch: a training step has 36 of weights
// and 18 of gradients, which torch copied with four to seven launches of some
// 3 us each (a step on 16 images 2.93 ms, 2.59 so).  32 items fill half of a
// launch's argument space.
constexpr int kRearrangeItems = 32, kRearrangeBlock = 1024;  // values a block
struct RearrangeArgs {
  Rearrangement items[kRearrangeItems];
  unsigned first[kRearrangeItems + 1];  // block of each item, then their number
};
template <bool BF16>
__global__ void __launch_bounds__(256) rearrange_kernel(RearrangeArgs a) {
  int i = 0;
  while (blockIdx.x >= a.first[i + 1]) ++i;
  const Rearrangement &m = a.items[i];
  const unsigned d1 = m.dims[1], d2 = m.dims[2], d3 = m.dims[3], n = m.dims[0] * d1 * d2 * d3;
#pragma unroll
  for (int q = 0; q < kRearrangeBlock / 256; ++q) {
    const unsigned e = (blockIdx.x - a.first[i]) * kRearrangeBlock + 256 * q + threadIdx.x;
    if (e >= n) return;
    const unsigned r3 = e / d3, i3 = e - r3 * d3, r2 = r3 / d2, i2 = r3 - r2 * d2;
    const unsigned i0 = r2 / d1, i1 = r2 - i0 * d1;
    float v = 0.f;
    if ((int)i3 < m.valid)
      v = m.src[m.offset + (long long)i0 * m.strides[0] + (long long)i1 * m.strides[1] +
                (long long)i2 * m.strides[2] + (long long)i3 * m.strides[3]];
    if (BF16)
      ((uint16_t *)m.dst)[e] = to_bf16(v);
    else
      ((float *)m.dst)[e] = v;
  }
}

unsigned blocks_of(long long n, int per) { return (unsigned)((n + per - 1) / per); }

}  // namespace

hipError_t launch_conv_gemm(const ConvGemm &a, hipStream_t s) {
  if (a.cin <= 0 || a.cin % 8 || a.in_stride % 8 || a.in_stride < a.cin || a.cout <= 0 ||
      a.rows <= 0 || a.H <= 0 || a.rows % a.H || a.W <= 0 ||
      (a.mode == kConv && a.ks != 1 && a.ks != 3) || (a.mode != kConv && a.ks != 1) ||
      a.mode < kConv || a.mode > kGather2x2 || (a.pre16 && a.mode != kConv))
    return hipErrorInvalidValue;
  if (((uintptr_t)a.in | (uintptr_t)a.w) & 15) return hipErrorInvalidValue;  // 16-byte loads
  const bool store8 = conv_stores8(a);
  if (a.mode == kConv && a.ks == 3 && a.cin % 16 == 0 && a.H % 4 == 0) {
    // two rows a wavefront where bands of 8 rows lie within an image and their
    // blocks still fill the device, four to a compute unit (with 16 images of
    // 316 x 188 the two finer levels; the coarser ones keep twice the blocks)
    const long long blocks = (long long)(a.rows / 4) * ((a.W + kC3Cols - 1) / kC3Cols) *
                             ((a.cout + kC3Chan - 1) / kC3Chan);
    const bool two = a.H % 8 == 0 && blocks >= 2 * kC3TwoRows;
    auto launch = [&](auto kernel, auto kernel8, long long n) {
      hipLaunchKernelGGL(store8 ? kernel8 : kernel, dim3(xcd_grid(n)), dim3(256), 0, s, a);
    };
    if (two)
      launch(conv3_lds_kernel<false, 2>, conv3_lds_kernel<true, 2>, blocks / 2);
    else
      launch(conv3_lds_kernel<false, 1>, conv3_lds_kernel<true, 1>, blocks);
    return hipGetLastError();
  }
  const long long M = (long long)a.rows * a.W, N = a.mode == kScatter ? 4LL * a.cout : a.cout;
  // 64 x 64 or 128 x 32 per wavefront, which reuses each operand; 32 x 32
  // where that leaves vector units (four a compute unit) without a wavefront
  // (2 x 2 scatter of 24 x 40 pixels x 16 images, 128 -> 64 channels: 44 us in
  // 64 x 64 tiles, 20 in 32 x 32; inference on one 316 x 188 image 324 against
  // 224 us)
  const bool wide = N > 32;
  const long long tiles = wide ? ((M + 63) / 64) * ((N + 63) / 64) : (M + 127) / 128;
  auto launch = [&](auto narrow, auto wide8, long long waves) {
    hipLaunchKernelGGL(store8 ? wide8 : narrow, dim3(xcd_grid((waves + 3) / 4)), dim3(256), 0, s, a);
  };
  if (tiles < 1024)
    launch(conv_mfma_kernel<1, 1, false>, conv_mfma_kernel<1, 1, true>,
           ((M + 31) / 32) * ((N + 31) / 32));
  else if (wide)
    launch(conv_mfma_kernel<2, 2, false>, conv_mfma_kernel<2, 2, true>, tiles);
  else
    launch(conv_mfma_kernel<4, 1, false>, conv_mfma_kernel<4, 1, true>, tiles);
  return hipGetLastError();
}

// Split lanes: up to 16 as the splits need, so that 16 neighbouring outputs are
// read together (with 4, as 344 splits had them, 9216 sums took 17 us); more
// where the outputs are too few to fill the device.
static void launch_reduce_splits(const SplitSum &a, const SplitSum &b, int nsplit, hipStream_t s) {
  int so = 1;
  while (so < 256 && (long long)so * 8 < nsplit && (so < 16 || a.n * so < 65536)) so *= 2;
  const int eo = 256 / so;
  hipLaunchKernelGGL(reduce_splits_kernel, dim3(blocks_of(a.n, eo) + blocks_of(b.n, eo)), dim3(256),
                     0, s, a, b, nsplit, so);
}

// Tile and splits.  A step costs a block the same in either tile, so the one
// that covers out in fewer is taken: 32 x 96 for up to 32 channels (32 x 288
// in 3 tiles instead of 5, half of which would be empty), mostly 64 x 64 else.
// As many blocks as the device's 256 compute units hold at once (four, three of
// the square tile, which needs more registers: with four of it, spilling, its
// layers took 36 and 110 us where they now take 28 and 97), of at least 512
// pixels a wavefront.
struct WgradPlan {
  bool flat;  // 32 x 96
  long long tiles;
};
static WgradPlan wgrad_plan(Wgrad &a, long long workspace_floats) {
  const long long P = (long long)a.rows * a.W;
  const long long square = (long long)((a.I + 63) / 64) * ((a.J + 63) / 64);
  const long long flat = (long long)((a.I + 31) / 32) * ((a.J + 95) / 96);
  const long long tiles = flat <= square ? flat : square;
  const long long blocks = flat <= square ? 1024 : 768;
  long long ns = (blocks + tiles - 1) / tiles;
  const long long max_ns = (P + 2047) / 2048;
  if (ns > max_ns) ns = max_ns;
  const long long fit = workspace_floats / ((long long)a.I * a.J + a.I);
  if (ns > fit) ns = fit;
  if (ns < 1) ns = 1;
  long long chunk = (P + ns - 1) / ns;
  chunk = (chunk + 63) / 64 * 64;
  a.nsplit = (int)((P + chunk - 1) / chunk);
  a.chunk = chunk;
  return {flat <= square, tiles * a.nsplit};
}

hipError_t launch_wgrad(Wgrad a, float *dw, float *db, float *workspace,
                        long long workspace_floats, hipStream_t s) {
  if (a.I <= 0 || a.J <= 0 || a.rows <= 0 || a.H <= 0 || a.rows % a.H || a.W <= 0 ||
      (a.ks != 1 && a.ks != 3) || a.rc <= 0 || a.rc % 8 || a.J != a.ks * a.ks * a.rc ||
      a.l_stride % 8 || a.r_stride % 8 || (((uintptr_t)a.l | (uintptr_t)a.r) & 15) ||
      (a.l_s2d && (a.lc <= 0 || a.lc % 8 || a.I != 4 * a.lc)))
    return hipErrorInvalidValue;
  const WgradPlan plan = wgrad_plan(a, workspace ? workspace_floats : 0);
  const long long n = (long long)a.I * a.J;
  const bool split = a.nsplit > 1;
  a.out = split ? workspace : dw;
  a.bias_out = db ? (split ? workspace + (long long)a.nsplit * n : db) : nullptr;
  auto launch = [&](auto square, auto flat) {
    hipLaunchKernelGGL(plan.flat ? flat : square, dim3(xcd_grid(plan.tiles)), dim3(256), 0, s, a);
  };
  if (a.W % 4 == 0)
    launch(wgrad_mfma_kernel<true, 2, 2>, wgrad_mfma_kernel<true, 1, 3>);
  else
    launch(wgrad_mfma_kernel<false, 2, 2>, wgrad_mfma_kernel<false, 1, 3>);
  if (split)
    launch_reduce_splits({workspace, dw, n}, {a.bias_out, db, db ? a.I : 0}, a.nsplit, s);
  return hipGetLastError();
}

hipError_t launch_rearrange(const Rearrangement *items, int n, bool to_bf16, hipStream_t s) {
  for (int at = 0; at < n; at += kRearrangeItems) {
    RearrangeArgs a{};
    const int count = n - at < kRearrangeItems ? n - at : kRearrangeItems;
    for (int i = 0; i < count; ++i) {
      const Rearrangement &m = a.items[i] = items[at + i];
      long long size = 1;
      for (int d : m.dims) {
        if (d <= 0) return hipErrorInvalidValue;
        size *= d;
        if (size > 0x7fffffff) return hipErrorInvalidValue;
      }
      a.first[i + 1] = a.first[i] + blocks_of(size, kRearrangeBlock);
    }
    const dim3 grid(a.first[count]);
    for (int i = count; i < kRearrangeItems; ++i) a.first[i + 1] = a.first[count];
    if (to_bf16)
      hipLaunchKernelGGL(rearrange_kernel<true>, grid, dim3(256), 0, s, a);
    else
      hipLaunchKernelGGL(rearrange_kernel<false>, grid, dim3(256), 0, s, a);
  }
  return hipGetLastError();
}

hipError_t launch_channel_sum(const uint16_t *src, int stride, int off, int c, long long P,
                              float *out, float *workspace, long long workspace_floats,
                              hipStream_t s) {
  if (c <= 0 || P <= 0 || off < 0 || off + c > stride) return hipErrorInvalidValue;
  long long ns = (P + 511) / 512;
  if (ns > 4096) ns = 4096;
  if (!workspace || ns > workspace_floats / c) ns = workspace ? workspace_floats / c : 1;
  if (ns < 1) ns = 1;
  const long long chunk = (P + ns - 1) / ns;
  ns = (P + chunk - 1) / chunk;
  hipLaunchKernelGGL(channel_sum_kernel, dim3(blocks_of(c, 64), (unsigned)ns), dim3(256), 0,
                     s, src, stride, off, c, P, chunk, ns > 1 ? workspace : out);
  if (ns > 1) launch_reduce_splits({workspace, out, c}, {}, (int)ns, s);
  return hipGetLastError();
}

hipError_t launch_conv_bf16(const uint16_t *in, const uint16_t *w, const float *bias,
                            void *out, bool out_f32, int h, int wd, int cin, int cout,
                            int ks, bool transposed, bool gelu, int out_stride,
                            int out_off, hipStream_t s) {
  ConvGemm a{};
  a.in = in;
  a.in_stride = cin;
  a.w = w;
  a.bias = bias;
  a.out16 = out_f32 ? nullptr : (uint16_t *)out;
  a.out32 = out_f32 ? (float *)out : nullptr;
  a.out_stride = out_stride;
  a.out_off = out_off;
  a.rows = h;
  a.H = h;
  a.W = wd;
  a.cin = cin;
  a.cout = cout;
  a.ks = ks;
  a.mode = transposed ? kScatter : kConv;
  a.gelu = gelu ? 1 : 0;
  return launch_conv_gemm(a, s);
}

hipError_t launch_maxpool2_bf16(const uint16_t *in, uint16_t *out, int h, int w, int c,
                                hipStream_t s) {
  if (h % 2 || w % 2 || c <= 0) return hipErrorInvalidValue;
  const long long n = (long long)(h / 2) * (w / 2) * c;
  if (c % 8 == 0 && n > 0 && n < (1LL << 34) && (((uintptr_t)in | (uintptr_t)out) & 15) == 0) {
    hipLaunchKernelGGL(maxpool2x8_kernel, dim3(blocks_of(n / 8, 256)), dim3(256), 0, s, in, out,
                       (unsigned)(n / 8), (unsigned)(w / 2), (unsigned)(c / 8));
    return hipGetLastError();
  }
  hipLaunchKernelGGL(maxpool2_kernel, dim3(blocks_of(n, 256)), dim3(256), 0, s, in, out, h,
                     w, c);
  return hipGetLastError();
}

hipError_t launch_pool_backward(const uint16_t *act, const uint16_t *z, const float *dpool,
                                const uint16_t *dskip, int skip_stride, int skip_off,
                                uint16_t *out, int rows, int w, int c, hipStream_t s) {
  if (rows % 2 || w % 2 || c <= 0 || (dpool && !act) ||
      (dskip && (skip_off < 0 || skip_off + c > skip_stride)))
    return hipErrorInvalidValue;
  const long long n = (long long)rows * w * c;
  const uintptr_t p = (uintptr_t)act | (uintptr_t)z | (uintptr_t)dpool | (uintptr_t)dskip |
                      (uintptr_t)out;
  if (c % 8 == 0 && n > 0 && n < (1LL << 34) && (p & 15) == 0 &&
      (!dskip || (skip_stride % 8 == 0 && skip_off % 8 == 0))) {
    hipLaunchKernelGGL(pool_backward8_kernel, dim3(blocks_of(n / 32, 256)), dim3(256), 0, s, act,
                       z, dpool, dskip, skip_stride, skip_off, out, (unsigned)(n / 32),
                       (unsigned)(w / 2), (unsigned)(c / 8));
    return hipGetLastError();
  }
  hipLaunchKernelGGL(pool_backward_kernel, dim3(blocks_of(n, 256)), dim3(256), 0, s, act, z,
                     dpool, dskip, skip_stride, skip_off, out, rows, w, c);
  return hipGetLastError();
}

}  // namespace psv
