// Pointwise (kernel size 1) convolution over [S, C, L] activations on the 16-bit matrix cores with fp32 accuracy.
//
// Two ways of putting fp32 operands on those cores, the same kernels for both (template parameter H):
//   * two fp16 terms (H): x is scaled by a power of two, hi = fp16(x), lo = fp16(x - hi); hi + lo holds x to 2^-23 or
//     better, and hi*hi + hi*lo + lo*hi (three v_mfma_f32_32x32x16_f16 products, fp32 accumulation) drops only lo*lo,
//     below 2^-22 of the product.  The scale keeps the terms inside fp16's exponent range: per row of A for the weights
//     (split_weight_f16_kernel, taken out per row of the result); for activations and gradients the power of two that
//     takes a largest magnitude into [2^14, 2^15): that of the sample in pw_gemm_kernel, whose columns are (sample,
//     position) pairs, that of the whole tensor in the weight gradient, which sums over samples (amax_kernel or the
//     producer of the tensor finds both, the kernels read them from a small device buffer).  Measured: 2^-23 of
//     sum |a||b| against float64.
//   * up to three bf16 terms: no scaling (bf16 has fp32's exponent range), six products for fp32 accuracy; described
//     next, and what the measurements below were taken with unless they say otherwise.  The fp16 split runs the qkv
//     shape in 0.19 ms (forward / input gradient) and 0.24 ms (weight gradient) against 0.27 and 0.30 ms.
//
// The reference computes the block Conv1d(k=1) -> BatchNorm1d -> LIF of its spiking self-attention with torch's
// convolution (layer/attention.py:310-329, 370-384; Conv2d(k=1) in model/spikformer.py:16-99).  A kernel-size-1
// convolution is the GEMM  Y[s] = W X[s]  per sample s, with X[s] a row-major [K, L] tile (tokens contiguous), and its
// backward the two GEMMs  dX[s] = W^T dY[s]  and  dW = sum_s dY[s] X[s]^T.  fp32 operands are split on the fly into up to
// three bf16 terms that sum to the value exactly (round to nearest, remainder, again); the products of the leading
// terms run on v_mfma_f32_32x32x16_bf16 with fp32 accumulation.  With three terms per operand and the six products
// whose combined order is at most two, the dropped part is below 2^-24 of each product: the accuracy of an fp32 GEMM
// at a multiple of the fp32 MFMA rate; an operand that is exact in bf16 (spikes, small counts) needs one term and
// halves the products.  Fewer terms trade accuracy for speed (two terms: about 2^-17 relative per product).
//
//   pw_gemm_kernel     C[s][m][l] = sum_k A[m][k] B[s][k][l]     (forward with A = W, input gradient with A = W^T)
//       A comes pre-split as bf16 planes [3][M_pad / 128][K_pad / 32][128][32] (split_weight_kernel, zero padded), B is
//       fp32 in memory.
//       The S * L columns of all samples form one column index, so tiles of 128 columns carry no padding whatever L
//       is.  A block of four wavefronts owns a 128 x 128 tile (each wavefront 64 x 64 = 2 x 2 MFMA tiles) and walks K
//       in steps of 32.  The matrix cores want, per lane, eight consecutive k of one row (A) or column (B): A tiles are
//       copied to LDS as they are; for B a work-item fetches eight k of two adjacent columns (consecutive lanes fetch
//       consecutive column pairs, so every access of a wavefront is one contiguous run), splits them and stores them
//       k-contiguous, which transposes the tile on the way in and leaves 16-byte fragment reads for both operands.
//       The global loads of the next two tiles are in flight while the current one is multiplied.
//       Measured on the qkv convolution of a Spikformer block (M = 1152, K = 384, 50 176 columns): 0.36 ms with six
//       products, 124 fp32-equivalent TFLOP/s.  Timing the kernel with parts cut out (only the loads 0.12 ms, only the
//       staging 0.05, only fragment reads + MFMA 0.15, empty loop + stores 0.07) gives parts that add up to the whole,
//       and neither wavefronts specialised as producers and consumers over two LDS buffers nor fewer, wider loads
//       changed the total: the phases do not hide behind each other on this chip at this matrix-core load.  Later
//       measurements on the same shape: tile requests made unconditional in the steady state of the K loop (a request
//       under a condition turns every later wait into a wait for all outstanding loads): 0.318 -> 0.301 ms; two LDS
//       buffers of half the depth with one barrier per step, staging of the next tile and multiplication of the current
//       one in the same step: 0.334 ms, and 0.352 ms with scheduler hints that ask for the staging instructions between
//       the matrix-core instructions; not kept.  Two groups of four wavefronts per block, each with its own tile and
//       one barrier apart so that one group multiplies while the other stages: 0.339 against 0.345 ms on random data,
//       not kept either.  The timestamp counter (clock64) around the phases of a K step (one wavefront, steady state):
//       with one block per compute unit staging 1150, multiplication 2160 (48 matrix-core instructions of 32 cycles
//       would be 1536), barriers 320 ticks, 45 k ticks per tile of 30.8 us; with two blocks 1280 / 3060 / 360 and 59 k
//       ticks per tile of 49.3 us: the second block adds a third to the throughput, not a factor of two.  How fast
//       the chip runs depends on what the matrix cores are fed: the same launch on an all-zero input takes 0.265
//       instead of 0.330 ms, and GRBM_GUI_ACTIVE over the kernel's duration gives 1.93 GHz here against 2.5 GHz in a
//       kernel that hardly uses them, so what a better overlap of the phases gains in cycles is partly lost in clock.
//       Raising the wavefront priority for the multiplication (s_setprio 2 around it): 0.348 and 0.331 ms
//       (Y = W X and dX) against 0.338 and 0.300; not kept.
//       By number of products (M = 1152, K = 384, random data): 1 product 0.15-0.16 ms, 2: 0.17-0.18, 3: 0.22,
//       6: 0.33-0.35.  The weight planes are stored tile by tile ([row tile][k step][row][k], for fp16 in
//       fragments of 32 rows x 16 k, 8 KiB per staged tile in a row) so that every 128-byte line a block fetches is used whole: 0.345 -> 0.338 ms, one-term activations
//       0.229 -> 0.215 ms.
//   pw_dw_kernel       dW[m][n] = sum_{s,l} dY[s][m][l] X[s][n][l]
//       both operands are contiguous along the contraction index l; a block owns a 128 x 128 tile of dW for a chunk
//       of samples and writes its partial tile, dw_reduce_kernel adds the chunks in a fixed order.
//   pw_dw_flat_kernel  the same on fp16 terms over rows of 29 positions and more, where dw_flat_plan finds a plan
// Blocks that share operand tiles are numbered so that they run on the same XCD (one L2 each, blocks are dealt
// round-robin over the eight XCDs).
#include <cmath>

#include "bn_map.h"
#include "sjhip_common.h"

namespace sjhip {

namespace {


typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

constexpr int kPwThreads = 256;
constexpr int kTile = 128;            // rows and columns of a block's output tile
constexpr int kTileK = 32;            // contraction elements per LDS stage (two MFMA k steps of 16)
constexpr int kRowBytes = 80;         // K-contiguous operand row in LDS: 32 bf16 + 16 bytes, so that the 16-byte fragment
                                      // reads of eight consecutive rows fall on all 32 banks
constexpr int kRowPlane = kTile * kRowBytes;
constexpr int kPlanePitch = 320;      // a k row of a B tile kept as it lies in memory (128 columns of fp16, n contiguous): 256
                                      // bytes + 64, so that the four k rows a transposing read of 32 lanes touches (64 bytes
                                      // of each) fall on distinct banks
static_assert(kTileK * kPlanePitch == kRowPlane, "a B tile takes the same LDS in either layout");
constexpr int kXcds = 8;
// where the B operand of pw_gemm_kernel comes from
constexpr int kBFloat = 0;   // fp32 [S][K][L], split into terms while it is staged
constexpr int kBBits = 1;    // bit-packed spikes over [S][K][L]
constexpr int kBPlanes = 2;  // fp16 term planes [TB][K][ld] with the columns of all samples in a row (split_planes_kernel)
typedef short s16x4 __attribute__((ext_vector_type(4)));
#ifndef SJHIP_PW_F16_WAVES
#define SJHIP_PW_F16_WAVES 3
#endif
// Wavefronts per SIMD of pw_gemm_kernel: with the fp16 split (two operand planes instead of three) 168 registers hold a
// wavefront's state (3 spilled), and a third resident block per compute unit is worth 9 % (191 -> 174 us on the qkv
// shape).  Not so for pw_dw_kernel, which splits both operands on the fly: 22 registers spilled, 237 -> 344 us; with
// one tile in flight instead of two it fits without spilling and takes the same 244 us, and the attention block's
// step 1.50 instead of 1.46 ms.
constexpr int pw_waves(bool h) { return h ? SJHIP_PW_F16_WAVES : 2; }
#ifndef SJHIP_PW_ROWS
#define SJHIP_PW_ROWS 1
#endif

__device__ __forceinline__ uint32_t pack_bf16(float lo, float hi) {
  bf16x2 p;
  p.x = (__bf16)lo;
  p.y = (__bf16)hi;
  return __builtin_bit_cast(uint32_t, p);
}
__device__ __forceinline__ float bf16_lo(uint32_t w) { return __builtin_bit_cast(float, w << 16); }
__device__ __forceinline__ float bf16_hi(uint32_t w) { return __builtin_bit_cast(float, w & 0xffff0000u); }

// Word t holds term t of (x0, x1): term 0 is the value rounded to bf16, term 1 the rounded remainder, term 2 what is
// left (exact for fp32 inputs: 3 x 8 significant bits).  The remainders are exact differences.
// With H the terms are fp16 (round to nearest, subnormals kept): two of them hold 22 to 24 significant bits of a value
// whose magnitude lies between 2^-2 and 2^16, which the callers arrange by scaling with a power of two.
template <int TERMS, bool H = false> __device__ __forceinline__ void split_pair(float x0, float x1, uint32_t (&w)[TERMS]) {
#pragma unroll
  for (int t = 0; t < TERMS; ++t) {
    if (H) {
      f16x2 p;
      p.x = (_Float16)x0;
      p.y = (_Float16)x1;
      w[t] = __builtin_bit_cast(uint32_t, p);
      if (t + 1 < TERMS) {
        x0 -= (float)p.x;
        x1 -= (float)p.y;
      }
    } else {
      w[t] = pack_bf16(x0, x1);
      if (t + 1 < TERMS) {
        x0 -= bf16_lo(w[t]);
        x1 -= bf16_hi(w[t]);
      }
    }
  }
}

// The terms of (s x0, s x1) for a power of two s, for the kernels' inner loops.  With two fp16 terms the remainder is one
// fused multiply-add per value, lo = fp16(fma(x, s, -hi)): s x and s x - hi are both exact in fp32, so this is the value
// that the separate product, conversion back and difference of split_pair give, and it compiles to the mixed-precision
// instruction that reads hi as fp16 and writes lo as fp16 (five vector instructions per pair of values instead of ten).
// Otherwise s is not applied (operands of one term, and bf16 terms, are not scaled).
template <int TERMS, bool H> __device__ __forceinline__ void split_scaled_pair(float x0, float x1, float s, uint32_t (&w)[TERMS]) {
  if constexpr (H && TERMS == 2) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    f32x2 y;
    y.x = x0 * s;
    y.y = x1 * s;
    const f16x2 hi = __builtin_convertvector(y, f16x2);
    f16x2 lo;
    lo.x = (_Float16)__builtin_fmaf(x0, s, -(float)hi.x);
    lo.y = (_Float16)__builtin_fmaf(x1, s, -(float)hi.y);
    w[0] = __builtin_bit_cast(uint32_t, hi);
    w[1] = __builtin_bit_cast(uint32_t, lo);
  } else {
    split_pair<TERMS, H>(x0, x1, w);
  }
}

// |x| of a number, 0 for an infinity or a NaN: non-finite elements take no part in choosing a scale (they still
// propagate through the products as they would in fp32).
__device__ __forceinline__ float finite_abs(float x) {
  const float a = fabsf(x);
  return a <= 3.4028234663852886e38f ? a : 0.0f;
}

// The power of two that brings a largest magnitude `amax` into [2^14, 2^15), and its inverse; 1 for a zero, subnormal
// or non-finite amax.  Multiplying by either is exact.
__device__ __forceinline__ void scale_for(float amax, float &scale, float &inverse) {
  const int field = (int)((__builtin_bit_cast(uint32_t, amax) >> 23) & 0xffu);
  scale = inverse = 1.0f;
  if (field == 0 || field == 255) return;
  int sf = 268 - field;  // biased exponent of 2^(14 - (field - 127))
  sf = sf < 1 ? 1 : (sf > 253 ? 253 : sf);
  scale = __builtin_bit_cast(float, (uint32_t)sf << 23);
  inverse = __builtin_bit_cast(float, (uint32_t)(254 - sf) << 23);
}

// Block number -> position in the order in which blocks that share tiles should be resident together: hardware block b
// runs on XCD b % 8, so XCD x gets the contiguous range of logical blocks it would get if the grid were cut in eight.
__device__ __forceinline__ int64_t xcd_order(int64_t b, int64_t n) {
  const int64_t q = n / kXcds, r = n % kXcds, x = b % kXcds, i = b / kXcds;
  return x * q + (x < r ? x : r) + i;
}

// the same in 32 bits (a 64-bit integer division is some hundred instructions, also where every lane has the same operands)
__device__ __forceinline__ uint32_t xcd_order32(uint32_t b, uint32_t n) {
  const uint32_t q = n / kXcds, r = n % kXcds, x = b % kXcds, i = b / kXcds;
  return x * q + (x < r ? x : r) + i;
}

// planes[t][r][c] = term t of src[r * ld_r + c * ld_c] for r < rows, c < cols, zero in the padding
__global__ void __launch_bounds__(256) split_weight_kernel(const float *src, int64_t rows, int64_t cols, int64_t ld_r,
                                                            int64_t ld_c, int64_t rows_pad, int64_t cols_pad,
                                                            uint16_t *planes) {
  const int64_t pairs = rows_pad * (cols_pad / 2);
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= pairs) return;
  const int64_t r = i / (cols_pad / 2), c = 2 * (i % (cols_pad / 2));
  float x0 = 0.0f, x1 = 0.0f;
  if (r < rows) {
    if (c < cols) x0 = src[r * ld_r + c * ld_c];
    if (c + 1 < cols) x1 = src[r * ld_r + (c + 1) * ld_c];
  }
  uint32_t w[3];
  split_pair<3>(x0, x1, w);
  // tile order: the 128 rows x 32 k that a block stages in one step are 8 KiB in a row, [row tile][k step][row][k]
  const int64_t at = (((r / kTile) * (cols_pad / kTileK) + c / kTileK) * kTile + r % kTile) * kTileK + c % kTileK;
#pragma unroll
  for (int t = 0; t < 3; ++t)
    reinterpret_cast<uint32_t *>(planes + (int64_t)t * rows_pad * cols_pad)[at / 2] = w[t];
}

// Where element (row r of 128, k c of 32) of a tile of fp16 planes lies: the 16 bytes (eight k) that a lane of
// v_mfma_f32_32x32x16_f16 takes, in lane order, so that a wavefront fetches the fragment of 32 rows and 16 k as 1 KiB in a row.
__device__ __forceinline__ int fragment_place(int r, int c) {
  return (r >> 5) * 1024 + (c >> 4) * 512 + (((c >> 3) & 1) * 32 + (r & 31)) * 8 + (c & 7);
}
// fp16 planes[t][tile order] = term t of scale_r * src[r][c], with a power-of-two scale per row r (a row of A is a row
// of the product, so the GEMM's epilogue takes the scale out again); the inverse scales follow the two planes as
// rows_pad floats.  One wavefront per row.  In evaluation mode (bn.map) it also makes the map of its row's batch norm
// channel, which depends on parameters only: a launch less between the convolution and the neuron.
__global__ void __launch_bounds__(256) split_weight_f16_kernel(const float *src, int64_t rows, int64_t cols, int64_t ld_r,
                                                                int64_t ld_c, int64_t rows_pad, int64_t cols_pad,
                                                                uint16_t *planes, float *amax_reset, int64_t amax_floats,
                                                                const BnEvalMap bn) {
  if (amax_reset && blockIdx.x == 0)
    for (int64_t i = threadIdx.x; i < amax_floats; i += 256) amax_reset[i] = 0.0f;
  const int lane = threadIdx.x & 63;
  const int64_t r = (int64_t)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (r >= rows_pad) return;
  float amax = 0.0f;
  if (r < rows) {
#pragma unroll 8
    for (int64_t c = lane; c < cols; c += 64) amax = fmaxf(amax, finite_abs(src[r * ld_r + c * ld_c]));
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) amax = fmaxf(amax, __shfl_xor(amax, d));
  float scale, inverse;
  scale_for(amax, scale, inverse);
#pragma unroll 4
  for (int64_t c = 2 * lane; c < cols_pad; c += 128) {
    float x0 = 0.0f, x1 = 0.0f;
    if (r < rows) {
      if (c < cols) x0 = src[r * ld_r + c * ld_c] * scale;
      if (c + 1 < cols) x1 = src[r * ld_r + (c + 1) * ld_c] * scale;
    }
    uint32_t w[2];
    split_pair<2, true>(x0, x1, w);
    const int64_t at = ((r / kTile) * (cols_pad / kTileK) + c / kTileK) * (kTile * kTileK) + fragment_place((int)(r % kTile), (int)(c % kTileK));
#pragma unroll
    for (int t = 0; t < 2; ++t)
      reinterpret_cast<uint32_t *>(planes + (int64_t)t * rows_pad * cols_pad)[at / 2] = w[t];
  }
  if (lane == 0) {
    reinterpret_cast<float *>(planes + 2 * rows_pad * cols_pad)[r] = inverse;
    if (bn.map && r < rows) store_bn_map(bn, (int)r);
  }
}

// The same planes of the transposed matrix: A[r][c] = src[c * ld_c + r], rows contiguous.  A wavefront per row would fetch
// one line per element; here a block takes 16 rows (64 contiguous bytes of every c) and four k steps: 64 x 16 work-items
// walk all of c for the rows' largest magnitudes (again for every block of the same rows, from L2), then each splits one
// pair of c.  [1536, 384]: 15 -> 9 us, [1152, 384] and [384, 384]: 19.7 -> 10.9 together.
constexpr int kSplitSteps = 4;
__global__ void __launch_bounds__(1024) split_weight_f16_transposed_kernel(const float *src, int64_t rows, int64_t cols, int64_t ld_c,
                                                                            int64_t rows_pad, int64_t cols_pad, uint16_t *planes) {
  __shared__ float part[16][17];
  const int ri = threadIdx.x & 15, ci = threadIdx.x >> 4;
  const int64_t r = (int64_t)blockIdx.x * 16 + ri;
  const bool row_ok = r < rows;
  const int64_t steps = cols_pad / kTileK, step = (int64_t)blockIdx.y * kSplitSteps + (ci >> 4), c = step * kTileK + 2 * (ci & 15);
  const float raw0 = row_ok && c < cols ? src[c * ld_c + r] : 0.0f;
  const float raw1 = row_ok && c + 1 < cols ? src[(c + 1) * ld_c + r] : 0.0f;
  float amax = 0.0f;
  if (row_ok) {
#pragma unroll 16
    for (int64_t i = ci; i < cols; i += 64) amax = fmaxf(amax, finite_abs(src[i * ld_c + r]));
  }
  amax = fmaxf(amax, __shfl_xor(amax, 16));  // the four c of a wavefront
  amax = fmaxf(amax, __shfl_xor(amax, 32));
  if ((threadIdx.x & 48) == 0) part[threadIdx.x >> 6][ri] = amax;
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 16; ++i) amax = fmaxf(amax, part[i][ri]);
  float scale, inverse;
  scale_for(amax, scale, inverse);
  if (step < steps) {
    uint32_t w[2];
    split_pair<2, true>(raw0 * scale, raw1 * scale, w);
    const int64_t at = ((r / kTile) * steps + step) * (kTile * kTileK) + fragment_place((int)(r % kTile), 2 * (ci & 15));
#pragma unroll
    for (int t = 0; t < 2; ++t) reinterpret_cast<uint32_t *>(planes + (int64_t)t * rows_pad * cols_pad)[at / 2] = w[t];
  }
  if (blockIdx.y == 0 && ci == 0) reinterpret_cast<float *>(planes + 2 * rows_pad * cols_pad)[r] = inverse;
}

// The largest magnitude of a tensor is kept as SJHIP_PW_AMAX_FLOATS non-negative floats whose maximum it is: blocks fold
// their share into word (block % SJHIP_PW_AMAX_FLOATS) with an integer atomic maximum (the bit patterns of non-negative
// floats order like unsigned integers, and a maximum does not depend on the order it is taken in).  Several words,
// and an atomic whose result is not used, so that a block neither meets tens of thousands of others on one address nor
// waits for memory before it ends: the kernel that writes the gradients of the qkv convolution takes 73 us with it
// (68 without), against 109 us with one word that a block reads first to skip atomics that would not raise it, and
// 93 us with that read spread over 256 words.
__device__ __forceinline__ void fold_amax(unsigned *amax_bits, float block_max) {
  atomicMax(amax_bits + blockIdx.x % SJHIP_PW_AMAX_FLOATS, __builtin_bit_cast(unsigned, block_max));
}
// The maximum of those words, in every lane of a wavefront.
__device__ __forceinline__ float tensor_amax(const float *amax) {
  static_assert(SJHIP_PW_AMAX_FLOATS == 256, "one 16-byte load per lane");
  const f32x4 v = reinterpret_cast<const f32x4 *>(amax)[threadIdx.x & 63];
  float m = fmaxf(fmaxf(v.x, v.y), fmaxf(v.z, v.w));
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) m = fmaxf(m, __shfl_xor(m, d));
  return m;
}
// The words of every sample's own largest magnitude follow the SJHIP_PW_AMAX_FLOATS words of the tensor's
// (SJHIP_PW_AMAX_SAMPLE_WORDS adjacent words per sample, whose maximum is the sample's amax: blocks that run at the
// same time belong to one sample, and atomics on one address are served one after the other): the GEMMs whose
// columns are (sample, position) pairs scale every sample by its own power of two (a sample whose values are all small
// beside another's keeps its significant bits), the weight gradient, which sums over the samples, by the tensor's.
__device__ __forceinline__ float sample_amax(const float *sample_words, int64_t s) {
  static_assert(SJHIP_PW_AMAX_SAMPLE_WORDS == 16, "four 16-byte loads per sample");
  const f32x4 *p = reinterpret_cast<const f32x4 *>(sample_words) + 4 * s;
  const f32x4 a = p[0], b = p[1], c = p[2], d = p[3];
  const f32x4 m = {fmaxf(fmaxf(a.x, b.x), fmaxf(c.x, d.x)), fmaxf(fmaxf(a.y, b.y), fmaxf(c.y, d.y)),
                   fmaxf(fmaxf(a.z, b.z), fmaxf(c.z, d.z)), fmaxf(fmaxf(a.w, b.w), fmaxf(c.w, d.w))};
  return fmaxf(fmaxf(m.x, m.y), fmaxf(m.z, m.w));
}
// x holds samples of per_sample elements each (a multiple of 4 when x is 16-byte aligned, so that a 16-byte access lies
// in one sample); a block takes 4096 consecutive elements.  One atomic per block for the tensor's words and one for
// a word of each of the (nearly always one, at most two) samples it lies in; what lies in further samples (samples
// shorter than a block) the work-items fold themselves.
constexpr int kAmaxChunk = 4096;
__global__ void __launch_bounds__(256) amax_kernel(const float *x, int64_t S, int64_t per_sample, unsigned *amax_bits) {
  const int64_t n = S * per_sample;
  __shared__ float part[4], part_first[4], part_second[4];
  unsigned *sample_bits = amax_bits + SJHIP_PW_AMAX_FLOATS + blockIdx.x % SJHIP_PW_AMAX_SAMPLE_WORDS;
  constexpr int64_t kW = SJHIP_PW_AMAX_SAMPLE_WORDS;
  const int64_t e0 = (int64_t)blockIdx.x * kAmaxChunk;
  const int64_t s0 = e0 / per_sample;                // the block's first sample (the same for every work-item)
  const int64_t next = (s0 + 1) * per_sample;        // first element of the following sample
  float amax = 0.0f;                                 // over everything the work-item reads
  float first = 0.0f, second = 0.0f;                 // over its elements of samples s0 and s0 + 1
  auto take = [&](int64_t e, float m) {
    amax = fmaxf(amax, m);
    if (e < next) first = fmaxf(first, m);
    else if (e < next + per_sample) second = fmaxf(second, m);
    else atomicMax(sample_bits + kW * (e / per_sample), __builtin_bit_cast(unsigned, m));  // (samples shorter than a block)
  };
  if ((reinterpret_cast<uintptr_t>(x) & 15u) == 0 && per_sample % 4 == 0) {
    f32x4 v[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t e = e0 + (int64_t)(k * 256 + threadIdx.x) * 4;
      v[k] = e + 4 <= n ? __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(x + e)) : (f32x4)(0.0f);
    }
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int64_t e = e0 + (int64_t)(k * 256 + threadIdx.x) * 4;
      if (e + 4 <= n) take(e, fmaxf(fmaxf(finite_abs(v[k].x), finite_abs(v[k].y)), fmaxf(finite_abs(v[k].z), finite_abs(v[k].w))));
    }
  } else {  // any alignment, any sample length: element by element
    for (int k = 0; k < 16; ++k) {
      const int64_t e = e0 + (int64_t)k * 256 + threadIdx.x;
      if (e < n) take(e, finite_abs(x[e]));
    }
  }
#pragma unroll
  for (int d = 32; d > 0; d >>= 1) {
    amax = fmaxf(amax, __shfl_xor(amax, d));
    first = fmaxf(first, __shfl_xor(first, d));
    second = fmaxf(second, __shfl_xor(second, d));
  }
  if ((threadIdx.x & 63) == 0) {
    part[threadIdx.x >> 6] = amax;
    part_first[threadIdx.x >> 6] = first;
    part_second[threadIdx.x >> 6] = second;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    fold_amax(amax_bits, fmaxf(fmaxf(part[0], part[1]), fmaxf(part[2], part[3])));
    if (e0 < n) atomicMax(sample_bits + kW * s0, __builtin_bit_cast(unsigned, fmaxf(fmaxf(part_first[0], part_first[1]), fmaxf(part_first[2], part_first[3]))));
    if (next < n && next < e0 + kAmaxChunk)
      atomicMax(sample_bits + kW * (s0 + 1), __builtin_bit_cast(unsigned, fmaxf(fmaxf(part_second[0], part_second[1]), fmaxf(part_second[2], part_second[3]))));
  }
}

struct PwGemmArgs {
  const uint16_t *a_planes;  // [3][M_pad / 128][K_pad / 32][128][32] bf16
  const float *b;            // [S][K][L]
  float *c;                  // [S][M][L]
  int64_t plane_stride;      // M_pad * K_pad
  int64_t ncols;             // S * Lq
  int M, K, K_pad, L;
  int Lq;                    // columns per sample of the column index: L rounded up to four (column_pitch), the rest hold zeros;
                             // kBPlanes: L
  float inv_Lq;              // 1 / Lq
  int m_blocks;
  float *stats;              // nullptr, or [2 x column blocks][M][2]: per row of c the sum and the sum of squares over
                             // each half (64 columns) of every column block
  const float *a_inverse;    // fp16 terms: the inverse scale of every (padded) row of A
  const float *b_amax;       // fp16 terms: nullptr (b needs no scale), or the words whose maximum is max |b|
  const float *b_amax_samples;  // kBFloat with two fp16 terms: the per-sample words of b's amax buffer (they follow b_amax's words)
  int64_t amax_s0, amax_S;      // the first sample of this launch, the samples of the tensor
  const uint16_t *b_planes;  // kBPlanes: fp16 terms of b, [TB][K][ld], column s * L + l of row k holds b[s][k][l]
  int64_t b_plane_stride;    // K * ld
  int ld;                    // columns per row of a plane: a multiple of 8, at least ncols
  int wide_out;              // L is a multiple of 4 and c is 16-byte aligned: the tile leaves through LDS as 16-byte row pieces
};
#ifndef SJHIP_PW_WIDE_OUT
#define SJHIP_PW_WIDE_OUT 1
#endif
typedef u32x4 u32x4_any __attribute__((aligned(4)));
// the elements skip .. 3 of v at the places 0 .. 3 - skip, zeros behind them: down by one where bit 0 of skip is set, then by two
// where bit 1 is (eight selects; chosen among four by the value of skip, the compiler branches for every vector)
template <typename V> __device__ __forceinline__ V moved_down(V v, int skip) {
  const bool one = (skip & 1) != 0, two = (skip & 2) != 0;
  V r;
  r.x = one ? v.y : v.x;
  r.y = one ? v.z : v.y;
  r.z = one ? v.w : v.z;
  r.w = one ? 0 : v.w;
  v.x = two ? r.z : r.x;
  v.y = two ? r.w : r.y;
  v.z = two ? 0 : r.z;
  v.w = two ? 0 : r.w;
  return v;
}
constexpr int kOutPitch = 68;                              // floats per row of the output staging buffer (64 columns + 4)
constexpr unsigned kOutLds = 4 * 32 * kOutPitch * 4;       // 32 rows x 64 columns per wavefront
constexpr int kStatPitch = 33;                             // floats per row of the transposing buffer: no bank conflicts
constexpr unsigned kStatLds = 4 * 64 * kStatPitch * 4;     // one buffer of 64 rows x 32 column pairs per wavefront

// Term pairs whose product is kept: combined order at most max(TA, TB) - 1.
template <int TA, int TB> struct Pairs {
  static constexpr int kMax = (TA > TB ? TA : TB) - 1;
  static __device__ __forceinline__ constexpr bool keep(int ta, int tb) { return ta + tb <= kMax; }
};

// One k step of 16 for a wavefront's 2 x 2 tiles: operands in registers, smallest terms first.
template <int TA, int TB, bool H>
__device__ __forceinline__ void mfma_step(const u32x4 (&af)[2][TA], const u32x4 (&bf)[2][TB], f32x16 (&acc)[2][2]) {
#pragma unroll
  for (int order = Pairs<TA, TB>::kMax; order >= 0; --order) {
#pragma unroll
    for (int ta = 0; ta < TA; ++ta) {
      const int tb = order - ta;
      if (tb < 0 || tb >= TB) continue;
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int nt = 0; nt < 2; ++nt)
          acc[mt][nt] = H ? __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, af[mt][ta]),
                                                                    __builtin_bit_cast(f16x8, bf[nt][tb]), acc[mt][nt], 0, 0, 0)
                          : __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, af[mt][ta]),
                                                                     __builtin_bit_cast(bf16x8, bf[nt][tb]), acc[mt][nt], 0, 0, 0);
    }
  }
}

// Fragment of a K-contiguous operand: row `row` of the tile, k group (lane / 32) of k step ks.
__device__ __forceinline__ u32x4 row_fragment(const uint8_t *plane, int row, int ks, int lane) {
  return *reinterpret_cast<const u32x4 *>(plane + row * kRowBytes + ks * 32 + (lane >> 5) * 16);
}

// BSRC == kBBits: b is a spike tensor that arrives bit-packed (the layout of sjhip_bit_pack over [S][K][L]: bit e % 8 of
// byte e / 8 is element e), 1/32 of the bytes of fp32 spikes; a work-item fetches the byte that holds its two columns of
// a row.
// BSRC == kBPlanes: b arrives as fp16 term planes that its producer wrote already scaled and split, rows of K with the
// columns of all samples in a row.  A tile of 32 k x 128 columns is copied to LDS as it lies in memory (16 bytes per
// work-item and row, no arithmetic), and the wavefronts fetch their fragments with the transposing LDS read
// (ds_read_b64_tr_b16: the 16 lanes of a group each point at four consecutive columns of a k row, four rows of 16
// columns in all, and lane j of the group receives column j of the four rows), which delivers the eight consecutive k of
// a column that the matrix cores want from a tile whose rows run along the columns.
template <int TA, int TB, bool H, int BSRC = kBFloat>
__global__ void __launch_bounds__(kPwThreads) __attribute__((amdgpu_waves_per_eu(pw_waves(H), pw_waves(H)))) pw_gemm_kernel(const PwGemmArgs a) {
  constexpr bool BITS = BSRC == kBBits;
  constexpr bool PLANES = BSRC == kBPlanes;
  static_assert(!BITS || TB == 1, "a bit-packed operand has one term");
  static_assert(!PLANES || H, "term planes are fp16");
  extern __shared__ __align__(16) uint8_t lds[];
  uint8_t *As = lds;                   // [TA][128][kRowBytes]
  uint8_t *Bs = lds + TA * kRowPlane;  // [TB][128][kRowBytes], column-major: a row holds 32 k of one column
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t logical = xcd_order(blockIdx.x, gridDim.x);
  const int mb = (int)(logical % a.m_blocks);
  const int64_t nb = logical / a.m_blocks;
  const int m0 = mb * kTile;
  const int64_t j0 = nb * kTile;
  const int M = a.M, K = a.K, L = a.L, Lq = a.Lq;
  const int K_pad = a.K_pad;

  // Addresses are a wavefront-uniform 64-bit base (scalar registers) plus a 32-bit per-lane byte offset, and every load
  // is unconditional (a branch per load would serialise them): offsets are clamped into the tensors and what lies
  // outside the matrices is zeroed, under one uniform branch, when the tile is staged.
  // A: two 16-byte chunks per term and thread; chunk q = tid + 256 i -> row q / 4, k chunk q % 4
  uint32_t a_off[2];
  int a_dst[2];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int q = tid + kPwThreads * i, row = H ? 32 * (q >> 7) + (q & 31) : q >> 2, kc = H ? (q >> 5) & 3 : q & 3;
    a_off[i] = (uint32_t)((mb * (K_pad / kTileK) * (kTile * kTileK) + 8 * q) * 2);
    a_dst[i] = row * kRowBytes + kc * 16;
  }
  // B: eight k (one fragment) of two adjacent columns, fetched as 8-byte accesses: columns 2 (tid % 64) and the next,
  // k group = the wavefront's number.  Consecutive lanes fetch consecutive column pairs, so every access of a wavefront
  // is one contiguous run, and a lane ends up with the eight k of a column that the matrix cores want from it.
  const int bc = 2 * (tid & 63);
  const int bk = __builtin_amdgcn_readfirstlane(wave * 8);
  const int64_t jc = j0 + bc;
  const int64_t sc = jc / Lq;
  const bool col_ok = jc < a.ncols && jc - sc * Lq < L;  // L is even, so the two columns are in one sample and both valid or both not
  uint32_t b_off = 0;  // byte offset of the column pair in row 0 of its sample; with BITS the bit index
  if (col_ok) b_off = (uint32_t)(((sc * K) * (int64_t)L + (jc - sc * Lq)) * (BITS ? 1 : 4));
  const bool edge_cols = __builtin_amdgcn_readfirstlane((j0 + kTile > a.ncols || L != Lq) ? 1 : 0) != 0;
  const char *a_base = reinterpret_cast<const char *>(a.a_planes);
  const char *b_base = reinterpret_cast<const char *>(a.b);
  // The scale of b: a sample's own power of two when b is split here (a work-item stages columns of one sample), the
  // tensor's when b arrives as planes (split with it).
  constexpr bool SAMPLE_SCALE = H && TB > 1 && BSRC == kBFloat;
  float b_scale = 1.0f, b_inverse = 1.0f;
  if (H && TB > 1 && !SAMPLE_SCALE && a.b_amax != nullptr) scale_for(tensor_amax(a.b_amax), b_scale, b_inverse);
  // A tile of 128 columns lies in at most two samples when a sample has that many positions: their two maxima are
  // fetched once per block from addresses that do not depend on the lane; shorter samples are looked up per column.
  const bool two_samples = Lq >= kTile;
  const int64_t tile_sample = j0 / Lq, next_sample_col = (tile_sample + 1) * Lq;
  float tile_amax[2] = {0.0f, 0.0f};
  if (SAMPLE_SCALE && a.b_amax_samples != nullptr && two_samples) {
    const int64_t s_a = a.amax_s0 + tile_sample, s_b = s_a + 1 < a.amax_S ? s_a + 1 : s_a;
    tile_amax[0] = sample_amax(a.b_amax_samples, s_a);
    tile_amax[1] = sample_amax(a.b_amax_samples, s_b);
  }
  auto column_amax = [&](int64_t j) {
    return two_samples ? (j < next_sample_col ? tile_amax[0] : tile_amax[1]) : sample_amax(a.b_amax_samples, a.amax_s0 + j / Lq);
  };
  if (SAMPLE_SCALE && a.b_amax_samples != nullptr && col_ok) scale_for(column_amax(jc), b_scale, b_inverse);
  // planes: 16-byte chunk pc (eight columns) of the k rows pr and pr + 16 of every plane
  const int pc = tid & 15, pr = tid >> 4;
  const uint32_t ld2 = PLANES ? (uint32_t)a.ld * 2u : 0u;
  const uint32_t p_col = (PLANES && j0 + 8 * pc < a.ld) ? 16u * pc : 0u;  // (ld is a multiple of 8: a chunk is inside a row or not)
  const char *bp_base = reinterpret_cast<const char *>(a.b_planes) + j0 * 2;

  // Two B tiles are in flight in registers (sets 0 and 1): a tile is requested two multiplications before it is staged,
  // which covers a miss to HBM.  The A tiles (weight planes, a few MB that every block reads) come from L2, one ahead.
  u32x4 ra[TA][2];
  u32x2 rb[2][8];       // [set][k]: the fp32 bit patterns of the two columns
  u32x4 rbp[2][TB][2];  // planes: [set][term][row pr + 16 i]  (of rb and rbp only the one that the mode uses exists)
  auto fetch_a = [&](int k0) {
#pragma unroll
    for (int t = 0; t < TA; ++t) {
      const char *plane = a_base + ((int64_t)t * a.plane_stride + (int64_t)(k0 / kTileK) * (kTile * kTileK)) * 2;
#pragma unroll
      for (int i = 0; i < 2; ++i) ra[t][i] = *reinterpret_cast<const u32x4 *>(plane + a_off[i]);
    }
  };
  auto fetch_b = [&](int k0, int set) {
    if constexpr (PLANES) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int k = k0 + pr + 16 * i;
        const uint32_t off = (uint32_t)(k < K ? k : K - 1) * ld2 + p_col;
#pragma unroll
        for (int t = 0; t < TB; ++t)
          rbp[set][t][i] = *reinterpret_cast<const u32x4 *>(bp_base + (int64_t)t * a.b_plane_stride * 2 + off);
      }
      return;
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int k = k0 + bk + i;
      if (BITS) {  // K * L is a multiple of 8 and L is even: the two bits share a byte
        const uint32_t e = b_off + (uint32_t)(k < K ? k : K - 1) * (uint32_t)L;
        rb[set][i].x = *reinterpret_cast<const uint8_t *>(b_base + (e >> 3));
        rb[set][i].y = e & 7u;
        continue;
      }
      const char *row = b_base + (int64_t)(k < K ? k : K - 1) * L * 4;
      rb[set][i] = *reinterpret_cast<const u32x2 *>(row + b_off);
    }
  };
  auto stage = [&](int k0, int set) {
#pragma unroll
    for (int t = 0; t < TA; ++t)
#pragma unroll
      for (int i = 0; i < 2; ++i) *reinterpret_cast<u32x4 *>(As + t * kRowPlane + a_dst[i]) = ra[t][i];
    if constexpr (PLANES) {
      if (edge_cols || k0 + kTileK > K) {  // rows beyond K and columns beyond the matrix hold zeros
        const int64_t left = a.ncols - (j0 + 8 * pc);
        const int nvalid = left < 0 ? 0 : (left > 8 ? 8 : (int)left);
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int n = (k0 + pr + 16 * i < K) ? nvalid : 0;
#pragma unroll
          for (int t = 0; t < TB; ++t) {
            u32x4 &v = rbp[set][t][i];
            v.x &= n >= 2 ? 0xffffffffu : (n == 1 ? 0xffffu : 0u);
            v.y &= n >= 4 ? 0xffffffffu : (n == 3 ? 0xffffu : 0u);
            v.z &= n >= 6 ? 0xffffffffu : (n == 5 ? 0xffffu : 0u);
            v.w &= n >= 8 ? 0xffffffffu : (n == 7 ? 0xffffu : 0u);
          }
        }
      }
#pragma unroll
      for (int t = 0; t < TB; ++t)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          *reinterpret_cast<u32x4 *>(Bs + t * kRowPlane + (pr + 16 * i) * kPlanePitch + pc * 16) = rbp[set][t][i];
      return;
    }
    if (edge_cols || k0 + kTileK > K) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (!(col_ok && k0 + bk + i < K)) rb[set][i] = (u32x2)(0u);
    }
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      uint32_t w[4][TB];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const u32x2 lo = rb[set][2 * i], hi = rb[set][2 * i + 1];
        float x0 = __builtin_bit_cast(float, c ? lo.y : lo.x), x1 = __builtin_bit_cast(float, c ? hi.y : hi.x);
        if (BITS) {
          x0 = (float)((lo.x >> (lo.y + c)) & 1u);
          x1 = (float)((hi.x >> (hi.y + c)) & 1u);
        }
        split_scaled_pair<TB, H>(x0, x1, b_scale, w[i]);
      }
#pragma unroll
      for (int t = 0; t < TB; ++t) {
        u32x4 v;
        v.x = w[0][t]; v.y = w[1][t]; v.z = w[2][t]; v.w = w[3][t];
        *reinterpret_cast<u32x4 *>(Bs + t * kRowPlane + (bc + c) * kRowBytes + bk * 2) = v;
      }
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

  auto multiply = [&]() {
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 af[2][TA], bf[2][TB];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int t = 0; t < TA; ++t) af[mt][t] = row_fragment(As + t * kRowPlane, wm * 64 + mt * 32 + (lane & 31), ks, lane);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          if constexpr (PLANES) {
            // group g = lane / 16 of a transposing read: columns 16 (g % 2) + 0..15 of the 32, k rows 8 (g / 2) + 0..3 (and + 4
            // in the second read) of the 16; lane i of the group points at columns 4 (i % 4) + 0..3 of row i / 4
            const int g = lane >> 4, i = lane & 15;
            const uint8_t *src = Bs + t * kRowPlane + (ks * 16 + 8 * (g >> 1) + (i >> 2)) * kPlanePitch +
                                 (wn * 64 + nt * 32 + 16 * (g & 1) + 4 * (i & 3)) * 2;
            typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
            const u32x2 k03 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(src)));
            const u32x2 k47 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(src + 4 * kPlanePitch)));
            bf[nt][t].x = k03.x; bf[nt][t].y = k03.y; bf[nt][t].z = k47.x; bf[nt][t].w = k47.y;
          } else {
            bf[nt][t] = row_fragment(Bs + t * kRowPlane, wn * 64 + nt * 32 + (lane & 31), ks, lane);
          }
        }
      mfma_step<TA, TB, H>(af, bf, acc);
    }
  };
  // One K step: stage the tile whose loads were requested earlier, request later tiles, multiply.  In the steady state
  // both requests are unconditional, so the compiler knows how many younger loads are outstanding when it waits for the
  // tile being staged and leaves them in flight; a request under a condition makes it wait for everything (vmcnt(0)),
  // which is tolerable only in the last steps.
  auto step = [&](int k0, int set, bool more_a, bool more_b) {
    __syncthreads();  // the previous tile has been read by every wavefront
    stage(k0, set);
    __syncthreads();
    if (more_a) fetch_a(k0 + kTileK);
    if (more_b) fetch_b(k0 + 2 * kTileK, set);
    multiply();
  };
  fetch_b(0, 0);
  fetch_a(0);
  fetch_b(kTileK, 1);  // rows beyond K are clamped, the tile is never staged then
  int k0 = 0;
  for (; k0 + 3 * kTileK < K_pad; k0 += 2 * kTileK) {
    step(k0, 0, true, true);
    step(k0 + kTileK, 1, true, true);
  }
  if (k0 < K_pad) step(k0, 0, k0 + kTileK < K_pad, k0 + 2 * kTileK < K_pad);
  if (k0 + kTileK < K_pad) step(k0 + kTileK, 1, k0 + 2 * kTileK < K_pad, false);
  if (k0 + 2 * kTileK < K_pad) step(k0 + 2 * kTileK, 0, false, false);

  // accumulator register r of a 32 x 32 tile: row 8 (r / 4) + 4 (lane / 32) + r % 4, column lane % 32
  float b_inv_col[2] = {b_inverse, b_inverse};  // of the two columns whose results this lane holds
  if (SAMPLE_SCALE && a.b_amax_samples != nullptr) {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int64_t j = j0 + wn * 64 + nt * 32 + (lane & 31);
      float unused;
      b_inv_col[nt] = 1.0f;
      if (j < a.ncols) scale_for(column_amax(j), unused, b_inv_col[nt]);
    }
  }
  if (H) {  // take the power-of-two scales of the row of A and of b out again: exact
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const float inv = a.a_inverse[m0 + wm * 64 + mt * 32 + 4 * (lane >> 5) + 8 * (r >> 2) + (r & 3)];
#pragma unroll
        for (int nt = 0; nt < 2; ++nt) acc[mt][nt][r] = acc[mt][nt][r] * inv * b_inv_col[nt];
      }
  }
  if (a.wide_out) {
    // The accumulators hold four rows of one column per group of registers, so a direct store writes 4-byte pieces of
    // 128-byte row segments, 64 instructions per wavefront.  Through LDS a wavefront's 64 x 64 tile leaves in two halves
    // of 32 rows as 16-byte pieces: a store instruction writes four rows of 256 contiguous bytes, 16 per wavefront.  A
    // piece of four columns lies in one sample (L is a multiple of 4).
    float *buf = reinterpret_cast<float *>(lds) + wave * (32 * kOutPitch);
    const int c4 = 4 * (lane & 15), rsub = lane >> 4;
    const int64_t j4 = j0 + wn * 64 + c4;
    const bool ok4 = j4 < a.ncols;
    const int64_t s4 = ok4 ? j4 / L : 0;
    float *cp4 = a.c + (s4 * M) * (int64_t)L + (ok4 ? (int)(j4 - s4 * L) : 0);
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      __syncthreads();  // the operand tiles (first half) or the rows of the first half (second) are no longer read
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r)
          buf[(8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * kOutPitch + nt * 32 + (lane & 31)] = acc[mt][nt][r];
      __syncthreads();
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const int row_local = 4 * i + rsub;
        const int row = m0 + wm * 64 + mt * 32 + row_local;
        const f32x4 v = *reinterpret_cast<const f32x4 *>(buf + row_local * kOutPitch + c4);
        if (ok4 && row < M) *reinterpret_cast<f32x4 *>(cp4 + (int64_t)row * L) = v;
      }
      // the batch-norm sums of these 32 rows over the wavefront's 64 columns (columns beyond the matrix hold exact
      // zeros): lane i adds row i from the staged half, in a fixed order
      if (a.stats && lane < 32) {
        const float *rowp = buf + lane * kOutPitch;
        float sum = 0.0f, squares = 0.0f;
#pragma unroll
        for (int j = 0; j < 16; ++j) {
          const f32x4 v = *reinterpret_cast<const f32x4 *>(rowp + 4 * j);
          sum += (v.x + v.y) + (v.z + v.w);
          squares = fmaf(v.x, v.x, squares); squares = fmaf(v.y, v.y, squares);
          squares = fmaf(v.z, v.z, squares); squares = fmaf(v.w, v.w, squares);
        }
        const int row = m0 + wm * 64 + mt * 32 + lane;
        if (row < M) {
          float *out = a.stats + ((2 * nb + wn) * (int64_t)M + row) * 2;
          out[0] = sum;
          out[1] = squares;
        }
      }
    }
    return;
  } else {
#pragma unroll
    for (int nt = 0; nt < 2; ++nt) {
      const int64_t j = j0 + wn * 64 + nt * 32 + (lane & 31);
      if (j >= a.ncols) continue;
      const int64_t s = j / Lq;
      const int l = (int)(j - s * Lq);
      if (l >= L) continue;
      float *cp = a.c + (s * M) * (int64_t)L + l;
  #pragma unroll
      for (int mt = 0; mt < 2; ++mt) {
        const int rbase = m0 + wm * 64 + mt * 32 + 4 * (lane >> 5);
  #pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int row = rbase + 8 * (r >> 2) + (r & 3);
          if (row < M) cp[(int64_t)row * L] = acc[mt][nt][r];
        }
      }
    }
  
}

  // Batch-norm statistics of the tile, so that no kernel has to read c again for them: per row the sum and the sum of
  // squares over the wavefront's 64 columns (columns beyond the matrix hold exact zeros).  A lane holds 32 rows of one
  // column pair; the values go through LDS, transposed, and lane i adds the 32 pairs of row i in a fixed order.
  if (a.stats) {
    __syncthreads();  // the operand tiles are no longer read
    float *buf = reinterpret_cast<float *>(lds) + wave * (64 * kStatPitch);
#pragma unroll
    for (int pass = 0; pass < 2; ++pass) {
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float v0 = acc[mt][0][r], v1 = acc[mt][1][r];
          const int row_local = mt * 32 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
          buf[row_local * kStatPitch + (lane & 31)] = pass == 0 ? v0 + v1 : v0 * v0 + v1 * v1;
        }
      __syncthreads();
      float sum = 0.0f;
#pragma unroll
      for (int j = 0; j < 32; ++j) sum += buf[lane * kStatPitch + j];
      const int row = m0 + wm * 64 + lane;
      if (row < M) a.stats[((2 * nb + wn) * (int64_t)M + row) * 2 + pass] = sum;
      __syncthreads();
    }
  }
}

// LDS of pw_gemm_rows_kernel: two B tiles (or the output staging of the epilogue, whichever is larger), then 128 floats
constexpr unsigned rows_inverse_offset(int tb) { return 2u * tb * kRowPlane > kOutLds ? 2u * tb * kRowPlane : kOutLds; }

// pw_gemm_rows_kernel: the same product, term order and batch-norm sums as pw_gemm_kernel<2, TB, true, kBFloat> (on rows of a
// multiple of four bit for bit), laid out for what a compute unit can move.  Measured per compute unit: LDS reads of 16 bytes per lane run at
// 256 bytes per cycle but writes at 64-78, and the vector memory path issues one wavefront load of 8 or 16 bytes per lane
// every 16 cycles (58 bytes per cycle from L1), so in pw_gemm_kernel a K step of a block costs about as many cycles of LDS
// (16 KB of A and 16 KB of B written, 64 KB read) and of the load path (32 eight-byte loads of B, 16 of A) as of the matrix
// cores (768 per SIMD).  Here
//   * a wavefront owns 32 rows of the tile and all 128 columns, and fetches its A fragments straight from the weight
//     planes (the 16 bytes a lane needs are contiguous in the tile-ordered planes): A never passes through LDS and no two
//     wavefronts fetch the same fragment;
//   * B is fetched as 16-byte pieces of a k row (four positions of one sample), half the load
//     instructions, split, and stored as it lies in memory (k rows of 128 columns); the wavefronts fetch their
//     fragments with the transposing LDS read, as pw_gemm_kernel does for term planes;
//   * two B tiles alternate in LDS, so a K step has one barrier.
// Per K step of a block: 16 KB written to and 64 KB read from LDS, 16 + 16 load instructions; 148 to 154 registers, three
// wavefronts per SIMD.
// The planes hold the 16 bytes of every lane of a fragment in lane order (fragment_place): eight lines per request instead of sixteen
// half used ones.  Where a column lies is worked out in 32 bits from one division per tile: as 64-bit divisions, eight of them in a
// wavefront's prologue and epilogue, it was half of the kernel's vector instructions at K = 384.  Both together, before / now, us:
// M = 1152, K = 384, 50 176 columns 194 / 187, M = 384, K = 1152 156 / 148; [64, 256, 100] -> 768 20.1 / 19.4, [16, 384, 196] -> 384
// 16.4 / 15.7, [4, 384, 196] -> 1152 16.1 / 15.4.
// BITS: b is a spike tensor that arrives bit-packed (as in pw_gemm_kernel, L a multiple of 4): a byte per piece, one term;
// M = K = 384, 50 176 columns: 41 us, pw_gemm_kernel 47.
// Samples of any length L >= 4: the column index gives every sample Lq = L rounded up to four columns, so that a piece
// lies in one sample; a piece that runs over the end of its row is fetched as the row's last four elements (at any
// 4-byte address) and moved down by one to three places with zeros behind it.
// (RAGGED is a template parameter: asked at run time the moves cost the aligned case 4 %, 106 -> 110 us at M = 1536, K = 384,
// 25 088 columns.)
// The products of a K step of such rows are summed by themselves, the small terms of both halves first, and reach the
// accumulators with one rounding (kStepSums); with one activation term, or few steps, what that rounding takes off is carried
// into the next step's sum (kStepSumsCompensated).  With one chain over all of K, as the rows of a multiple of four have it, the
// error against float64 was above that of the library's fp32 GEMM, which serves these lengths otherwise.  Relative 2-norm,
// library / chain / now: spikes, [48, 512, 49] -> 128 channels 1.11e-7 / 1.54e-7 / 9.9e-8 (6.8e-8 as one term); real values,
// [4, 1536, 49] -> 512 3.5e-7 / 4.4e-7 / 1.6e-7.  Over 70 shapes of 96 to 576 channels, 7 x 7 and 9 x 9, in units of the library's
// error: forward 0.78 on average and 0.96 at most (chain 1.25 and 1.53; step sums alone 0.87 and 1.09), input gradient 0.33 and 1.02,
// where the library settles on its most exact algorithm.  Where the line lies: the step sums alone exceed the library's
// error with one term (96 to 576 channels, by 3 to 9 %) and with two terms up to 128 channels (1 %); carried everywhere,
// [96, 512, 81] -> 512 takes 30.7 us instead of 26.2.
// 256 registers, two wavefronts per SIMD: [128, 384, 49] -> 1536 (624 blocks, more than are resident then) 37.9 us with one chain,
// 44.1 now, its input gradient 53.1 and 51.8, [96, 512, 81] -> 512 25.8 and 26.2.
enum RowSums { kOneChain = 0, kStepSums = 1, kStepSumsCompensated = 2 };
template <int TB, bool BITS, int SUMS>
__global__ void __launch_bounds__(kPwThreads) __attribute__((amdgpu_waves_per_eu(SUMS == kOneChain ? 3 : 2, SUMS == kOneChain ? 3 : 2))) pw_gemm_rows_kernel(const PwGemmArgs a) {
  constexpr int TA = 2;
  constexpr bool RAGGED = SUMS != kOneChain, COMPENSATED = SUMS == kStepSumsCompensated;
  constexpr int kBuf = TB * kRowPlane;  // one B tile: [TB][32 k][kPlanePitch]
  extern __shared__ __align__(16) uint8_t lds[];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const uint32_t logical = xcd_order32(blockIdx.x, gridDim.x);
  const uint32_t nb = logical / (uint32_t)a.m_blocks;
  const int mb = (int)(logical - nb * (uint32_t)a.m_blocks);
  // Columns are counted in 32 bits (a launch has fewer than 2^31), and a column's sample from that of the tile's first column, the
  // one quotient that is formed by a division: `at` = position in that sample + column in the tile, less than Lq + 128.
  const uint32_t j0 = nb * kTile, ncols = (uint32_t)a.ncols;
  const int M = a.M, K = a.K, L = a.L, Lq = RAGGED ? a.Lq : a.L;
  const uint32_t tile_sample = j0 / (uint32_t)Lq;
  const int l0 = (int)(j0 - tile_sample * (uint32_t)Lq);
  const bool two_samples = Lq >= kTile;
  // (exact: at + 1/2 is at least 1 / (2 Lq) of a sample away from a whole number, with Lq + 128 below 2^24 far more than the product's error)
  auto samples_on = [&](int at) { return two_samples ? (at >= Lq ? 1 : 0) : (int)(((float)at + 0.5f) * a.inv_Lq); };
  const int steps = a.K_pad / kTileK;

  // the inverse row scales of the tile wait in LDS (beyond the operand tiles) for the epilogue
  float *inverse_lds = reinterpret_cast<float *>(lds + rows_inverse_offset(TB));
  const float inverse_mine = tid < kTile ? a.a_inverse[mb * kTile + tid] : 0.0f;

  // A: lane (r, g) wants k chunk 2 ks + g (eight k, 16 bytes) of row r of the wavefront's 32 rows
  const char *a_base = reinterpret_cast<const char *>(a.a_planes) + (int64_t)mb * steps * (kTile * kTileK * 2);
  const uint32_t a_lane = (uint32_t)((wave * 1024 + lane * 8) * 2);
  // B: the 16 bytes of columns 4 (tid % 32) .. + 3 in the k rows tid / 32 + 8 i
  const int q4 = tid & 31, kr = tid >> 5;
  const bool col_ok = j0 + 4 * q4 < ncols;
  const int b_ds = col_ok ? samples_on(l0 + 4 * q4) : 0;
  uint32_t b_off = 0;
  int b_skip = 0;  // places that the piece is moved down
  if (col_ok) {
    const int l = l0 + 4 * q4 - b_ds * Lq, first = RAGGED ? min(l, L - 4) : l;
    b_off = ((tile_sample + (uint32_t)b_ds) * (uint32_t)K * (uint32_t)L + (uint32_t)first) * (BITS ? 1u : 4u);  // with BITS the bit index
    b_skip = l - first;
  }
  const uint32_t row_bytes = (uint32_t)L * (BITS ? 1u : 4u);
  // places of the rows kr + 8 i of a K step from its first row; rows beyond K repeat the last one (a minimum of offsets: one instruction)
  uint32_t b_row[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) b_row[i] = b_off + (uint32_t)(kr + 8 * i) * row_bytes;
  const bool edge_cols = __builtin_amdgcn_readfirstlane(j0 + kTile > ncols ? 1 : 0) != 0;
  const char *b_base = reinterpret_cast<const char *>(a.b);
  float b_scale = 1.0f, b_inverse = 1.0f;
  const bool per_sample = TB > 1 && a.b_amax_samples != nullptr;
  if (TB > 1 && !per_sample && a.b_amax != nullptr) scale_for(tensor_amax(a.b_amax), b_scale, b_inverse);
  float tile_amax[2] = {0.0f, 0.0f};
  if (per_sample && two_samples) {
    const int64_t s_a = a.amax_s0 + tile_sample, s_b = s_a + 1 < a.amax_S ? s_a + 1 : s_a;
    tile_amax[0] = sample_amax(a.b_amax_samples, s_a);
    tile_amax[1] = sample_amax(a.b_amax_samples, s_b);
  }
  auto column_amax = [&](int ds) {
    return two_samples ? tile_amax[ds] : sample_amax(a.b_amax_samples, a.amax_s0 + tile_sample + ds);
  };
  if (per_sample && col_ok) scale_for(column_amax(b_ds), b_scale, b_inverse);

  // [ks][term]: the fragments of the step being multiplied, refilled as they are used up; kStepSums: those of the next step
  // arrive in the other set
  u32x4 af[SUMS == kStepSums ? 4 : 2][TA];
  u32x4 rb[2][4];   // [set][i]: k row kr + 8 i of a tile, fp32 bit patterns of four columns
  auto fetch_a = [&](int tile, int ks, int set = 0) {  // every request is unconditional: k steps beyond the last repeat it
    const int t_ = tile < steps ? tile : steps - 1;
    const char *src = a_base + (int64_t)t_ * (kTile * kTileK * 2) + ks * 1024;
#pragma unroll
    for (int ta = 0; ta < TA; ++ta) af[2 * set + ks][ta] = *reinterpret_cast<const u32x4 *>(src + (int64_t)ta * a.plane_stride * 2 + a_lane);
  };
  auto fetch_b = [&](int tile, int set) {
    const int t_ = tile < steps ? tile : steps - 1;
    const uint32_t first = (uint32_t)(t_ * kTileK) * row_bytes;            // the same for every lane
    const uint32_t last = b_off + (uint32_t)(K - 1 - t_ * kTileK) * row_bytes;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const uint32_t at = min(b_row[i], last);
      if constexpr (BITS) rb[set][i].x = *reinterpret_cast<const uint8_t *>(b_base + ((at + first) >> 3)) >> ((at + first) & 7u);
      else rb[set][i] = *reinterpret_cast<const u32x4_any *>(b_base + first + at);
    }
  };
  auto stage = [&](int tile, int set) {
    uint8_t *Bs = lds + (tile & 1) * kBuf;
    if constexpr (RAGGED) {
#pragma unroll
      for (int i = 0; i < 4; ++i) rb[set][i] = moved_down(rb[set][i], b_skip);
    }
    if (edge_cols || (tile + 1) * kTileK > K) {
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (!(col_ok && tile * kTileK + kr + 8 * i < K)) rb[set][i] = (u32x4)(0u);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      if constexpr (BITS) {  // four positions: 0 or 1 in fp16
        const uint32_t four = rb[set][i].x;
        u32x2 v;
        v.x = (four & 1u) * 0x3c00u | (four & 2u) * 0x1e000000u;
        v.y = (four & 4u) * 0x0f00u | (four & 8u) * 0x07800000u;
        *reinterpret_cast<u32x2 *>(Bs + (kr + 8 * i) * kPlanePitch + q4 * 8) = v;
        continue;
      }
      // (the components go through scalars first: a bit cast applied to a vector component directly reads component 0)
      const uint32_t u0 = rb[set][i].x, u1 = rb[set][i].y, u2 = rb[set][i].z, u3 = rb[set][i].w;
      float x0 = __builtin_bit_cast(float, u0), x1 = __builtin_bit_cast(float, u1);
      float x2 = __builtin_bit_cast(float, u2), x3 = __builtin_bit_cast(float, u3);
      uint32_t w01[TB], w23[TB];
      split_scaled_pair<TB, true>(x0, x1, b_scale, w01);
      split_scaled_pair<TB, true>(x2, x3, b_scale, w23);
#pragma unroll
      for (int tb = 0; tb < TB; ++tb) {
        u32x2 v;
        v.x = w01[tb]; v.y = w23[tb];
        *reinterpret_cast<u32x2 *>(Bs + tb * kRowPlane + (kr + 8 * i) * kPlanePitch + q4 * 8) = v;
      }
    }
  };

  auto clear = [](f32x16 &v) {
#pragma unroll
    for (int q = 0; q < 16; ++q) v[q] = 0.0f;
  };
  // part: the sum of a K step; COMPENSATED: between the steps, what the last addition to acc rounded off, on which the next
  // step's products are summed
  f32x16 acc[4], part[COMPENSATED ? 4 : 2];
#pragma unroll
  for (int nt = 0; nt < 4; ++nt) {
    clear(acc[nt]);
    if constexpr (COMPENSATED) clear(part[nt]);
  }
  // the transposing read: group g = lane / 16 fetches columns 16 (g % 2) + 0..15 of the 32, k rows 8 (g / 2) + 0..3 (and
  // + 4 in the second read) of the 16; lane i of the group points at columns 4 (i % 4) + 0..3 of row i / 4
  const int tr_g = lane >> 4, tr_i = lane & 15;
  const uint32_t tr_off = (uint32_t)((8 * (tr_g >> 1) + (tr_i >> 2)) * kPlanePitch + (16 * (tr_g & 1) + 4 * (tr_i & 3)) * 2);
  typedef __attribute__((address_space(3))) s16x4 lds_s16x4;
  auto fragment_b = [&](const uint8_t *Bs, int tb, int ks, int nt) {
    const uint8_t *src = Bs + tb * kRowPlane + ks * 16 * kPlanePitch + nt * 64;
    const u32x2 k03 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(src)));
    const u32x2 k47 = __builtin_bit_cast(u32x2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4 *)(src + 4 * kPlanePitch)));
    u32x4 v;
    v.x = k03.x; v.y = k03.y; v.z = k47.x; v.w = k47.y;
    return v;
  };
  auto multiply = [&](auto parity, int tile, int next_a) {  // parity: of the tile
    const uint8_t *Bs = lds + (tile & 1) * kBuf + tr_off;
    if constexpr (RAGGED) {
      constexpr int set = COMPENSATED ? 0 : decltype(parity)::value;
      if constexpr (!COMPENSATED) {
        fetch_a(next_a, 0, set ^ 1);
        fetch_a(next_a, 1, set ^ 1);
        __builtin_amdgcn_sched_barrier(0);
      }
#pragma unroll
      for (int pair = 0; pair < 4; pair += 2) {
        u32x4 bf[2][2][TB];
        constexpr int stay = COMPENSATED ? 1 : 0;
#pragma unroll
        for (int n = 0; n < 2; ++n) {
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int tb = 0; tb < TB; ++tb) bf[n][ks][tb] = fragment_b(Bs, tb, ks, pair + n);
          if constexpr (!COMPENSATED) clear(part[n]);
        }
        // smallest terms first, of both halves of the step
#pragma unroll
        for (int order = Pairs<TA, TB>::kMax; order >= 0; --order) {
#pragma unroll
          for (int ta = 0; ta < TA; ++ta) {
            const int tb = order - ta;
            if (tb < 0 || tb >= TB) continue;
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
              for (int n = 0; n < 2; ++n)
                part[stay * pair + n] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, af[2 * set + ks][ta]),
                                                                                __builtin_bit_cast(f16x8, bf[n][ks][tb]), part[stay * pair + n], 0, 0, 0);
          }
        }
#pragma unroll
        for (int n = 0; n < 2; ++n) {
          const f32x16 sum = acc[pair + n] + part[stay * pair + n];
          if constexpr (COMPENSATED) part[pair + n] -= sum - acc[pair + n];
          acc[pair + n] = sum;
        }
        if constexpr (COMPENSATED) {
          if (pair == 2) {
            fetch_a(next_a, 0);
            fetch_a(next_a, 1);
          }
          __builtin_amdgcn_sched_barrier(0);
        }
      }
      return;
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      u32x4 bf[4][TB];
#pragma unroll
      for (int nt = 0; nt < 4; ++nt)
#pragma unroll
        for (int tb = 0; tb < TB; ++tb) bf[nt][tb] = fragment_b(Bs, tb, ks, nt);
      // smallest terms first, as mfma_step
#pragma unroll
      for (int order = Pairs<TA, TB>::kMax; order >= 0; --order) {
#pragma unroll
        for (int ta = 0; ta < TA; ++ta) {
          const int tb = order - ta;
          if (tb < 0 || tb >= TB) continue;
#pragma unroll
          for (int nt = 0; nt < 4; ++nt)
            acc[nt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, af[ks][ta]),
                                                              __builtin_bit_cast(f16x8, bf[nt][tb]), acc[nt], 0, 0, 0);
        }
      }
      fetch_a(next_a, ks);
      __builtin_amdgcn_sched_barrier(0);  // (the requests stay here: left alone, the compiler moves them to the end of the step)
    }
  };

  fetch_b(0, 0);
  fetch_a(0, 0);
  fetch_a(0, 1);
  fetch_b(1, 1);
  stage(0, 0);
  if (tid < kTile) inverse_lds[tid] = inverse_mine;
  fetch_b(2, 0);
  __syncthreads();
  // step i: tile i + 1 (requested two steps ago) goes into the other LDS buffer, tile i + 3 is requested into the registers
  // that frees, tile i is multiplied while the A fragments of tile i + 1 replace the ones used up
  int i = 0;
  for (; i + 1 < steps; i += 2) {
    stage(i + 1, 1);
    fetch_b(i + 3, 1);
    __builtin_amdgcn_sched_barrier(0);
    multiply(std::integral_constant<int, 0>(), i, i + 1);
    __syncthreads();
    if (i + 2 < steps) stage(i + 2, 0);
    fetch_b(i + 4, 0);
    __builtin_amdgcn_sched_barrier(0);
    multiply(std::integral_constant<int, 1>(), i + 1, i + 2);
    __syncthreads();
  }
  if (i < steps) {
    multiply(std::integral_constant<int, 0>(), i, i);
    __syncthreads();
  }

  // accumulator register q of a 32 x 32 tile: row 8 (q / 4) + 4 (lane / 32) + q % 4, column lane % 32
  float b_inv_col[4] = {b_inverse, b_inverse, b_inverse, b_inverse};
  if (per_sample) {
#pragma unroll
    for (int nt = 0; nt < 4; ++nt) {
      const int col = nt * 32 + (lane & 31);
      float unused;
      b_inv_col[nt] = 1.0f;
      if (j0 + col < ncols) scale_for(column_amax(samples_on(l0 + col)), unused, b_inv_col[nt]);
    }
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const f32x4 inv4 = *reinterpret_cast<const f32x4 *>(inverse_lds + wave * 32 + 8 * g + 4 * (lane >> 5));
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const float inv = e == 0 ? inv4.x : (e == 1 ? inv4.y : (e == 2 ? inv4.z : inv4.w));
#pragma unroll
      for (int nt = 0; nt < 4; ++nt) acc[nt][4 * g + e] = acc[nt][4 * g + e] * inv * b_inv_col[nt];
    }
  }
  // The tile leaves through LDS (the operand tiles are no longer read: the barrier above) in pieces of 32 rows x 64
  // columns per wavefront, as in pw_gemm_kernel: a store instruction writes four rows of 256 contiguous bytes, and lane i
  // adds row i of the staged piece for the batch-norm sums, in the same order.
  float *buf = reinterpret_cast<float *>(lds) + wave * (32 * kOutPitch);
  const int c4 = 4 * (lane & 15), rsub = lane >> 4;
  const int wave_row0 = mb * kTile + wave * 32;
#pragma unroll
  for (int half = 0; half < 2; ++half) {
    const int col4 = half * 64 + c4;
    const bool ok4 = j0 + col4 < ncols;
    const int ds4 = ok4 ? samples_on(l0 + col4) : 0, l4 = ok4 ? l0 + col4 - ds4 * Lq : 0;
    const int left = L - l4;  // positions of the sample from here on
    float *at4 = a.c + ((int64_t)(tile_sample + ds4) * M + (wave_row0 + rsub)) * (int64_t)L + l4;
    const int64_t step4 = 4 * (int64_t)L;
    __builtin_amdgcn_wave_barrier();  // the piece staged before has been read (LDS serves a wavefront's accesses in order)
#pragma unroll
    for (int ntl = 0; ntl < 2; ++ntl)
#pragma unroll
      for (int q = 0; q < 16; ++q)
        buf[(8 * (q >> 2) + 4 * (lane >> 5) + (q & 3)) * kOutPitch + ntl * 32 + (lane & 31)] = acc[2 * half + ntl][q];
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < 8; ++q) {
      const int row_local = 4 * q + rsub;
      const int row = wave_row0 + row_local;
      const f32x4 v = *reinterpret_cast<const f32x4 *>(buf + row_local * kOutPitch + c4);
      float *at = at4;
      at4 += step4;
      if (ok4 && row < M) {
        if (!RAGGED || left >= 4) {
          *reinterpret_cast<f32x4_any *>(at) = v;
        } else {
          at[0] = v.x;
          if (left > 1) at[1] = v.y;
          if (left > 2) at[2] = v.z;
        }
      }
    }
    if (a.stats && lane < 32) {
      const float *rowp = buf + lane * kOutPitch;
      float sum = 0.0f, squares = 0.0f;
#pragma unroll
      for (int j = 0; j < 16; ++j) {
        const f32x4 v = *reinterpret_cast<const f32x4 *>(rowp + 4 * j);
        sum += (v.x + v.y) + (v.z + v.w);
        squares = fmaf(v.x, v.x, squares); squares = fmaf(v.y, v.y, squares);
        squares = fmaf(v.z, v.z, squares); squares = fmaf(v.w, v.w, squares);
      }
      const int row = wave_row0 + lane;
      if (row < M) {
        float *out = a.stats + ((2 * (int64_t)nb + half) * M + row) * 2;
        out[0] = sum;
        out[1] = squares;
      }
    }
  }
}

struct PwDwArgs {
  const float *dy;   // [S][M][L]
  const float *x;    // [S][N][L]
  float *partials;   // [chunks][M][N]
  int64_t S;
  int M, N, L;
  int Lq;    // L rounded up to four: a row that four does not divide ends with a group that is partly zeros
  int s_per_chunk;
  int flat;  // the K steps run over the positions of all samples of a chunk in a row (see pw_dw_kernel)
  int m_blocks, n_blocks;
  const float *dy_amax, *x_amax;  // fp16 terms: nullptr (no scale), or the words whose maximum is the tensor's max |.|
};

// Two LDS buffers where x has one fp16 term (spikes, 2 x 30 KiB): the next tile is split and stored while the current one is
// multiplied, with one barrier per K step instead of two.  One buffer / two, us with the reduction, three processes of each in
// turn on one machine, shapes that pw_dw_flat_kernel leaves to this one: x as fp32 spikes, dy [1024, 512, 16], x [1024, 512, 16]
// 68.8 / 65.9, [256, 1152, 16] and [256, 384, 16] 44.7 / 43.9, [64, 2048, 16] and [64, 512, 16] 37.9 / 37.5, both [128, 512, 16] 31.3 / 31.7,
// [512, 768, 25] and [512, 256, 25] 38.6 / 38.2, both [64, 256, 49] 19.3 / 19.6; as bits 70.5 / 68.4, 44.4 / 44.4, 38.1 / 37.6, 32.5 / 32.6.
// With two terms of x (2 x 40 KiB) two buffers measured, on shapes that pw_dw_flat_kernel has taken over, 210.4 -> 214.0, 138.8 -> 138.4,
// 74.7 -> 74.5: those keep one, and every launch stays within the default limit of dynamic LDS.  (The bf16 split's three planes per
// operand would leave one block per compute unit.)
constexpr bool dw_two_buffers(bool h, int tb) { return h && tb == 1; }
// four elements at a 16-byte or, with ANY, at a 4-byte address
template <bool ANY> __device__ __forceinline__ f32x4 load4(const char *p) {
  if (ANY) return *reinterpret_cast<const f32x4_any *>(p);
  return *reinterpret_cast<const f32x4 *>(p);
}

// BITS: x is a spike tensor that arrives bit-packed (as in pw_gemm_kernel); a work-item fetches the byte whose low or
// high half holds its four consecutive positions of a row (L and N * L are multiples of 4 and 8).
template <int TA, int TB, bool H, bool BITS = false, bool RAGGED = false>
__global__ void __launch_bounds__(kPwThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) pw_dw_kernel(const PwDwArgs a) {
  static_assert(!BITS || (TB == 1 && !RAGGED), "a bit-packed operand has one term and rows of a multiple of four");
  static_assert(H || !RAGGED, "rows of other lengths run on fp16 terms");
  extern __shared__ __align__(16) uint8_t lds[];
  // [TA][128][kRowBytes] of dy, then [TB][128][kRowBytes] of x; DOUBLE: twice
  uint8_t *As = lds, *Bs = lds + TA * kRowPlane;
  constexpr bool DOUBLE = dw_two_buffers(H, TB);
  constexpr int kBuf = DOUBLE ? (TA + TB) * kRowPlane : 0;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t logical = xcd_order(blockIdx.x, gridDim.x);
  const int tiles = a.m_blocks * a.n_blocks;
  const int chunk = (int)(logical / tiles);
  const int tile = (int)(logical % tiles);
  const int mb = tile % a.m_blocks, nb = tile / a.m_blocks;
  const int m0 = mb * kTile, n0 = nb * kTile;
  const int M = a.M, N = a.N, L = a.L, Lq = RAGGED ? a.Lq : a.L;
  const int64_t s_begin = (int64_t)chunk * a.s_per_chunk;
  const int64_t s_end = s_begin + a.s_per_chunk < a.S ? s_begin + a.s_per_chunk : a.S;
  const int l_steps = (Lq + kTileK - 1) / kTileK;
  // flat: the contraction index runs over the quads (four positions) of all samples of the chunk in a row, so a K step of
  // eight quads may take the last quads of one sample and the first of the next, and only the last step of a chunk is
  // partly empty (a row of 196 positions is 6.125 steps instead of 7).  Needs at least eight quads per sample (a step
  // then touches two samples at most) and samples of less than 2^31 bytes (a lane's offset reaches into the second).
  const bool flat = a.flat != 0;
  const int Q = Lq >> 2;
  const int n_samples = (int)(s_end - s_begin);
  const int64_t total_quads = (int64_t)n_samples * Q;
  const int64_t iters = flat ? (total_quads + 7) / 8 : (int64_t)n_samples * l_steps;
  const uint32_t a_sample = (uint32_t)(M * L * 4), b_sample = (uint32_t)(N * L * (BITS ? 1 : 4));  // bytes; with BITS bits
  int f_s = 0, f_q = 0;  // flat: sample and quad at which the next step to be fetched begins
  int g_s = 0, g_q = 0;  // flat: the same for the next step to be staged

  // a thread fetches quad q4 (four consecutive l) of rows rr, rr + 32, rr + 64, rr + 96 of both operand tiles; addresses
  // are a uniform base (the sample) plus 32-bit per-lane offsets (row; position), loads are unconditional from clamped
  // offsets and the outside of the matrices is zeroed when the tile is staged
  const int q4 = tid & 7, rr = tid >> 3;
  uint32_t a_off[4], b_off[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = rr + 32 * i;
    a_off[i] = (uint32_t)((m0 + row < M ? m0 + row : M - 1) * L * 4);
    b_off[i] = (uint32_t)((n0 + row < N ? n0 + row : N - 1) * L * (BITS ? 1 : 4));  // bytes; with BITS bits
  }
  const bool edge_rows = __builtin_amdgcn_readfirstlane((m0 + kTile > M || n0 + kTile > N) ? 1 : 0) != 0;
  const char *dy_base = reinterpret_cast<const char *>(a.dy);
  const char *x_base = reinterpret_cast<const char *>(a.x);
  float a_scale = 1.0f, a_inverse = 1.0f, b_scale = 1.0f, b_inverse = 1.0f;
  if (H && TA > 1 && a.dy_amax != nullptr) scale_for(tensor_amax(a.dy_amax), a_scale, a_inverse);
  if (H && TB > 1 && a.x_amax != nullptr) scale_for(tensor_amax(a.x_amax), b_scale, b_inverse);
  f32x4 ra[2][4], rb[2][4];  // two tiles in flight, as in pw_gemm_kernel
  auto fetch = [&](int64_t it, int set) {  // (called for it = 0, 1, 2, ... in this order)
    int64_t s;
    uint32_t l_off, sa = 0, sb = 0;
    if (flat) {
      int q = f_q + q4;
      const bool second = q >= Q;
      if (second) q -= Q;
      const bool ok = f_s + (second ? 1 : 0) < n_samples;
      s = s_begin + f_s;
      l_off = ok ? (uint32_t)(RAGGED ? min(4 * q, L - 4) : 4 * q) * 4u : 0u;
      if (ok && second) {
        sa = a_sample;
        sb = b_sample;
      }
      f_q += 8;
      if (f_q >= Q) {
        f_q -= Q;
        ++f_s;
      }
    } else {
      s = s_begin + it / l_steps;
      const int l = (int)(it % l_steps) * kTileK + 4 * q4;
      l_off = (uint32_t)(min(l, L - 4) * 4);
    }
    const char *pa = dy_base + (s * M) * (int64_t)L * 4;
    const char *pb = x_base + (BITS ? ((s * N) * (int64_t)L >> 3) : (s * N) * (int64_t)L * 4);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      ra[set][i] = load4<RAGGED>(pa + (a_off[i] + sa + l_off));
      if (BITS) {
        const uint32_t e = b_off[i] + sb + (l_off >> 2);
        rb[set][i].x = __builtin_bit_cast(float, (uint32_t)*reinterpret_cast<const uint8_t *>(pb + (e >> 3)));
      } else {
        rb[set][i] = load4<RAGGED>(pb + (b_off[i] + sb + l_off));
      }
    }
  };
  auto stage = [&](int64_t it, int set) {  // (called for it = 0, 1, 2, ... in this order)
    bool l_ok, tail;
    int lq;  // the position of the work-item's quad in its row (for the bit offset)
    if (flat) {
      int q = g_q + q4;
      const bool second = q >= Q;
      if (second) q -= Q;
      l_ok = g_s + (second ? 1 : 0) < n_samples;
      lq = l_ok ? 4 * q : 0;
      tail = (int64_t)g_s * Q + g_q + 8 > total_quads;
      g_q += 8;
      if (g_q >= Q) {
        g_q -= Q;
        ++g_s;
      }
    } else {
      const int l0 = (int)(it % l_steps) * kTileK;
      l_ok = l0 + 4 * q4 < L;
      lq = l_ok ? l0 + 4 * q4 : L - 4;
      tail = l0 + kTileK > L;
    }
    if constexpr (RAGGED) {  // (as in pw_gemm_rows_kernel)
      const int skip = lq - min(lq, L - 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        ra[set][i] = moved_down(ra[set][i], skip);
        rb[set][i] = moved_down(rb[set][i], skip);
      }
    }
    if (edge_rows || tail) {
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        if (!(l_ok && m0 + rr + 32 * i < M)) ra[set][i] = (f32x4)(0.0f);
        if (!(l_ok && n0 + rr + 32 * i < N)) rb[set][i] = (f32x4)(0.0f);
      }
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int off = (rr + 32 * i) * kRowBytes + q4 * 8;
      {
        uint32_t w01[TA], w23[TA];
        const f32x4 v = ra[set][i];
        split_scaled_pair<TA, H>(v.x, v.y, a_scale, w01);
        split_scaled_pair<TA, H>(v.z, v.w, a_scale, w23);
#pragma unroll
        for (int t = 0; t < TA; ++t) {
          u32x2 w;
          w.x = w01[t];
          w.y = w23[t];
          *reinterpret_cast<u32x2 *>(As + set * kBuf + t * kRowPlane + off) = w;
        }
      }
      {
        uint32_t w01[TB], w23[TB];
        f32x4 v = rb[set][i];
        if (BITS) {  // (a whole sample is a multiple of 8 bits: the shift does not depend on the sample)
          const uint32_t e = b_off[i] + (uint32_t)lq;
          const uint32_t four = __builtin_bit_cast(uint32_t, rb[set][i].x) >> (e & 7u);
          v.x = (float)(four & 1u);
          v.y = (float)((four >> 1) & 1u);
          v.z = (float)((four >> 2) & 1u);
          v.w = (float)((four >> 3) & 1u);
        }
        split_scaled_pair<TB, H>(v.x, v.y, b_scale, w01);
        split_scaled_pair<TB, H>(v.z, v.w, b_scale, w23);
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          u32x2 w;
          w.x = w01[t];
          w.y = w23[t];
          *reinterpret_cast<u32x2 *>(Bs + set * kBuf + t * kRowPlane + off) = w;
        }
      }
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

  auto multiply = [&](int64_t it, int set) {
    // the second half of the last stage of a row (flat: of the chunk) may hold nothing
    const int ksteps = flat ? ((it + 1 == iters && total_quads - 8 * it <= 4) ? 1 : 2)
                            : (((int)(it % l_steps) * kTileK + 16 < L) ? 2 : 1);
    for (int ks = 0; ks < ksteps; ++ks) {
      u32x4 af[2][TA], bf[2][TB];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int t = 0; t < TA; ++t) af[mt][t] = row_fragment(As + set * kBuf + t * kRowPlane, wm * 64 + mt * 32 + (lane & 31), ks, lane);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int t = 0; t < TB; ++t) bf[nt][t] = row_fragment(Bs + set * kBuf + t * kRowPlane, wn * 64 + nt * 32 + (lane & 31), ks, lane);
      mfma_step<TA, TB, H>(af, bf, acc);
    }
  };
  if (iters > 0) fetch(0, 0);
  if (iters > 1) fetch(1, 1);
  int64_t it = 0;
  if constexpr (DOUBLE) {
    // step it: tile it + 1 (requested two steps ago) goes into the other LDS buffer, tile it + 3 is requested into the
    // registers that frees, tile it is multiplied; one barrier.  Requests are unconditional in the steady state only.
    auto step = [&](int64_t it, int set, bool stage_next, bool more) {
      if (stage_next) stage(it + 1, set ^ 1);
      if (more) fetch(it + 3, set ^ 1);
      __builtin_amdgcn_sched_barrier(0);
      multiply(it, set);
      __syncthreads();
    };
    if (iters > 0) stage(0, 0);
    if (iters > 2) fetch(2, 0);
    __syncthreads();
    for (; it + 4 < iters; it += 2) {
      step(it, 0, true, true);
      step(it + 1, 1, true, true);
    }
    if (it < iters) step(it, 0, it + 1 < iters, it + 3 < iters);
    if (it + 1 < iters) step(it + 1, 1, it + 2 < iters, false);
    if (it + 2 < iters) step(it + 2, 0, it + 3 < iters, false);
    if (it + 3 < iters) step(it + 3, 1, false, false);
  } else {
    // as in pw_gemm_kernel: unconditional requests in the steady state, conditions only in the last steps
    auto step = [&](int64_t it, int set, bool more) {
      __syncthreads();
      stage(it, set);
      __syncthreads();
      if (more) fetch(it + 2, set);
      multiply(it, set);
    };
    for (; it + 3 < iters; it += 2) {
      step(it, 0, true);
      step(it + 1, 1, true);
    }
    if (it < iters) step(it, 0, it + 2 < iters);
    if (it + 1 < iters) step(it + 1, 1, false);
    if (it + 2 < iters) step(it + 2, 0, false);
  }

  float *out = a.partials + (int64_t)chunk * M * N;
  if (H) {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[mt][nt][r] = acc[mt][nt][r] * a_inverse * b_inverse;
  }
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int col = n0 + wn * 64 + nt * 32 + (lane & 31);
    if (col >= N) continue;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int rbase = m0 + wm * 64 + mt * 32 + 4 * (lane >> 5);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = rbase + 8 * (r >> 2) + (r & 3);
        if (row < M) out[(int64_t)row * N + col] = acc[mt][nt][r];
      }
    }
  }
}

// pw_dw_flat_kernel: the weight gradient on fp16 terms where the contraction runs over the positions of all samples in a row (rows of at
// least eight quads), the same products as pw_dw_kernel.  That kernel's K step (qkv shape: dy [256, 1152, 196], x [256, 384, 196], cycles of
// a wavefront) was 1245 of split and LDS writes, 839 until the eight loads of the next tile had been accepted, 400 at barriers and 1301 of
// multiplication, one after the other, for 768 of the matrix cores.  Here
//   * the step is one straight line: behind every few multiplications stands a piece of the next tile's split and the request that
//     refills its registers, so that nothing is issued in a burst; two LDS buffers, one barrier; rows of 64 bytes with exchanged
//     chunks instead of padded ones, no bank conflicts.  With the requests taken out a step then takes 1606 cycles for two
//     wavefronts per SIMD, 1536 being the matrix cores' own;
//   * with them 2700: the loads bound it (128 x 128 tiles move 32 KB per step and tile through a compute unit's memory path).  A block is
//     eight wavefronts, 128 rows of dy by 128 WN of x: with WN = 3 64 KB for three tiles.  acc 96 + two tiles in flight 64 + fragments
//     of a half step and the next one's: 246 registers, two wavefronts per SIMD, one block per compute unit.
// Kernel and reduction, calls repeated on the same tensors, pw_dw_kernel / this one, us: this shape 208 / 168, x as bits 141 / 117; dy
// [128, 1536, 196], x [128, 384, 196] 137 / 116; both [256, 384, 196] 73 / 63; both [128, 512, 49] 43.2 / 29.8; both [16, 384, 196]
// 21.4 / 16.6; dy [4, 1152, 196], x [4, 384, 196] 19.7 / 15.3.  Inside a training step, where dy has just been written over: this shape
// 234 / 172, its projection (384 rows of dy, x as bits) 69 / 52, dy [128, 1536, 196] 159 / 142.
// No result is further from float64 than pw_dw_kernel's: sums of 32 bits are no longer than that kernel's chunks were (dw_longest_sum),
// where needed a chunk leaves several partial tiles.  With WN = 1 registers are left for sums of their own for the products of small
// terms: those of the large ones are rounded a third (one term of x: half) as often and may be longer.  Relative 2-norm of the error, before /
// now: qkv shape 4.6e-7 / 3.8e-7, spikes 2.5e-7 / 2.1e-7; [128, 512, 49] 1.48e-7 / 1.29e-7, spikes 9.8e-8 / 5.7e-8; dy [32, 1152, 64], x
// [32, 384, 64] 1.22e-7 / 1.14e-7; dy [20, 1376, 49], x [20, 480, 49] 1.19e-7 / 1.11e-7.
struct PwDwFlatArgs {
  const float *dy, *x;
  float *partials;
  int S, M, N, L, Lq;
  int m_blocks, n_blocks;
  int total_quads;      // S * Lq / 4
  int steps_per_chunk;  // K steps (eight quads) per partial tile
  int steps_per_sum;    // K steps, an even number, after which the accumulators go out and start again
  int sums;             // partial tiles per chunk: steps_per_chunk / steps_per_sum, rounded up
  const float *dy_amax, *x_amax;
};
constexpr int kDwThreads = 512;
constexpr int kDwRow = 64;  // bytes of a row of a plane: 32 fp16
constexpr unsigned dw_flat_buffer(int tb, int wn) { return (2u + (unsigned)(tb * wn)) * kTile * kDwRow; }
template <int TB, bool BITS, bool RAGGED, int WN>
__global__ void __launch_bounds__(kDwThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) pw_dw_flat_kernel(const PwDwFlatArgs a) {
  static_assert(!BITS || (TB == 1 && !RAGGED), "a bit-packed operand has one term and rows of a multiple of four");
  constexpr int TA = 2, NT = kTile * WN, kPlaneA = kTile * kDwRow, kPlaneB = NT * kDwRow, kBuf = (int)dw_flat_buffer(TB, WN);
  constexpr int UA = 2, UB = 2 * WN, U = UA + UB;  // 16-byte pieces of a K step per work-item: rows of dy, rows of x
  extern __shared__ __align__(16) uint8_t lds[];   // two buffers of [TA][128][kDwRow] of dy, then [TB][NT][kDwRow] of x
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 2, wn = wave & 3;
  const uint32_t logical = xcd_order32(blockIdx.x, gridDim.x);
  const uint32_t tiles = (uint32_t)(a.m_blocks * a.n_blocks);
  const uint32_t chunk = logical / tiles, tile = logical - chunk * tiles;
  const uint32_t nb = tile / (uint32_t)a.m_blocks, mb = tile - nb * (uint32_t)a.m_blocks;
  const int m0 = (int)mb * kTile, n0 = (int)nb * NT;
  const int M = a.M, N = a.N, L = a.L, Lq = RAGGED ? a.Lq : a.L;
  const int Q = Lq >> 2;  // quads (four positions) per sample, at least eight: the eight quads of a K step lie in two samples at most
  const int first_quad = (int)chunk * a.steps_per_chunk * 8;
  const int quads = min(a.steps_per_chunk * 8, a.total_quads - first_quad);  // of this chunk
  const int iters = (quads + 7) / 8;
  const uint32_t a_sample = (uint32_t)(M * L * 4), b_sample = (uint32_t)(N * L * (BITS ? 1 : 4));  // bytes; with BITS bits

  // a work-item fetches quad q4 of the rows rr + 64 i of both tiles.  Rows beyond the matrices repeat the last one: what they hold
  // reaches only rows and columns of the tile that are not written.
  const int q4 = tid & 7, rr = tid >> 3;
  uint32_t a_off[UA], b_off[UB];
#pragma unroll
  for (int i = 0; i < UA; ++i) a_off[i] = (uint32_t)(min(m0 + rr + 64 * i, M - 1) * L * 4);
#pragma unroll
  for (int i = 0; i < UB; ++i) b_off[i] = (uint32_t)(min(n0 + rr + 64 * i, N - 1) * L * (BITS ? 1 : 4));
  float a_scale = 1.0f, a_inverse = 1.0f, b_scale = 1.0f, b_inverse = 1.0f;

  // where a K step begins: sample, quad in it, quads of the chunk before it
  struct Place {
    int s, q, done = 0;
    __device__ __forceinline__ void next(int Q) {
      q += 8;
      done += 8;
      if (q >= Q) {
        q -= Q;
        ++s;
      }
    }
  };
  const int s_first = (int)((uint32_t)first_quad / (uint32_t)Q);
  Place fetched{s_first, first_quad - s_first * Q}, staged = fetched;
  f32x4 ra[2][UA], rb[2][UB];  // two tiles in flight; BITS: a byte in rb[..].x
  const char *pa, *pb;         // of the tile being fetched
  uint32_t la, lb;
  auto aim = [&]() {  // at the next tile to be fetched (quads beyond the chunk: some place in the tensors)
    int q = fetched.q + q4;
    const bool second = q >= Q;
    if (second) q -= Q;
    const bool ok = fetched.done + q4 < quads;
    const int l = ok ? (RAGGED ? min(4 * q, L - 4) : 4 * q) : 0;
    la = (uint32_t)l * 4u + (ok && second ? a_sample : 0u);
    lb = (BITS ? (uint32_t)l : (uint32_t)l * 4u) + (ok && second ? b_sample : 0u);
    const int64_t s = min(fetched.s, a.S - 1);
    pa = reinterpret_cast<const char *>(a.dy) + (s * M) * (int64_t)L * 4;
    pb = reinterpret_cast<const char *>(a.x) + (BITS ? ((s * N) * (int64_t)L >> 3) : (s * N) * (int64_t)L * 4);
    fetched.next(Q);
  };
  auto fetch_unit = [&](int u, int set) {
    if (u < UA) ra[set][u] = load4<RAGGED>(pa + (a_off[u] + la));
    else if constexpr (BITS) rb[set][u - UA].x = __builtin_bit_cast(float, (uint32_t)*reinterpret_cast<const uint8_t *>(pb + ((b_off[u - UA] + lb) >> 3)));
    else rb[set][u - UA] = load4<RAGGED>(pb + (b_off[u - UA] + lb));
  };
  // A row's four 16-byte chunks (eight positions each) are exchanged by bits 2 and 3 of the row: the 16 rows a 16-byte fragment read
  // of 16 lanes touches, and the four rows an 8-byte write of 32 lanes touches, fall on distinct banks
  const uint32_t w_at = (uint32_t)(rr * kDwRow + (((q4 >> 1) ^ ((rr >> 2) & 3)) << 4) + (q4 & 1) * 8);
  int place_q = 0, skip = 0;  // of the tile being staged
  bool place_ok = true;
  auto aim_stage = [&]() {
    int q = staged.q + q4;
    if (q >= Q) q -= Q;
    place_ok = staged.done + q4 < quads;
    place_q = place_ok ? 4 * q : 0;
    if (RAGGED) skip = place_q - min(place_q, L - 4);
    staged.next(Q);
  };
  auto stage_unit = [&](int u, int set, int buf, bool masked) {
    uint8_t *dst = lds + buf * kBuf + w_at + (u < UA ? u * (64 * kDwRow) : TA * kPlaneA + (u - UA) * (64 * kDwRow));
    f32x4 v = u < UA ? ra[set][u < UA ? u : 0] : rb[set][u < UA ? 0 : u - UA];
    if (u >= UA && BITS) {  // (a whole sample is a multiple of 8 bits: the shift does not depend on the sample)
      const uint32_t four = __builtin_bit_cast(uint32_t, v.x) >> ((b_off[u < UA ? 0 : u - UA] + (uint32_t)place_q) & 7u);
      u32x2 w = {(four & 1u) * 0x3c00u | (four & 2u) * 0x1e000000u, (four & 4u) * 0x0f00u | (four & 8u) * 0x07800000u};
      if (masked && !place_ok) w = (u32x2)(0u);
      *reinterpret_cast<u32x2 *>(dst) = w;
      return;
    }
    if constexpr (RAGGED) v = moved_down(v, skip);
    if (masked && !place_ok) v = (f32x4)(0.0f);
    if (u < UA) {
      uint32_t w01[TA], w23[TA];
      split_scaled_pair<TA, true>(v.x, v.y, a_scale, w01);
      split_scaled_pair<TA, true>(v.z, v.w, a_scale, w23);
#pragma unroll
      for (int t = 0; t < TA; ++t) *reinterpret_cast<u32x2 *>(dst + t * kPlaneA) = u32x2{w01[t], w23[t]};
    } else {
      uint32_t w01[TB], w23[TB];
      split_scaled_pair<TB, true>(v.x, v.y, b_scale, w01);
      split_scaled_pair<TB, true>(v.z, v.w, b_scale, w23);
#pragma unroll
      for (int t = 0; t < TB; ++t) *reinterpret_cast<u32x2 *>(dst + t * kPlaneB) = u32x2{w01[t], w23[t]};
    }
  };

  // SEP: the products of small terms have sums of their own, so that those of the large ones are rounded once where they would be three
  // times (one term of x: once for twice)
  constexpr bool SEP = WN == 1;
  f32x16 acc[2][WN], small[SEP ? 2 : 1][SEP ? WN : 1];
  auto clear = [&]() {
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int nt = 0; nt < WN; ++nt)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          acc[mt][nt][r] = 0.0f;
          if (SEP) small[SEP ? mt : 0][SEP ? nt : 0][r] = 0.0f;
        }
  };
  clear();
  const uint32_t r_at = (uint32_t)((lane & 31) * kDwRow + (((lane >> 5) ^ ((lane >> 2) & 3)) << 4));  // (the second half: bit 5 flipped)
  u32x4 af[2][2][TA], bf[2][WN][TB];  // [half][tile][term]
  auto read_term = [&](int buf, int ks, int ta, int tb) {  // the fragments of term ta of dy, tb of x (-1: none)
    const uint8_t *src = lds + buf * kBuf + (r_at ^ (ks * 32u));
    if (ta >= 0) {
#pragma unroll
      for (int t = 0; t < 2; ++t) af[ks][t][ta] = *reinterpret_cast<const u32x4 *>(src + ta * kPlaneA + (wm * 64 + t * 32) * kDwRow);
    }
    if (tb >= 0) {
#pragma unroll
      for (int t = 0; t < WN; ++t) bf[ks][t][tb] = *reinterpret_cast<const u32x4 *>(src + TA * kPlaneA + tb * kPlaneB + (wn * (32 * WN) + t * 32) * kDwRow);
    }
  };
  // Tile `it` (in LDS buffer P) is multiplied while tile it + 1 is split into the other buffer and tile it + 3 requested into the
  // registers that frees, a piece of either between every few multiplications.
  auto step = [&](auto parity, auto steady, bool stage_next, bool masked, bool more) {
    constexpr int P = decltype(parity)::value;
    constexpr bool STEADY = decltype(steady)::value;
    constexpr int kProducts = TB == 2 ? 3 : 2, kMfmas = 2 * kProducts * 2 * WN;
    if (STEADY || stage_next) aim_stage();
    if (STEADY || more) aim();
    read_term(P, 0, 0, TB - 1);
    read_term(P, 0, 1, TB == 2 ? 0 : -1);
    int n = 0, u = 0;
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int g = 0; g < kProducts; ++g) {
        // smallest terms first: (hi, lo), (lo, hi), (hi, hi); one term of x: (lo, x), (hi, x)
        const int ta = g == kProducts - 2 ? 1 : 0, tb = TB == 2 && g == 0 ? 1 : 0;
        if (ks == 0 && g == kProducts - 1) read_term(P, 1, 1, TB - 1);  // (into the registers of the small terms)
        if (ks == 1 && g == 0) read_term(P, 1, 0, TB == 2 ? 0 : -1);
#pragma unroll
        for (int mt = 0; mt < 2; ++mt)
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) {
            f32x16 &sum = SEP && g < kProducts - 1 ? small[SEP ? mt : 0][SEP ? nt : 0] : acc[mt][nt];
            sum = __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(f16x8, af[ks][mt][ta]), __builtin_bit_cast(f16x8, bf[ks][nt][tb]), sum, 0, 0, 0);
            ++n;
            if (n * U >= (u + 1) * kMfmas) {
              if (STEADY) {
                stage_unit(u, P ^ 1, P ^ 1, false);
                fetch_unit(u, P ^ 1);
                __builtin_amdgcn_sched_barrier(0);
              } else {
                if (stage_next) stage_unit(u, P ^ 1, P ^ 1, masked);
                if (more) fetch_unit(u, P ^ 1);
              }
              ++u;
            }
          }
      }
    __syncthreads();
  };

  // The accumulators into the next of the chunk's partial tiles.  (The address and the bounds pass through
  // an empty asm: out of the loop, where the compiler would keep them, the addresses and masks of 32 WN stores spill.  Not inlined
  // everywhere, the accumulators would live in scratch memory.)
  int64_t slot = (int64_t)chunk * a.sums;
  auto flush = [&]() __attribute__((always_inline)) {
    float *at = a.partials + (slot * M + (m0 + wm * 64 + 4 * (lane >> 5))) * N + (n0 + wn * (32 * WN) + (lane & 31));
    int rows_left = M - (m0 + wm * 64 + 4 * (lane >> 5)), cols_left = N - (n0 + wn * (32 * WN) + (lane & 31));
    asm volatile("" : "+v"(at), "+v"(rows_left), "+v"(cols_left));
#pragma unroll
    for (int mt = 0; mt < 2; ++mt)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        if (mt * 32 + 8 * (r >> 2) + (r & 3) < rows_left) {
#pragma unroll
          for (int nt = 0; nt < WN; ++nt) {
            const float sum = SEP ? acc[mt][nt][r] + small[SEP ? mt : 0][SEP ? nt : 0][r] : acc[mt][nt][r];
            if (nt * 32 < cols_left) at[nt * 32] = sum * a_inverse * b_inverse;
          }
        }
        at += (r & 3) < 3 ? N : 5 * N;
      }
    clear();
    ++slot;
  };

  const std::integral_constant<int, 0> even;
  const std::integral_constant<int, 1> odd;
  // (every block has a K step; tiles beyond the last are requested at some place of the tensors and not staged)
  aim();
#pragma unroll
  for (int u = 0; u < U; ++u) fetch_unit(u, 0);
  aim();
#pragma unroll
  for (int u = 0; u < U; ++u) fetch_unit(u, 1);
  if (a.dy_amax != nullptr) scale_for(tensor_amax(a.dy_amax), a_scale, a_inverse);
  if (TB > 1 && a.x_amax != nullptr) scale_for(tensor_amax(a.x_amax), b_scale, b_inverse);
  aim_stage();
#pragma unroll
  for (int u = 0; u < U; ++u) stage_unit(u, 0, 0, iters == 1);
  aim();
#pragma unroll
  for (int u = 0; u < U; ++u) fetch_unit(u, 0);
  __syncthreads();
  int it = 0, sum_end = a.steps_per_sum;
  auto cut = [&]() {  // before a pair of steps: a full sum goes out
    if (it >= sum_end) {
      flush();
      sum_end += a.steps_per_sum;
    }
  };
  for (; it + 4 < iters; it += 2) {  // (tile it + 2, staged by the second step, is not the last one)
    cut();
    step(even, std::true_type(), true, false, true);
    step(odd, std::true_type(), true, false, true);
  }
  for (; it < iters; it += 2) {  // at most four tiles are left; the last one may be partly empty
    cut();
    step(even, std::false_type(), it + 1 < iters, it + 2 >= iters, it + 3 < iters);
    if (it + 1 < iters) step(odd, std::false_type(), it + 2 < iters, it + 3 >= iters, false);
  }
  const int64_t slots_end = ((int64_t)chunk + 1) * a.sums;
  do flush();  // (again: a last chunk shorter than the others, the accumulators are zeros then)
  while (slot < slots_end);
}

struct PwDwPlanesArgs {
  const uint16_t *dy_planes;  // [2][M][ld] fp16 terms of dy, column s * L + l of row m holds dy[s][m][l]
  const uint16_t *x_planes;   // [TB][N][ld], likewise
  float *partials;            // [chunks][M][N]
  int64_t dy_plane_stride, x_plane_stride;  // M * ld, N * ld
  int64_t ncols;              // S * L
  int ld;
  int M, N;
  int64_t steps_per_chunk;    // K steps (32 columns each) per partial tile
  int m_blocks, n_blocks;
  const float *dy_amax, *x_amax;
};

// The weight gradient from term planes: dW[m][n] = sum_j dy[m][j] x[n][j] with both operands contiguous along the
// contraction index j (the columns of all samples in a row), so a tile of either is copied to LDS as it lies in memory,
// 16 bytes per work-item and row, and read back as fragments; no arithmetic on the way, and no sample boundaries.
template <int TB>
__global__ void __launch_bounds__(kPwThreads) __attribute__((amdgpu_waves_per_eu(2, 2))) pw_dw_planes_kernel(const PwDwPlanesArgs a) {
  constexpr int TA = 2;
  extern __shared__ __align__(16) uint8_t lds[];
  uint8_t *As = lds;                   // [TA][128][kRowBytes]
  uint8_t *Bs = lds + TA * kRowPlane;  // [TB][128][kRowBytes]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t logical = xcd_order(blockIdx.x, gridDim.x);
  const int tiles = a.m_blocks * a.n_blocks;
  const int chunk = (int)(logical / tiles);
  const int tile = (int)(logical % tiles);
  const int mb = tile % a.m_blocks, nb = tile / a.m_blocks;
  const int m0 = mb * kTile, n0 = nb * kTile;
  const int M = a.M, N = a.N;
  const int64_t steps_total = (a.ncols + kTileK - 1) / kTileK;
  const int64_t it_begin = (int64_t)chunk * a.steps_per_chunk;
  const int64_t it_end = it_begin + a.steps_per_chunk < steps_total ? it_begin + a.steps_per_chunk : steps_total;
  const int64_t iters = it_end - it_begin;

  // a work-item copies the 16-byte chunks q = tid and tid + 256 of a tile: row q / 4, eight columns 8 (q % 4)
  const uint32_t ld2 = (uint32_t)a.ld * 2u;
  uint32_t a_off[2], b_off[2];
  int dst[2];
  const int kc = tid & 3;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int row = (tid >> 2) + 64 * i;
    a_off[i] = (uint32_t)(m0 + row < M ? m0 + row : M - 1) * ld2;
    b_off[i] = (uint32_t)(n0 + row < N ? n0 + row : N - 1) * ld2;
    dst[i] = row * kRowBytes + kc * 16;
  }
  const bool edge_rows = __builtin_amdgcn_readfirstlane((m0 + kTile > M || n0 + kTile > N) ? 1 : 0) != 0;
  const char *dy_base = reinterpret_cast<const char *>(a.dy_planes);
  const char *x_base = reinterpret_cast<const char *>(a.x_planes);
  float a_scale, a_inverse = 1.0f, b_scale, b_inverse = 1.0f;
  if (a.dy_amax != nullptr) scale_for(tensor_amax(a.dy_amax), a_scale, a_inverse);
  if (TB > 1 && a.x_amax != nullptr) scale_for(tensor_amax(a.x_amax), b_scale, b_inverse);
  u32x4 ra[2][TA][2], rb[2][TB][2];  // two tiles in flight
  auto fetch = [&](int64_t it, int set) {
    const int64_t j = (it_begin + it) * kTileK;  // first column of the step; a chunk beyond the row is fetched from its start
    const uint32_t col = (j + 8 * kc < a.ld) ? (uint32_t)kc * 16u : 0u;
    const char *pa = dy_base + j * 2, *pb = x_base + j * 2;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int t = 0; t < TA; ++t) ra[set][t][i] = *reinterpret_cast<const u32x4 *>(pa + (int64_t)t * a.dy_plane_stride * 2 + (a_off[i] + col));
#pragma unroll
      for (int t = 0; t < TB; ++t) rb[set][t][i] = *reinterpret_cast<const u32x4 *>(pb + (int64_t)t * a.x_plane_stride * 2 + (b_off[i] + col));
    }
  };
  auto stage = [&](int64_t it, int set) {
    const int64_t j = (it_begin + it) * kTileK;
    const bool tail = j + kTileK > a.ncols;
    if (edge_rows || tail) {  // rows beyond the matrices and columns beyond the last sample hold zeros
      const int64_t left = a.ncols - (j + 8 * kc);
      const int nvalid = left < 0 ? 0 : (left > 8 ? 8 : (int)left);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int row = (tid >> 2) + 64 * i;
        const int na = m0 + row < M ? nvalid : 0, nb_ = n0 + row < N ? nvalid : 0;
#pragma unroll
        for (int t = 0; t < TA; ++t) {
          u32x4 &v = ra[set][t][i];
          v.x &= na >= 2 ? 0xffffffffu : (na == 1 ? 0xffffu : 0u);
          v.y &= na >= 4 ? 0xffffffffu : (na == 3 ? 0xffffu : 0u);
          v.z &= na >= 6 ? 0xffffffffu : (na == 5 ? 0xffffu : 0u);
          v.w &= na >= 8 ? 0xffffffffu : (na == 7 ? 0xffffu : 0u);
        }
#pragma unroll
        for (int t = 0; t < TB; ++t) {
          u32x4 &v = rb[set][t][i];
          v.x &= nb_ >= 2 ? 0xffffffffu : (nb_ == 1 ? 0xffffu : 0u);
          v.y &= nb_ >= 4 ? 0xffffffffu : (nb_ == 3 ? 0xffffu : 0u);
          v.z &= nb_ >= 6 ? 0xffffffffu : (nb_ == 5 ? 0xffffu : 0u);
          v.w &= nb_ >= 8 ? 0xffffffffu : (nb_ == 7 ? 0xffffu : 0u);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
#pragma unroll
      for (int t = 0; t < TA; ++t) *reinterpret_cast<u32x4 *>(As + t * kRowPlane + dst[i]) = ra[set][t][i];
#pragma unroll
      for (int t = 0; t < TB; ++t) *reinterpret_cast<u32x4 *>(Bs + t * kRowPlane + dst[i]) = rb[set][t][i];
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int mt = 0; mt < 2; ++mt)
#pragma unroll
    for (int nt = 0; nt < 2; ++nt)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mt][nt][r] = 0.0f;

  auto multiply = [&](int64_t it) {
    // the second half of the last step of the matrix may hold nothing
    const int ksteps = (a.ncols - (it_begin + it) * kTileK <= 16) ? 1 : 2;
    for (int ks = 0; ks < ksteps; ++ks) {
      u32x4 af[2][TA], bf[2][TB];
#pragma unroll
      for (int mt = 0; mt < 2; ++mt)
#pragma unroll
        for (int t = 0; t < TA; ++t) af[mt][t] = row_fragment(As + t * kRowPlane, wm * 64 + mt * 32 + (lane & 31), ks, lane);
#pragma unroll
      for (int nt = 0; nt < 2; ++nt)
#pragma unroll
        for (int t = 0; t < TB; ++t) bf[nt][t] = row_fragment(Bs + t * kRowPlane, wn * 64 + nt * 32 + (lane & 31), ks, lane);
      mfma_step<TA, TB, true>(af, bf, acc);
    }
  };
  // as in pw_gemm_kernel: unconditional requests in the steady state, conditions only in the last steps
  auto step = [&](int64_t it, int set, bool more) {
    __syncthreads();
    stage(it, set);
    __syncthreads();
    if (more) fetch(it + 2, set);
    multiply(it);
  };
  if (iters > 0) fetch(0, 0);
  if (iters > 1) fetch(1, 1);
  int64_t it = 0;
  for (; it + 3 < iters; it += 2) {
    step(it, 0, true);
    step(it + 1, 1, true);
  }
  if (it < iters) step(it, 0, it + 2 < iters);
  if (it + 1 < iters) step(it + 1, 1, false);
  if (it + 2 < iters) step(it + 2, 0, false);

  float *out = a.partials + (int64_t)chunk * M * N;
  const float inv = a_inverse * b_inverse;
#pragma unroll
  for (int nt = 0; nt < 2; ++nt) {
    const int col = n0 + wn * 64 + nt * 32 + (lane & 31);
    if (col >= N) continue;
#pragma unroll
    for (int mt = 0; mt < 2; ++mt) {
      const int rbase = m0 + wm * 64 + mt * 32 + 4 * (lane >> 5);
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int row = rbase + 8 * (r >> 2) + (r & 3);
        if (row < M) out[(int64_t)row * N + col] = acc[mt][nt][r] * inv;
      }
    }
  }
}

// planes[t][c][s * L + l] = term t of scale * x[s][c][l] for x [S][C][L] fp32: two fp16 terms (TERMS == 2: the scale is the
// power of two that the words of amax give, as in the kernels that split on the fly) or one (TERMS == 1: values that
// fp16 holds exactly, no scale).  A work-item takes four consecutive l.
template <int TERMS>
__global__ void __launch_bounds__(256) split_planes_kernel(const float *x, int64_t quads, int C, int L, const float *amax,
                                                            uint16_t *planes, int64_t plane_stride, int ld) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  float scale = 1.0f, inverse = 1.0f;
  if (TERMS > 1 && amax != nullptr) scale_for(tensor_amax(amax), scale, inverse);
  if (i >= quads) return;
  const int qpr = L >> 2;
  const int64_t row = i / qpr;  // s * C + c
  const int l = (int)(i - row * qpr) * 4;
  const int64_t s = row / C;
  const int c = (int)(row - s * C);
  f32x4 v = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(x) + i);
  v *= scale;
  uint32_t w01[TERMS], w23[TERMS];
  split_pair<TERMS, true>(v.x, v.y, w01);
  split_pair<TERMS, true>(v.z, v.w, w23);
  uint16_t *dst = planes + (int64_t)c * ld + s * L + l;
#pragma unroll
  for (int t = 0; t < TERMS; ++t) {
    u32x2 w;
    w.x = w01[t];
    w.y = w23[t];
    *reinterpret_cast<u32x2 *>(dst + (int64_t)t * plane_stride) = w;
  }
}

__global__ void __launch_bounds__(256) dw_reduce_scalar_kernel(const float *partials, int chunks, int64_t count, float *out) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= count) return;
  double sum = 0.0;
  for (int c = 0; c < chunks; ++c) sum += (double)partials[(int64_t)c * count + i];
  out[i] = (float)sum;
}

// count a multiple of 4 and 16-byte aligned buffers: four elements per work-item, the chunks in their order, eight
// loads in flight; in 64 bits, which the loads hide (error of the weight gradient against float64, relative 2-norm, [64, 512, 49]
// spikes, 96 output channels: 1.67e-7 with fp32 sums over the 64 chunks, 8.3e-8 now; the library's fp32 1.49e-7)
__global__ void __launch_bounds__(256) dw_reduce_kernel(const float *partials, int chunks, int64_t count, float *out) {
  const int64_t i = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) * 4;
  if (i >= count) return;
  typedef double f64x4 __attribute__((ext_vector_type(4)));
  f64x4 sum = {0.0, 0.0, 0.0, 0.0};
  int c = 0;
  auto add = [&](auto loads) {  // (all of them in flight before the first is used)
    constexpr int kLoads = decltype(loads)::value;
    for (; c + kLoads <= chunks; c += kLoads) {
      f32x4 v[kLoads];
#pragma unroll
      for (int u = 0; u < kLoads; ++u) v[u] = __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(partials + (int64_t)(c + u) * count + i));
#pragma unroll
      for (int u = 0; u < kLoads; ++u) sum += __builtin_convertvector(v[u], f64x4);
    }
  };
  add(std::integral_constant<int, 8>());
  add(std::integral_constant<int, 2>());
  add(std::integral_constant<int, 1>());
  *reinterpret_cast<f32x4 *>(out + i) = __builtin_convertvector(sum, f32x4);
}

int64_t round_up(int64_t v, int64_t m) { return (v + m - 1) / m * m; }
int64_t column_pitch(int64_t L) { return round_up(L, 4); }

template <int TA, int TB, bool H = false, int BSRC = kBFloat>
int launch_gemm_terms(const PwGemmArgs &a, int64_t blocks, hipStream_t stream) {
  unsigned lds = (TA + TB) * kRowPlane;
  if (a.stats && lds < kStatLds) lds = kStatLds;
  if (a.wide_out && lds < kOutLds) lds = kOutLds;
  hipLaunchKernelGGL((pw_gemm_kernel<TA, TB, H, BSRC>), dim3((unsigned)blocks), dim3(kPwThreads), lds, stream, a);
  return check_launch("pwconv_gemm");
}

// Rows of other lengths: compensated sums for one activation term, and for two up to so many K (see pw_gemm_rows_kernel).
constexpr int kCompensateK = 192;
template <int TB, bool BITS = false>
int launch_gemm_rows(const PwGemmArgs &a, int64_t blocks, hipStream_t stream) {
  const unsigned lds = rows_inverse_offset(TB) + kTile * 4;
  auto launch = [&](auto bits, auto sums) {
    hipLaunchKernelGGL((pw_gemm_rows_kernel<TB, decltype(bits)::value, decltype(sums)::value>), dim3((unsigned)blocks), dim3(kPwThreads), lds, stream, a);
  };
  if (BITS || a.L == a.Lq) launch(std::bool_constant<BITS>(), std::integral_constant<int, kOneChain>());
  else if (TB == 1 || a.K <= kCompensateK) launch(std::false_type(), std::integral_constant<int, kStepSumsCompensated>());
  else if constexpr (TB == 2) launch(std::false_type(), std::integral_constant<int, kStepSums>());
  return check_launch("pwconv_gemm");
}

template <int TA, int TB, bool H, bool BITS, bool RAGGED>
int launch_dw(const PwDwArgs &a, int64_t blocks, hipStream_t stream) {
  constexpr unsigned lds = (dw_two_buffers(H, TB) ? 2 : 1) * (TA + TB) * kRowPlane;
  static_assert(lds <= 64u * 1024u, "within the default limit of dynamic LDS");
  hipLaunchKernelGGL((pw_dw_kernel<TA, TB, H, BITS, RAGGED>), dim3((unsigned)blocks), dim3(kPwThreads), lds, stream, a);
  return check_launch("pwconv_grad_weight");
}
template <int TA, int TB, bool H = false, bool BITS = false>
int launch_dw_terms(const PwDwArgs &a, int64_t blocks, hipStream_t stream) {
  if constexpr (H && !BITS) {
    if (a.L != a.Lq) return launch_dw<TA, TB, H, false, true>(a, blocks, stream);
  }
  return launch_dw<TA, TB, H, BITS, false>(a, blocks, stream);
}

bool dw_flat(int64_t S, int64_t M, int64_t N, int64_t L) {
  return L >= 29 && M * L < (int64_t(1) << 29) && N * L < (int64_t(1) << 29) && S < (int64_t(1) << 31) && S * column_pitch(L) < (int64_t(1) << 31);
}

// Samples per partial tile of dW.  Two blocks are resident per compute unit (512 on the chip); the chunk count is the
// largest that keeps tiles x chunks within one (few tiles) or two full generations of resident blocks, so that no
// generation runs nearly empty.  Measured, kernel + reduction: 27 tiles: 38 chunks (1026 blocks) 312 + 11 us, 37 chunks
// 305 + 11, 19 chunks (513 blocks) 444 + 7, 18 chunks 318 + 7; 9 tiles: 114 chunks 101 + 11, 113 chunks 99 + 11,
// 56 chunks 85 + 7.
int dw_samples_per_chunk(int64_t S, int tiles) {
  const int rounds = tiles >= 16 ? 2 : 1;
  int64_t chunks = (int64_t)rounds * 512 / tiles;
  if (chunks < 1) chunks = 1;
  if (chunks > S) chunks = S;
  return (int)((S + chunks - 1) / chunks);
}

// How pw_dw_flat_kernel cuts a weight gradient: tiles of 128 x 128 wn, the contraction's K steps into `chunks` of `spc`, a chunk's sums
// into `sums` of `sps` steps (even: the steps run in pairs).  Wide tiles load least per multiplication, narrow ones fill the chip where
// there are few K steps; every partial tile is written and read once.  The fastest by this estimate of the widths and some numbers of
// chunks that fill the chip at most once: 6 us for a block's first loads and its end, per K step 0.2 us + 0.3 us for each 128 columns of
// multiplication and up to 0.35 us more for their loads with the whole chip at work (one term of x: less), partial tiles at 5.5 TB/s.
// The figures were fitted to calls repeated on the same tensors, which find in the cache in front of the memory what fits there.  Inside a
// training step narrow tiles take a quarter longer than estimated, wide ones a twentieth: dy [128, 1536, 196], x [128, 384, 196], for which
// the estimate prefers wn = 1 (113 us against 123), measured 138 + 7 there with wn = 1, 142 + 12 with 2, 110 + 18 with 3; dy
// [256, 1152, 196], x [256, 384, 196] (wn = 3) 211 + 7, 200 + 13, 156 + 17.
struct DwFlatPlan {
  int wn, m_blocks, n_blocks, chunks, spc, sums, sps;  // wn = 0: pw_dw_kernel
};
// partial tiles that pw_dw_kernel leaves, and the most that a plan may: as many more as fill the chip with the widest tiles
int64_t dw_sample_chunks(int64_t M, int64_t N, int64_t S) {
  const int spc = dw_samples_per_chunk(S, (int)(round_up(M, kTile) / kTile * (round_up(N, kTile) / kTile)));
  return (S + spc - 1) / spc;
}
int64_t dw_partial_tiles(int64_t M, int64_t N, int64_t S) {
  return dw_sample_chunks(M, N, S) + 768 / (round_up(M, kTile) / kTile * (round_up(N, kTile) / kTile)) + 1;
}
// K steps that a sum of 32 bits may hold, so that its error stays below that of pw_dw_kernel's sums over `quads` quads.  The error that
// rounding leaves in a sum grows with its length times the roundings per step:
//   * wide tiles round as that kernel does, after each product of terms: no longer than its sums;
//   * narrow ones round the sum of the large products a third as often: 5/2 of the length, where that is one step only (eight quads)
//     no more than it; with one term of x half as often: twice the length, less a step and a half for the addition of both sums at
//     the end (spikes, whose large products add up almost exactly, could take more, but not other values of one term; packed and
//     dense spikes give the same bits).
// Error against float64 / pw_dw_kernel's, 206 shapes of 29 to 400 positions: fp32 x 0.53 to 1.00, bfloat16 values in one term 0.50
// to 1.00, spikes 0.35 to 1.00.  (Before, with 5/2 for one term, and short lengths of wide tiles rounded up to two: up to 1.42, 1.49, 1.37.)
// With one term and sums of less than three steps so many partial tiles would be written that pw_dw_kernel is as fast, us flat / that
// kernel: [64, 256 x 256, 49] 26.5 / 19.7, [8, 1536 x 512, 81] 28.1 / 25.4, [32, 1152 x 384, 64] 30.8 / 28.9, [64, 1024 x 256, 64]
// 29.6 / 31.5; from three steps on it is not: [100, 1152 x 384, 32] 26.7 / 32.4.
constexpr int64_t kDwOneTermQuads = 24;
int64_t dw_longest_sum(int64_t quads, int wn, int x_terms) {
  if (wn > 1 || quads < 9) return quads / 8;
  return x_terms == 1 ? (quads - 6) / 4 : 5 * quads / 16;
}
DwFlatPlan dw_flat_plan(int64_t S, int64_t M, int64_t N, int64_t L, int dy_terms, int x_terms) {
  if (dy_terms != (SJHIP_PW_F16 | 2) || (x_terms != 1 && x_terms != 2) || !dw_flat(S, M, N, L)) return {};
  const int64_t steps = (S * (column_pitch(L) / 4) + 7) / 8;
  const int tiles128 = (int)(round_up(M, kTile) / kTile * (round_up(N, kTile) / kTile));
  const int64_t quads = dw_samples_per_chunk(S, tiles128) * (column_pitch(L) / 4);  // of pw_dw_kernel's sums
  if (x_terms == 1 && quads < kDwOneTermQuads) return {};
  const int64_t room = dw_partial_tiles(M, N, S);
  const float tile_us = (float)M * (float)N * 1.45e-6f;  // a partial tile written and read
  DwFlatPlan best = {};
  float best_us = 0.0f;
  for (int wn = 1; wn <= 3; ++wn) {
    DwFlatPlan p;
    p.wn = wn;
    p.m_blocks = (int)((M + kTile - 1) / kTile);
    p.n_blocks = (int)((N + kTile * wn - 1) / (kTile * wn));
    const int64_t tiles = (int64_t)p.m_blocks * p.n_blocks;
    const int64_t longest = dw_longest_sum(quads, wn, x_terms);
    const float width = (float)wn * (x_terms == 1 ? (wn == 1 ? 0.95f : 0.7f) : 1.0f);
    int64_t want = tiles >= 256 ? 1 : 256 / tiles;
    if (want > steps) want = steps;
    for (int k = 0; k < 6 && want >= 1; ++k, want = want * 5 / 8) {
      const int64_t spc = (steps + want - 1) / want, chunks = (steps + spc - 1) / spc;
      int64_t sums = 1, sps = round_up(spc, 2);
      if (spc > longest) {
        if (longest < 2) continue;  // (a sum of its own for every step would cost more than it gains)
        const int64_t even = longest / 2 * 2;
        sums = (spc + even - 1) / even;
        sps = round_up((spc + sums - 1) / sums, 2);
        sums = (spc + sps - 1) / sps;  // (an even length may need fewer)
      }
      if (chunks * sums > room) continue;
      const float rounds = (float)((tiles * chunks + 255) / 256), fill = fminf(1.0f, (float)(tiles * chunks) / 256.0f);
      const float us = rounds * (6.0f + (float)spc * (0.2f + (0.3f + 0.35f * fill) * width)) + (float)(chunks * sums) * tile_us;
      if (best.wn == 0 || us < best_us) {
        best_us = us;
        p.chunks = (int)chunks; p.spc = (int)spc; p.sums = (int)sums; p.sps = (int)sps;
        best = p;
      }
    }
  }
  return best;
}

}  // namespace

int64_t pwconv_planes_elems(int64_t rows, int64_t cols) { return 3 * round_up(rows, kTile) * round_up(cols, kTileK); }

int launch_pwconv_split_weight(const float *w, int64_t rows, int64_t cols, int transpose, uint16_t *planes,
                               hipStream_t stream) {
  // planes hold the matrix A of a later GEMM, K-contiguous: A = W ([rows][cols]) or A = W^T ([cols][rows])
  const int64_t ar = transpose ? cols : rows, ac = transpose ? rows : cols;
  const int64_t rows_pad = round_up(ar, kTile), cols_pad = round_up(ac, kTileK);
  const int64_t pairs = rows_pad * (cols_pad / 2);
  const int64_t blocks = (pairs + 255) / 256;
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_split_weight: %lld x %lld", (long long)rows, (long long)cols);
  hipLaunchKernelGGL(split_weight_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, w, ar, ac,
                     transpose ? (int64_t)1 : cols, transpose ? cols : (int64_t)1, rows_pad, cols_pad, planes);
  return check_launch("pwconv_split_weight");
}

int launch_pwconv_split_weight_f16(const float *w, int64_t rows, int64_t cols, int transpose, uint16_t *planes,
                                   float *amax_reset, int64_t amax_floats, hipStream_t stream) {
  const int64_t ar = transpose ? cols : rows, ac = transpose ? rows : cols;
  const int64_t rows_pad = round_up(ar, kTile), cols_pad = round_up(ac, kTileK);
  const int64_t blocks = rows_pad / 4;
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_split_weight_f16: %lld x %lld", (long long)rows, (long long)cols);
  if (transpose && !amax_reset) {
    const int64_t step_blocks = (cols_pad / kTileK + kSplitSteps - 1) / kSplitSteps;
    if (step_blocks <= 65535) {
      hipLaunchKernelGGL(split_weight_f16_transposed_kernel, dim3((unsigned)(rows_pad / 16), (unsigned)step_blocks), dim3(1024), 0, stream,
                         w, ar, ac, cols, rows_pad, cols_pad, planes);
      return check_launch("pwconv_split_weight_f16");
    }
  }
  hipLaunchKernelGGL(split_weight_f16_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, w, ar, ac,
                     transpose ? (int64_t)1 : cols, transpose ? cols : (int64_t)1, rows_pad, cols_pad, planes, amax_reset, amax_floats, BnEvalMap{});
  return check_launch("pwconv_split_weight_f16");
}

int launch_pwconv_split_weight_f16_bn(const float *w, int64_t rows, int64_t cols, uint16_t *planes, float *amax_reset,
                                      int64_t amax_floats, const BnEvalMap &bn, hipStream_t stream) {
  if (rows != bn.C || rows > (1 << 24) || !bn.running_mean || !bn.running_var)
    return fail(SJHIP_ERR_INVALID, "pwconv_split_weight_f16: %lld rows, batch norm of %d channels; evaluation mode needs the running statistics", (long long)rows, bn.C);
  const int64_t rows_pad = round_up(rows, kTile), cols_pad = round_up(cols, kTileK);
  hipLaunchKernelGGL(split_weight_f16_kernel, dim3((unsigned)(rows_pad / 4)), dim3(256), 0, stream, w, rows, cols, cols, (int64_t)1, rows_pad,
                     cols_pad, planes, amax_reset, amax_floats, bn);
  return check_launch("pwconv_split_weight_f16");
}

int launch_pwconv_amax(const float *x, int64_t S, int64_t per_sample, float *amax, hipStream_t stream) {
  const int64_t n = S * per_sample, blocks = (n + kAmaxChunk - 1) / kAmaxChunk;
  if (S > 0x7fffffffLL || blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_amax: %lld samples of %lld elements", (long long)S, (long long)per_sample);
  hipLaunchKernelGGL(amax_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, x, S, per_sample, reinterpret_cast<unsigned *>(amax));
  return check_launch("pwconv_amax");
}

namespace {
const int64_t kPwOffsetLimit = int64_t(1) << 30;  // per-lane offsets into A and B are 32-bit byte offsets
const int64_t kPwPlaneLimit = int64_t(1) << 30;   // elements of one fp16 plane: 32-bit byte offsets within it
int64_t gemm_samples_per_launch(int64_t K, int64_t L) { return (kPwOffsetLimit - 1) / (K * L); }
}  // namespace

int64_t pwconv_gemm_stats_rows(int64_t K, int64_t S, int64_t L) {
  if (K < 1 || L < 1 || K * L >= kPwOffsetLimit) return 0;
  const int64_t s_step = gemm_samples_per_launch(K, L);
  int64_t rows = 0;
  for (int64_t s0 = 0; s0 < S; s0 += s_step) {
    const int64_t s_count = S - s0 < s_step ? S - s0 : s_step;
    rows += 2 * ((s_count * column_pitch(L) + kTile - 1) / kTile);
  }
  return rows;
}

int launch_pwconv_gemm(const uint16_t *a_planes, int a_terms, int64_t M, int64_t K, const float *b, int b_terms,
                       const float *b_amax, int64_t S, int64_t L, float *c, float *stats, hipStream_t stream, bool b_bits) {
  // fp16 planes and at least four positions (bits: a multiple of four): the kernel that keeps A out of LDS, whose pieces are
  // four positions of one sample.  What is left of the fp16 forms for pw_gemm_kernel are two positions, and bits with L % 4 == 2.
  const bool rows_kernel = SJHIP_PW_ROWS != 0 && a_terms == (SJHIP_PW_F16 | 2) && (b_bits ? L % 4 == 0 && b_terms == 1 : L >= 4 && (b_terms == 1 || b_terms == 2));
  if ((L % 2 != 0 && !rows_kernel) || !aligned16(a_planes) || (!b_bits && (reinterpret_cast<uintptr_t>(b) & 7u)))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_gemm: L=%lld must be even (or, on fp16 planes and fp32 activations, at least 4), the weight planes 16-byte and the activations 8-byte aligned", (long long)L);
  if (b_bits && ((K * L) % 8 != 0 || a_terms != (SJHIP_PW_F16 | 2) || b_terms != 1))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_gemm: bit-packed activations need K*L=%lld to be a multiple of 8, fp16 weight planes and one activation term", (long long)(K * L));
  const int64_t limit = kPwOffsetLimit;
  if (round_up(M, kTile) * round_up(K, kTileK) >= limit || K * L >= limit)
    return fail(SJHIP_ERR_TOO_LARGE, "pwconv_gemm: M=%lld K=%lld L=%lld", (long long)M, (long long)K, (long long)L);
  const int64_t s_step = gemm_samples_per_launch(K, L);
  ProfileScope prof(KC_PW_GEMM, stream);
  for (int64_t s0 = 0; s0 < S; s0 += s_step) {
    const int64_t s_count = S - s0 < s_step ? S - s0 : s_step;
    PwGemmArgs a;
    a.a_planes = a_planes; a.c = c + s0 * M * L;
    a.b = b_bits ? reinterpret_cast<const float *>(reinterpret_cast<const uint8_t *>(b) + s0 * K * L / 8) : b + s0 * K * L;
    a.M = (int)M; a.K = (int)K; a.K_pad = (int)round_up(K, kTileK); a.L = (int)L; a.Lq = (int)column_pitch(L); a.inv_Lq = 1.0f / (float)a.Lq;
    a.plane_stride = round_up(M, kTile) * a.K_pad;
    a.ncols = s_count * a.Lq;
    a.m_blocks = (int)(round_up(M, kTile) / kTile);
    a.stats = stats;
    a.a_inverse = reinterpret_cast<const float *>(a_planes + 2 * a.plane_stride);
    a.b_amax = b_amax;
    a.b_amax_samples = b_amax ? b_amax + SJHIP_PW_AMAX_FLOATS : nullptr;
    a.amax_s0 = s0; a.amax_S = S;
    a.b_planes = nullptr; a.b_plane_stride = 0; a.ld = 0;
    a.wide_out = (SJHIP_PW_WIDE_OUT != 0 && L % 4 == 0 && aligned16(c)) ? 1 : 0;
    if (stats) stats += 2 * ((a.ncols + kTile - 1) / kTile) * M * 2;
    const int64_t blocks = a.m_blocks * ((a.ncols + kTile - 1) / kTile);
    if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_gemm: %lld blocks", (long long)blocks);
    int rc;
    if (rows_kernel) {
      rc = b_bits ? launch_gemm_rows<1, true>(a, blocks, stream)
                  : (b_terms == 2 ? launch_gemm_rows<2>(a, blocks, stream) : launch_gemm_rows<1>(a, blocks, stream));
      if (rc != SJHIP_OK) return rc;
      continue;
    }
    switch (a_terms * 10 + b_terms) {
      case 33: rc = launch_gemm_terms<3, 3>(a, blocks, stream); break;
      case 31: rc = launch_gemm_terms<3, 1>(a, blocks, stream); break;
      case 22: rc = launch_gemm_terms<2, 2>(a, blocks, stream); break;
      case 21: rc = launch_gemm_terms<2, 1>(a, blocks, stream); break;
      case 11: rc = launch_gemm_terms<1, 1>(a, blocks, stream); break;
      case (SJHIP_PW_F16 | 2) * 10 + 2: rc = launch_gemm_terms<2, 2, true>(a, blocks, stream); break;
      case (SJHIP_PW_F16 | 2) * 10 + 1:
        rc = b_bits ? launch_gemm_terms<2, 1, true, kBBits>(a, blocks, stream) : launch_gemm_terms<2, 1, true>(a, blocks, stream);
        break;
      default: return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_gemm: %d weight terms with %d activation terms (bf16: 3/3, 3/1, 2/2, 2/1, 1/1; fp16: 2/2, 2/1)", a_terms, b_terms);
    }
    if (rc != SJHIP_OK) return rc;
  }
  return SJHIP_OK;
}

int64_t pwconv_dw_workspace_floats(int64_t M, int64_t N, int64_t S) { return dw_partial_tiles(M, N, S) * M * N; }

int64_t pwconv_dw_workspace_floats_for(int64_t M, int64_t N, int64_t S, int64_t L, int dy_terms, int x_terms) {
  const DwFlatPlan plan = dw_flat_plan(S, M, N, L, dy_terms, x_terms);
  return (plan.wn != 0 ? (int64_t)plan.chunks * plan.sums : dw_sample_chunks(M, N, S)) * M * N;
}

template <int TB, bool BITS, bool RAGGED, int WN> static int launch_dw_flat(const PwDwFlatArgs &a, int64_t blocks, hipStream_t stream) {
  constexpr unsigned lds = 2 * dw_flat_buffer(TB, WN);
  if constexpr (lds > 64u * 1024u) {
    static OncePerDevice once;
    if (allow_dynamic_lds(once, reinterpret_cast<const void *>(&pw_dw_flat_kernel<TB, BITS, RAGGED, WN>), (int)lds) != hipSuccess)
      return fail(SJHIP_ERR_LAUNCH, "pwconv_grad_weight: %u bytes of LDS", lds);
  }
  hipLaunchKernelGGL((pw_dw_flat_kernel<TB, BITS, RAGGED, WN>), dim3((unsigned)blocks), dim3(kDwThreads), lds, stream, a);
  return check_launch("pwconv_grad_weight");
}

int launch_pwconv_grad_weight(const float *dy, int dy_terms, const float *dy_amax, const float *x, int x_terms,
                              const float *x_amax, int64_t S, int64_t M, int64_t N, int64_t L, float *dw, float *workspace,
                              hipStream_t stream, bool x_bits) {
  if (x_bits && ((N * L) % 8 != 0 || dy_terms != (SJHIP_PW_F16 | 2) || x_terms != 1))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_grad_weight: bit-packed activations need N*L=%lld to be a multiple of 8, two fp16 gradient terms and one activation term", (long long)(N * L));
  // (other lengths: fp16 terms only, the GEMM beside it has no bf16 form for them)
  if ((L % 4 != 0 && (x_bits || L < 4 || !(dy_terms & SJHIP_PW_F16))) || !aligned16(dy) || (!x_bits && !aligned16(x)))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_grad_weight: L=%lld must be a multiple of 4 (or, with fp16 terms and fp32 activations, at least 4) and the tensors 16-byte aligned", (long long)L);
  if (M * L >= (int64_t(1) << 30) || N * L >= (int64_t(1) << 30) || M * N >= (int64_t(1) << 40))  // 32-bit per-lane byte offsets
    return fail(SJHIP_ERR_TOO_LARGE, "pwconv_grad_weight: M=%lld N=%lld L=%lld", (long long)M, (long long)N, (long long)L);
  auto reduce = [&](int chunks) {
    const int64_t count = M * N;
    if (count % 4 == 0 && aligned16(workspace) && aligned16(dw))
      hipLaunchKernelGGL(dw_reduce_kernel, dim3((unsigned)((count / 4 + 255) / 256)), dim3(256), 0, stream, workspace, chunks, count, dw);
    else
      hipLaunchKernelGGL(dw_reduce_scalar_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, workspace, chunks, count, dw);
    return check_launch("pwconv_grad_weight(reduce)");
  };
  const DwFlatPlan plan = dw_flat_plan(S, M, N, L, dy_terms, x_terms);
  if (plan.wn != 0) {
    PwDwFlatArgs f;
    f.dy = dy; f.x = x; f.partials = workspace; f.dy_amax = dy_amax; f.x_amax = x_amax;
    f.S = (int)S; f.M = (int)M; f.N = (int)N; f.L = (int)L; f.Lq = (int)column_pitch(L);
    f.m_blocks = plan.m_blocks; f.n_blocks = plan.n_blocks;
    f.total_quads = (int)(S * f.Lq / 4);
    f.steps_per_chunk = plan.spc; f.steps_per_sum = plan.sps; f.sums = plan.sums;
    const int64_t blocks = (int64_t)plan.m_blocks * plan.n_blocks * plan.chunks;
    if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_grad_weight: %lld blocks", (long long)blocks);
    ProfileScope prof(KC_PW_GRAD_WEIGHT, stream);
    auto by_width = [&](auto terms, auto bits, auto ragged) {
      constexpr int TB = decltype(terms)::value;
      constexpr bool BITS = decltype(bits)::value, RAGGED = decltype(ragged)::value;
      if (plan.wn == 3) return launch_dw_flat<TB, BITS, RAGGED, 3>(f, blocks, stream);
      if (plan.wn == 2) return launch_dw_flat<TB, BITS, RAGGED, 2>(f, blocks, stream);
      return launch_dw_flat<TB, BITS, RAGGED, 1>(f, blocks, stream);
    };
    const std::integral_constant<int, 1> one;
    const std::integral_constant<int, 2> two;
    int rc;
    if (x_bits) rc = by_width(one, std::true_type(), std::false_type());
    else if (x_terms == 1) rc = L % 4 != 0 ? by_width(one, std::false_type(), std::true_type()) : by_width(one, std::false_type(), std::false_type());
    else rc = L % 4 != 0 ? by_width(two, std::false_type(), std::true_type()) : by_width(two, std::false_type(), std::false_type());
    return rc == SJHIP_OK ? reduce(plan.chunks * plan.sums) : rc;
  }
  PwDwArgs a;
  a.dy = dy; a.x = x; a.partials = workspace; a.S = S;
  a.dy_amax = dy_amax; a.x_amax = x_amax;
  a.flat = (L >= 32 && M * L < (int64_t(1) << 29) && N * L < (int64_t(1) << 29)) ? 1 : 0;
  a.M = (int)M; a.N = (int)N; a.L = (int)L; a.Lq = (int)column_pitch(L);
  a.m_blocks = (int)(round_up(M, kTile) / kTile);
  a.n_blocks = (int)(round_up(N, kTile) / kTile);
  const int tiles = a.m_blocks * a.n_blocks;
  a.s_per_chunk = dw_samples_per_chunk(S, tiles);
  const int chunks = (int)((S + a.s_per_chunk - 1) / a.s_per_chunk);
  const int64_t blocks = (int64_t)tiles * chunks;
  int rc;
  {
    ProfileScope prof(KC_PW_GRAD_WEIGHT, stream);
    const int key = dy_terms * 10 + x_terms;
    switch (key) {
      case 33: rc = launch_dw_terms<3, 3>(a, blocks, stream); break;
      case 31: rc = launch_dw_terms<3, 1>(a, blocks, stream); break;
      case 22: rc = launch_dw_terms<2, 2>(a, blocks, stream); break;
      case 21: rc = launch_dw_terms<2, 1>(a, blocks, stream); break;
      case 11: rc = launch_dw_terms<1, 1>(a, blocks, stream); break;
      case (SJHIP_PW_F16 | 2) * 10 + 2: rc = launch_dw_terms<2, 2, true>(a, blocks, stream); break;
      case (SJHIP_PW_F16 | 2) * 10 + 1:
        rc = x_bits ? launch_dw_terms<2, 1, true, true>(a, blocks, stream) : launch_dw_terms<2, 1, true>(a, blocks, stream);
        break;
      default: return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_grad_weight: %d gradient terms with %d activation terms (bf16: 3/3, 3/1, 2/2, 2/1, 1/1; fp16: 2/2, 2/1)", dy_terms, x_terms);
    }
    if (rc != SJHIP_OK) return rc;
    rc = reduce(chunks);
  }
  return rc;
}

// ---- operands that arrive as fp16 term planes -------------------------------------------------------------------------
namespace {
// K steps per partial tile of the weight gradient from planes: as dw_samples_per_chunk, over the steps of 32 columns
int64_t dw_planes_steps_per_chunk(int64_t ncols, int tiles) {
  const int64_t steps = (ncols + kTileK - 1) / kTileK;
  const int rounds = tiles >= 16 ? 2 : 1;
  int64_t chunks = (int64_t)rounds * 512 / tiles;
  if (chunks < 1) chunks = 1;
  if (chunks > steps) chunks = steps > 0 ? steps : 1;
  return (steps + chunks - 1) / chunks;
}
}  // namespace

int64_t pwconv_plane_ld(int64_t S, int64_t L) { return round_up(S * L, 8); }

int launch_pwconv_split_planes(const float *x, int64_t S, int64_t C, int64_t L, int terms, const float *amax, uint16_t *planes,
                               hipStream_t stream) {
  if (S < 1 || C < 1 || L < 1 || L % 4 != 0 || !aligned16(x) || !aligned16(planes) || (terms != 1 && terms != 2))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_split_planes: S=%lld C=%lld L=%lld (a multiple of 4), %d terms (1 or 2), 16-byte aligned buffers", (long long)S, (long long)C, (long long)L, terms);
  if (terms == 2 && (amax == nullptr || !aligned16(amax)))
    return fail(SJHIP_ERR_INVALID, "pwconv_split_planes: two terms need the 16-byte aligned amax buffer of the tensor");
  const int64_t ld = pwconv_plane_ld(S, L);
  if (C > (1 << 24) || L > (1 << 24) || C * ld >= kPwPlaneLimit)
    return fail(SJHIP_ERR_TOO_LARGE, "pwconv_split_planes: S=%lld C=%lld L=%lld", (long long)S, (long long)C, (long long)L);
  const int64_t quads = S * C * (L / 4), blocks = (quads + 255) / 256;
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_split_planes: %lld elements", (long long)(quads * 4));
  if (terms == 2)
    hipLaunchKernelGGL(split_planes_kernel<2>, dim3((unsigned)blocks), dim3(256), 0, stream, x, quads, (int)C, (int)L, amax, planes, C * ld, (int)ld);
  else
    hipLaunchKernelGGL(split_planes_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, stream, x, quads, (int)C, (int)L, amax, planes, C * ld, (int)ld);
  return check_launch("pwconv_split_planes");
}

int64_t pwconv_gemm_planes_stats_rows(int64_t S, int64_t L) { return 2 * ((S * L + kTile - 1) / kTile); }

int launch_pwconv_gemm_planes(const uint16_t *a_planes, int64_t M, int64_t K, const uint16_t *b_planes, int b_terms,
                              const float *b_amax, int64_t S, int64_t L, float *c, float *stats, hipStream_t stream) {
  if (M < 1 || K < 1 || S < 1 || L < 1 || !aligned16(a_planes) || !aligned16(b_planes) || (b_terms != 1 && b_terms != 2))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_gemm_planes: M=%lld K=%lld S=%lld L=%lld, %d activation terms (1 or 2), 16-byte aligned planes", (long long)M, (long long)K, (long long)S, (long long)L, b_terms);
  if (b_terms == 2 && (b_amax == nullptr || !aligned16(b_amax)))
    return fail(SJHIP_ERR_INVALID, "pwconv_gemm_planes: two activation terms need the 16-byte aligned amax buffer they were scaled by");
  const int64_t ld = pwconv_plane_ld(S, L);
  if (round_up(M, kTile) * round_up(K, kTileK) >= kPwOffsetLimit || K * ld >= kPwPlaneLimit || M * L >= (int64_t(1) << 40))
    return fail(SJHIP_ERR_TOO_LARGE, "pwconv_gemm_planes: M=%lld K=%lld S=%lld L=%lld", (long long)M, (long long)K, (long long)S, (long long)L);
  PwGemmArgs a;
  a.a_planes = a_planes; a.b = nullptr; a.c = c;
  a.M = (int)M; a.K = (int)K; a.K_pad = (int)round_up(K, kTileK); a.L = a.Lq = (int)L; a.inv_Lq = 1.0f / (float)L;
  a.plane_stride = round_up(M, kTile) * a.K_pad;
  a.ncols = S * L;
  a.m_blocks = (int)(round_up(M, kTile) / kTile);
  a.stats = stats;
  a.a_inverse = reinterpret_cast<const float *>(a_planes + 2 * a.plane_stride);
  a.b_amax = b_terms == 2 ? b_amax : nullptr;
  a.b_amax_samples = nullptr; a.amax_s0 = 0; a.amax_S = 0;
  a.b_planes = b_planes; a.b_plane_stride = K * ld; a.ld = (int)ld;
  a.wide_out = (SJHIP_PW_WIDE_OUT != 0 && L % 4 == 0 && aligned16(c)) ? 1 : 0;
  const int64_t blocks = a.m_blocks * ((a.ncols + kTile - 1) / kTile);
  if (blocks > 0x7fffffffLL) return fail(SJHIP_ERR_TOO_LARGE, "pwconv_gemm_planes: %lld blocks", (long long)blocks);
  ProfileScope prof(KC_PW_GEMM, stream);
  return b_terms == 2 ? launch_gemm_terms<2, 2, true, kBPlanes>(a, blocks, stream)
                      : launch_gemm_terms<2, 1, true, kBPlanes>(a, blocks, stream);
}

int64_t pwconv_dw_planes_workspace_floats(int64_t M, int64_t N, int64_t S, int64_t L) {
  const int tiles = (int)(round_up(M, kTile) / kTile * (round_up(N, kTile) / kTile));
  const int64_t steps = (S * L + kTileK - 1) / kTileK, spc = dw_planes_steps_per_chunk(S * L, tiles);
  return (steps + spc - 1) / spc * M * N;
}

int launch_pwconv_grad_weight_planes(const uint16_t *dy_planes, const float *dy_amax, const uint16_t *x_planes, int x_terms,
                                     const float *x_amax, int64_t S, int64_t M, int64_t N, int64_t L, float *dw,
                                     float *workspace, hipStream_t stream) {
  if (M < 1 || N < 1 || S < 1 || L < 1 || !aligned16(dy_planes) || !aligned16(x_planes) || (x_terms != 1 && x_terms != 2))
    return fail(SJHIP_ERR_UNSUPPORTED, "pwconv_grad_weight_planes: M=%lld N=%lld S=%lld L=%lld, %d activation terms (1 or 2), 16-byte aligned planes", (long long)M, (long long)N, (long long)S, (long long)L, x_terms);
  if (dy_amax == nullptr || !aligned16(dy_amax) || (x_terms == 2 && (x_amax == nullptr || !aligned16(x_amax))))
    return fail(SJHIP_ERR_INVALID, "pwconv_grad_weight_planes: operands of two terms need the 16-byte aligned amax buffers they were scaled by");
  const int64_t ld = pwconv_plane_ld(S, L);
  if (M * ld >= kPwPlaneLimit || N * ld >= kPwPlaneLimit || M * N >= (int64_t(1) << 40))
    return fail(SJHIP_ERR_TOO_LARGE, "pwconv_grad_weight_planes: M=%lld N=%lld S=%lld L=%lld", (long long)M, (long long)N, (long long)S, (long long)L);
  PwDwPlanesArgs a;
  a.dy_planes = dy_planes; a.x_planes = x_planes; a.partials = workspace;
  a.dy_plane_stride = M * ld; a.x_plane_stride = N * ld; a.ncols = S * L; a.ld = (int)ld;
  a.M = (int)M; a.N = (int)N;
  a.m_blocks = (int)(round_up(M, kTile) / kTile);
  a.n_blocks = (int)(round_up(N, kTile) / kTile);
  a.dy_amax = dy_amax; a.x_amax = x_terms == 2 ? x_amax : nullptr;
  const int tiles = a.m_blocks * a.n_blocks;
  a.steps_per_chunk = dw_planes_steps_per_chunk(a.ncols, tiles);
  const int64_t steps = (a.ncols + kTileK - 1) / kTileK;
  const int chunks = (int)((steps + a.steps_per_chunk - 1) / a.steps_per_chunk);
  const int64_t blocks = (int64_t)tiles * chunks;
  ProfileScope prof(KC_PW_GRAD_WEIGHT, stream);
  const unsigned lds = (2 + x_terms) * kRowPlane;
  if (x_terms == 2) hipLaunchKernelGGL(pw_dw_planes_kernel<2>, dim3((unsigned)blocks), dim3(kPwThreads), lds, stream, a);
  else hipLaunchKernelGGL(pw_dw_planes_kernel<1>, dim3((unsigned)blocks), dim3(kPwThreads), lds, stream, a);
  int rc = check_launch("pwconv_grad_weight_planes");
  if (rc != SJHIP_OK) return rc;
  const int64_t count = M * N;
  if (count % 4 == 0 && aligned16(workspace) && aligned16(dw))
    hipLaunchKernelGGL(dw_reduce_kernel, dim3((unsigned)((count / 4 + 255) / 256)), dim3(256), 0, stream, workspace, chunks, count, dw);
  else
    hipLaunchKernelGGL(dw_reduce_scalar_kernel, dim3((unsigned)((count + 255) / 256)), dim3(256), 0, stream, workspace, chunks, count, dw);
  return check_launch("pwconv_grad_weight_planes(reduce)");
}

}  // namespace sjhip
