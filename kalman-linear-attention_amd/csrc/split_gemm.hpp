// split_gemm.hpp -- y = x W^T in fp32 on the fp16 matrix cores, on gfx950.
//
// The fp32 MFMA of gfx950 runs at a sixteenth of the fp16 rate. An fp32 value
// scaled to |s| < 2^15 is the sum of two fp16 values hi = fp16(s) and
// lo = fp16(s - hi) up to one unit of its own last place (hi carries 11 bits,
// lo 11 more and the sign a bit), so
//   x w = hi_x hi_w + hi_x lo_w + lo_x hi_w   (+ lo_x lo_w, below 2^-22 of it)
// with every product exact and every sum fp32: three MFMA products, a third of
// the fp16 rate, and sums that round three times a 16-wide step of k instead of
// up to 16 times. A sum of many terms is so closer to the exact one than the fp32
// product's, a sum of few is not. Relative error (2-norm) against float64, normal
// entries, this product / the library's fp32 product: k = 1 8.1e-8 / 2.5e-8, k = 4
// 8.2e-8 / 4.0e-8, k = 16 8.8e-8 / 7.4e-8, k = 28 9.7e-8 / 9.6e-8, k = 32 9.5e-8 /
// 1.03e-7, k = 64 1.1e-7 / 1.4e-7, k = 512 2.6e-7 / 4.1e-7, k = 1024 3.6e-7 /
// 5.7e-7, k = 1365 4.1e-7 / 6.6e-7, k = 2048 5.0e-7 / 8.1e-7.
//
// Each row of x and of W is scaled by the power of two that brings its largest
// magnitude into [2^14, 2^15); the scales go back in with one ldexp per output.
// Entries more than 2^16 below their row's largest lose low bits of lo to fp16's
// smallest spacing, up to 2^-39 of the row's largest value each: nothing beside the
// row's other terms, but all there is where those are multiplied by zeros (a feature
// of 1e9 that the weights ignore). So the row split counts c, the entries that lose,
// and h, those below 2^6 at the row's scale. The other operand lies below 2^15, so an
// output is off by (c_x + c_w) 2^-10 of its scale at most. At least k - h_x - h_w of its
// terms are 2^12 and more, so their fp32 rounding alone comes to 2^-12 of that number:
// where h + 4 c of the two rows is k or less, no fp32 sum promises more. Rows of
// dense weights and activations have 0.01 to 0.3 k of it, ReLU's 0.55 k. Where it is
// more, an output that the loss could move by more than 2^-26 sqrt(k) of the sum the
// matrix cores gave is summed in plain fp32 from the operands (split_exact_block), as
// is every output of a row with an infinity or a NaN. (That is 0.83 of the fp32
// product's 2-norm error, for losses that all add up against the other operand's
// largest value; over 400 random pairs of operands of wide range 2^-23 in its place
// gave the same largest error.) 8188 x 4096, k 1024, this product / the library's, us:
// normal entries 210 / 501; one row of NaNs 321 / 483; every output formed again 1130 /
// 475; one feature of 1.7e9 778 / 486; log-normal entries of sigma 1 210 / 500, 4 1170 /
// 476.
//
// What surrounds a product in a block is folded in: before it the RMSNorm of x's
// rows (formed as the rows are split, never stored in fp32: 13.1 us at 4096 x 512
// with W [2730, 512], against 7.2 + 11.9 apart), after it the residual add (22 us
// against 21 + 5.4) or the MLP's SwiGLU (whose gate and up features lie in
// neighbouring 32-row blocks of the split W, so one wave holds both: 42 us against
// 66 + 13.6). The layer's skip and gate before out_proj stay a kernel of their own:
// formed here their three operands' loads wait on one another, 29 us at 2048 x
// 1024 against 9 + 11 apart.
//
// Two kernels. split_rows_kernel writes both operands' hi and lo planes in the
// order the product reads them: 1 KiB fragments of 32 rows x 16 k, a lane's
// eight fp16 contiguous, so that the product moves them with 16-byte accesses
// through LDS and straight into the MFMA operands, with no transposition and no
// bank conflicts. split_gemm_kernel is the tiled product.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "causal_conv.hpp"
#include "scan_ops.hpp"

namespace kla {

typedef _Float16 f16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));

constexpr int kSplitRows = 32;                       // rows of a fragment
constexpr int kSplitK = 32;                          // k of a pair of fragments (a chunk)
constexpr int kSplitChunk = kSplitRows * kSplitK * 2;   // fp16 of a chunk: 2 k halves x 2 planes x 512
constexpr int kSplitExp = 14;                        // scaled rows lie in [2^14, 2^15)
// A row's word. Its exponent + kSplitBias; kSplitZero for a row of zeros; the least sum
// that may stand against its loss, c 2^16 / sqrt(k), as the exponent of a float,
// rounded up (infinite for a row with an infinity or a NaN); and
// h + 4 c in units of k / kSplitShare, rounded up.
constexpr int kSplitBias = 160, kSplitShare = 8192;
constexpr uint32_t kSplitZero = 1u << 23;
constexpr uint32_t kSplitNoRow = kSplitZero | kSplitBias << 14;

__device__ __forceinline__ int split_exp(uint32_t word) { return static_cast<int>(word >> 14 & 0x1ff) - kSplitBias; }
__device__ __forceinline__ float split_lost(uint32_t word) { return __uint_as_float(word >> 24 << 23); }
__device__ __forceinline__ int split_share(uint32_t word) { return static_cast<int>(word & 0x3fff); }

struct SplitOperand {
  const float *src;    // [rows, k], row stride ld
  int64_t ld, rows;
  _Float16 *dst;       // [blocks][chunks][2 k halves][2 planes][64 lanes][8]
  uint32_t *words;     // [blocks * 32]: by row, s = src * 2^(kSplitExp - split_exp(word))
  int64_t blocks;      // 32-row blocks
};

struct SplitParams {
  SplitOperand op[2];  // x, W
  int64_t k;
  int64_t chunks;      // ceil(k / 32)
  float share, least;  // kSplitShare / k, 2^16 / sqrt(k)
  // NORM: x -> (x * rsqrt(mean(x^2) + eps)) * norm_w
  const float *norm_w;
  float eps;
  // Nonzero: W's blocks alternate between rows 32 i .. (gate) and glu_off + 32 i ..
  // (up) of two halves of glu_rows rows.
  int64_t glu_off, glu_rows;
};

// One workgroup takes 32 rows. Lane l of a wave holds, for each of the wave's
// chunks, the 16 values k = 32 chunk + 16 (l / 32) + 0..15 of row l % 32 (64
// contiguous bytes: the two halves of a wave read whole 128-byte lines), and
// fragment f of the chunk is its values 8 f .. 8 f + 7. Which k a lane's eight
// values are does not matter to the product as long as both operands agree.
// NC > 0: the chunks of a wave stay in registers between the row maximum and
// the conversion (at most NC of them); NC = 0 reads the rows twice. It moves 8
// bytes an element (read, written), at 3.6 to 4.5 TB/s from 4096 rows on.
constexpr int kSplitThreads = 512;

// Four floats at any 4-byte boundary: global loads of gfx950 need no more, so
// rows of odd length ([512, 1365]) load as widely as aligned ones.
typedef float f32x4_any_t __attribute__((ext_vector_type(4), aligned(4)));

template <int N>
__device__ __forceinline__ void split_load(float (&x)[N], const float *row, int64_t k0, int64_t k) {
#pragma unroll
  for (int i = 0; i < N / 4; ++i) {
    f32x4_any_t v = {0.0f, 0.0f, 0.0f, 0.0f};
    const int64_t at = k0 + 4 * i;
    if (at + 4 <= k) {
      v = *reinterpret_cast<const f32x4_any_t *>(row + at);
    } else {
      if (at < k) v.x = row[at];
      if (at + 1 < k) v.y = row[at + 1];
      if (at + 2 < k) v.z = row[at + 2];
    }
    x[4 * i] = v.x;
    x[4 * i + 1] = v.y;
    x[4 * i + 2] = v.z;
    x[4 * i + 3] = v.w;
  }
}

template <int NC, bool NORM>
__global__ void __launch_bounds__(kSplitThreads) split_rows_kernel(SplitParams p) {
  constexpr int NWV = kSplitThreads / kWave;
  __shared__ uint32_t s_max[NWV][kSplitRows];
  __shared__ float s_sum[NORM ? NWV : 1][kSplitRows];
  __shared__ int s_count[2][NWV][kSplitRows];
  const bool second = static_cast<int64_t>(blockIdx.x) >= p.op[0].blocks;
  const SplitOperand &op = p.op[second ? 1 : 0];
  const int64_t blk = static_cast<int64_t>(blockIdx.x) - (second ? p.op[0].blocks : 0);
  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid % kWave, wave = tid / kWave;
  const int r = lane % kSplitRows, half = lane / kSplitRows;
  int64_t row = blk * kSplitRows + r;
  bool in = row < op.rows;
  if (second && p.glu_off) {
    row = (blk / 2) * kSplitRows + r;
    in = row < p.glu_rows;
    row += blk % 2 ? p.glu_off : 0;
  }
  const int64_t src_row = in ? row : 0, kin = in ? p.k : 0;
  const float *src = op.src + src_row * op.ld;
  const bool norm = NORM && !second;

  auto load = [&](float (&v)[16], int64_t ch) { split_load(v, src, ch * kSplitK + 16 * half, kin); };

  constexpr int HELD = NC > 0 ? NC : 1;
  float x[HELD][16];
  uint32_t top = 0;     // the largest magnitude's bits (of x norm_w, before the row's scale, with the norm)
  float squares = 0.0f;
  auto scan = [&](const float (&v)[16], int64_t ch) {
    float w[16];
    if (norm) split_load(w, p.norm_w, ch * kSplitK + 16 * half, kin);
#pragma unroll
    for (int i = 0; i < 16; ++i) {
      uint32_t b = __float_as_uint(v[i]) & 0x7fffffffu;
      if (norm) {
        squares = fmaf(v[i], v[i], squares);
        const uint32_t c = __float_as_uint(v[i] * w[i]) & 0x7fffffffu;
        b = b >= 0x7f800000u ? b : c;
      }
      top = b > top ? b : top;
    }
  };
  if constexpr (NC > 0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) load(x[i], wave + static_cast<int64_t>(i) * NWV);
#pragma unroll
    for (int i = 0; i < NC; ++i) scan(x[i], wave + static_cast<int64_t>(i) * NWV);
  } else {
    for (int64_t ch = wave; ch < p.chunks; ch += NWV) {
      load(x[0], ch);
      scan(x[0], ch);
    }
  }
  const uint32_t other = __shfl_xor(top, 32);
  top = other > top ? other : top;
  if (half == 0) s_max[wave][r] = top;
  if constexpr (NORM) {
    squares += __shfl_xor(squares, 32);
    if (half == 0) s_sum[wave][r] = squares;
  }
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NWV; ++w) top = s_max[w][r] > top ? s_max[w][r] : top;
  float scale = 1.0f;
  if constexpr (NORM) {
    if (norm) {
      float ss = 0.0f;
#pragma unroll
      for (int w = 0; w < NWV; ++w) ss += s_sum[w][r];
      scale = rsqrtf(ss / static_cast<float>(p.k) + p.eps);
    }
  }
  // (With the norm the bound on the row's largest magnitude may round up to a power
  // of two: |s| then stays below 2^15 (1 + 2^-22).)
  const bool marked = top >= 0x7f800000u;
  float bound = __uint_as_float(top);
  if (NORM && !marked) bound *= scale;
  // The exponent of the row's largest magnitude (that of 1 for a row of zeros).
  int ex = 0;
  if (!marked && bound != 0.0f) ex = __builtin_amdgcn_frexp_expf(bound) - 1;

  int lossy = 0, small = 0;    // this lane's part of c and h
  const int shift = kSplitExp - ex;
  // What loses: 0 < |u| < 2^-2 of the row's scale (from there on lo is good to 2^-23 of s),
  // as one unsigned comparison of the bits without the sign.
  const uint32_t quarter = __float_as_uint(ldexpf(0.25f, -shift)) << 1;
  const uint32_t below = quarter ? quarter - 1 : 0;
  auto put = [&](const float (&v)[16], int64_t ch) {
    _Float16 *out = op.dst + (blk * p.chunks + ch) * kSplitChunk + lane * 8;
    float w[16];
    if (norm) split_load(w, p.norm_w, ch * kSplitK + 16 * half, kin);
#pragma unroll
    for (int f = 0; f < 2; ++f) {
      f16x8_t hi, lo;
#pragma unroll
      for (int i = 0; i < 8; ++i) {
        const float u = norm ? (v[8 * f + i] * scale) * w[8 * f + i] : v[8 * f + i];
        const float s = ldexpf(u, shift);
        hi[i] = static_cast<_Float16>(s);
        lo[i] = static_cast<_Float16>(s - static_cast<float>(hi[i]));
        small += fabsf(s) < 0x1p6f;
        lossy += (__float_as_uint(u) << 1) - 1 < below;
      }
      *reinterpret_cast<f16x8_t *>(out + (2 * f) * 512) = hi;
      *reinterpret_cast<f16x8_t *>(out + (2 * f + 1) * 512) = lo;
    }
  };
  if constexpr (NC > 0) {
#pragma unroll
    for (int i = 0; i < NC; ++i) {
      const int64_t ch = wave + static_cast<int64_t>(i) * NWV;
      if (ch < p.chunks) put(x[i], ch);
    }
  } else {
    for (int64_t ch = wave; ch < p.chunks; ch += NWV) {
      load(x[0], ch);
      put(x[0], ch);
    }
  }
  lossy += __shfl_xor(lossy, 32);
  small += __shfl_xor(small, 32);
  if (half == 0) s_count[0][wave][r] = lossy, s_count[1][wave][r] = small;
  __syncthreads();
  if (wave == 0 && half == 0) {
    float c = 0.0f, h = static_cast<float>(p.k - p.chunks * kSplitK);    // (less the zeros past the rows' end)
#pragma unroll
    for (int w = 0; w < NWV; ++w) {
      c += static_cast<float>(s_count[0][w][r]);
      h += static_cast<float>(s_count[1][w][r]);
    }
    uint32_t word = static_cast<uint32_t>(ex + kSplitBias) << 14;
    if (marked) {
      word |= 0xffu << 24 | 0x3fff;
    } else if (in) {
      const float share = ceilf((h + 4.0f * c) * p.share);
      const uint32_t lost = __float_as_uint(c * p.least);
      word |= (lost + 0x7fffffu) >> 23 << 24 | static_cast<uint32_t>(fminf(share, 0x3fff));
    }
    op.words[blk * kSplitRows + r] = word | (!marked && bound == 0.0f ? kSplitZero : 0u);
  }
}

enum SplitEpilogue { kGemmPlain = 0, kGemmResidual = 1, kGemmSwiglu = 2 };

struct SplitGemmParams {
  const _Float16 *xs, *ws;       // split planes of x (tokens) and W (features)
  const uint32_t *xe, *we;       // row words
  const float *x, *norm_w;       // x itself (row stride ldx) and the RMSNorm's weight or NULL: split_exact_block
  const float *w, *bias;         // W itself (row stride ldw: split_exact_block), bias by W's rows or NULL
  const float *res;              // [rows, n], row stride ldres (kGemmResidual)
  float *y;                      // [rows, n], row stride ldy
  int64_t ldx, ldw, ldres, ldy, rows, n, k, chunks;
  float eps;
  int64_t glu_off;               // kGemmSwiglu: W row of the up half of output column 0
  int64_t xblocks, wblocks;      // 32-row blocks of x and of W
  int64_t tiles_n, tiles_t;      // output tiles over W's blocks and tokens
};

// silu(g) u, as the MLP forms it.
__device__ __forceinline__ float swiglu_value(float g, float u) { return activation(kActSilu, g) * u; }

// The kernel's arguments, read where they are used (and not before).
typedef const __attribute__((address_space(4))) SplitGemmParams *SplitGemmArgs;

// The fp32 products of 32 rows of W from w0 and 32 of x from t0 (rows past the last of
// either read the last again), formed by one wave from the operands as they are on the
// fp32 matrix cores, in the layout of split_gemm_kernel's sums. Lane l loads k = 16 i +
// 8 (l / 32) + 0..7 of its two rows, a step ahead of the eight products that use them; a
// value depends on its two rows alone.
template <bool NORM>
__device__ __forceinline__ f32x16_t split_exact_block(SplitGemmArgs p, int64_t t0, int64_t w0, int64_t w_last) {
  constexpr int64_t kStep = 16;
  const int lane = static_cast<int>(threadIdx.x) % kWave;
  const int r = lane % kSplitRows;
  const int64_t k = p->k, own = lane / kSplitRows * 8;
  const float *x = p->x + (t0 + r < p->rows ? t0 + r : p->rows - 1) * p->ldx;
  const float *w = p->w + (w0 + r < w_last ? w0 + r : w_last) * p->ldw;
  float scale = 1.0f;
  if constexpr (NORM) {
    float ss = 0.0f;
#pragma unroll 1
    for (int64_t k0 = own; k0 < k; k0 += kStep) {
      float v[8];
      split_load(v, x, k0, k);
#pragma unroll
      for (int i = 0; i < 8; ++i) ss = fmaf(v[i], v[i], ss);
    }
    ss += __shfl_xor(ss, 32);
    scale = rsqrtf(ss / static_cast<float>(k) + p->eps);
  }
  f32x16_t acc;
#pragma unroll
  for (int i = 0; i < 16; ++i) acc[i] = 0.0f;
  float xv[8], wv[8];
  split_load(xv, x, own, k);
  split_load(wv, w, own, k);
#pragma unroll 1
  for (int64_t k0 = 0; k0 < k; k0 += kStep) {
    float xn[8], wn[8];
    split_load(xn, x, k0 + kStep + own, k);
    split_load(wn, w, k0 + kStep + own, k);
    if constexpr (NORM) {
      float nw[8];
      split_load(nw, p->norm_w, k0 + own, k);
#pragma unroll
      for (int i = 0; i < 8; ++i) xv[i] = (xv[i] * scale) * nw[i];
    }
#pragma unroll
    for (int i = 0; i < 8; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(wv[i], xv[i], acc, 0, 0, 0);
#pragma unroll
    for (int i = 0; i < 8; ++i) xv[i] = xn[i], wv[i] = wn[i];
  }
  return acc;
}

typedef __attribute__((address_space(3))) void *lds_ptr_t;

// An array's address in LDS.
__device__ __forceinline__ uint32_t lds_address(f16x8_t *p) {
  return static_cast<uint32_t>(reinterpret_cast<uintptr_t>((lds_ptr_t)p));
}

// One fragment from memory to LDS address `dst`, 16 bytes a lane in lane order
// (`src` and `dst` the same in every lane). Written out, because the compiler cannot tell the
// stages of a kernel apart and would wait for every load in flight before each
// read of LDS; the caller holds the waits. No register is loaded, the address
// registers are read as the load issues, and m0 (the LDS address) is put back.
__device__ __forceinline__ void fragment_to_lds(const char *src, uint32_t lane_off, uint32_t dst) {
#ifdef __OPTIMIZE__
  uint32_t m0;
  asm volatile("s_mov_b32 %0, m0\n\ts_mov_b32 m0, %1\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %2, %3\n\ts_mov_b32 m0, %0"
               : "=&s"(m0)
               : "s"(dst), "v"(lane_off), "s"(src)
               : "memory");
#else
  // (An unoptimised build keeps no value in a scalar register.)
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void *)(src + lane_off),
                                   (lds_ptr_t)static_cast<uintptr_t>(dst), 16, 0, 0);
#endif
}

// WAVN x WAVT waves, each FN x FT fragments of 32 features x 32 tokens. W is
// the MFMA's A operand, so a lane ends with four consecutive features of one
// token (D[8 (i / 4) + 4 (lane / 32) + i % 4][lane % 32]) and stores them as one
// 16-byte word. Steps of 16 KH k (KH halves of a chunk) go straight from memory
// into ST stages of LDS, ST - 1 steps ahead of the products.
//
// Bound by the matrix cores and what feeds them: a wave alone keeps them half busy
// (LDS reads and the barrier of a step), so two or three workgroups share a CU,
// and this load draws the clock down (torch's bf16 product of 8192^3 reaches 1.32
// PFLOP/s here; 417 TFLOP/s of fp32 product are 1.25 of fp16). Split + product /
// the library's fp32 product, us:
//   8188 x 4096, k 2048   46 + 329 /  961      4096 x 50304, k 512   36 + 697 / 1539
//   8188 x 1024, k 2048   40 +  94 /  264      4096 x 2048, k 1024   11 +  52 /  124
//   2048 x 2048, k 1024   10 +  31 /   67       256 x 2048, k 512     8 +   8 /   19
// The first through registers instead of straight into LDS: 426; with the
// compiler's waits (every load before each read of LDS) 397; 128 x 128 tiles with
// whole chunks, two stages: 354, with half chunks, three stages: 341.
template <int EPI, int WAVN, int WAVT, int FN, int FT, int KH, int ST, int OCC>
__global__ void __launch_bounds__(WAVN * WAVT * kWave, OCC) split_gemm_kernel(SplitGemmParams p) {
  constexpr int NW = WAVN * WAVT;
  constexpr int BN = WAVN * FN, BT = WAVT * FT;          // 32-row blocks of the tile
  constexpr int TN = BN * kSplitRows, TT = BT * kSplitRows;
  constexpr int FRAGS = (BN + BT) * 2 * KH;               // 1 KiB fragments of a step (KH halves x 2 planes)
  constexpr int LD = FRAGS / NW;
  static_assert(FRAGS % NW == 0, "whole fragments per wave");
  static_assert(ST >= 2 && ST <= 4, "2 to 4 stages");
  // One array per stage: a stage's reads then wait for that stage's loads only.
  __shared__ f16x8_t s_0[FRAGS * 64], s_1[FRAGS * 64], s_2[ST > 2 ? FRAGS * 64 : 1], s_3[ST > 3 ? FRAGS * 64 : 1];
  __shared__ __align__(16) int s_we[TN];
  __shared__ __align__(16) float s_bias[TN];
  __shared__ int s_xe[TT];
  __shared__ int s_doubt[NW];    // by wave, of the rows whose words it read
  // By wave, block of its features, four features of it and token block: the lanes
  // whose outputs split_exact_block forms.
  constexpr int STEP = EPI == kGemmSwiglu ? 2 : 1;
  __shared__ uint64_t s_exact[NW][FN / STEP * 4 * FT];

  const int tid = static_cast<int>(threadIdx.x);
  const int lane = tid % kWave;
  const int wave = __builtin_amdgcn_readfirstlane(tid / kWave);
  const int wn = wave % WAVN, wt = wave / WAVN;

  // Workgroup i runs on XCD i % 8; give each XCD a contiguous run of tiles, and
  // walk those in bands of 8 feature tiles so that the tiles in flight on an XCD
  // share operand rows in its L2.
  int64_t idx = blockIdx.x;
  const int64_t total = p.tiles_n * p.tiles_t;
  if (total % 8 == 0) idx = (idx % 8) * (total / 8) + idx / 8;
  constexpr int64_t BAND = 8;
  const int64_t band = idx / (BAND * p.tiles_t);
  const int64_t width = p.tiles_n - band * BAND < BAND ? p.tiles_n - band * BAND : BAND;
  const int64_t rest = idx - band * BAND * p.tiles_t;
  const int64_t tn = band * BAND + rest % width, tt = rest / width;

  // Fragment wave + j NW of the tile's FRAGS: block / (2 KH), half and plane % (2 KH).
  const char *from[LD];
#pragma unroll
  for (int j = 0; j < LD; ++j) {
    const int e = wave + j * NW;
    const int b = e / (2 * KH);
    const bool isw = b < BN;
    int64_t blk = isw ? tn * BN + b : tt * BT + (b - BN);
    const int64_t last = (isw ? p.wblocks : p.xblocks) - 1;
    blk = blk < last ? blk : last;      // rows past the end: any block, never stored
    from[j] = reinterpret_cast<const char *>((isw ? p.ws : p.xs) + blk * p.chunks * kSplitChunk) + (e % (2 * KH)) * 1024;
  }
  const uint32_t lane_off = static_cast<uint32_t>(lane) * 16;
  auto load = [&](f16x8_t *stage, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < LD; ++j)
      fragment_to_lds(from[j] + static_cast<int64_t>(c) * (kSplitChunk * KH), lane_off,
                      lds_address(stage) + (wave + j * NW) * 1024);
  };

  f32x16_t acc[FN][FT];
#pragma unroll
  for (int a = 0; a < FN; ++a)
#pragma unroll
    for (int b = 0; b < FT; ++b)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[a][b][i] = 0.0f;

  auto products = [&](const f16x8_t *stage) __attribute__((always_inline)) {
    const f16x8_t *sw = stage + wn * FN * (128 * KH) + lane;
    const f16x8_t *sx = stage + (BN + wt * FT) * (128 * KH) + lane;
#pragma unroll
    for (int f = 0; f < KH; ++f) {
      f16x8_t wh[FN], wl[FN], xh[FT], xl[FT];
#pragma unroll
      for (int a = 0; a < FN; ++a) {
        wh[a] = sw[a * (128 * KH) + (2 * f) * 64];
        wl[a] = sw[a * (128 * KH) + (2 * f + 1) * 64];
      }
#pragma unroll
      for (int b = 0; b < FT; ++b) {
        xh[b] = sx[b * (128 * KH) + (2 * f) * 64];
        xl[b] = sx[b * (128 * KH) + (2 * f + 1) * 64];
      }
#pragma unroll
      for (int q = 0; q < 3; ++q)
#pragma unroll
        for (int a = 0; a < FN; ++a)
#pragma unroll
          for (int b = 0; b < FT; ++b)
            acc[a][b] = __builtin_amdgcn_mfma_f32_32x32x16_f16(q == 0 ? wl[a] : wh[a], q == 1 ? xl[b] : xh[b],
                                                               acc[a][b], 0, 0, 0);
    }
  };
  const int chunks = static_cast<int>(p.chunks) * (2 / KH);
  // Step c: wait for its loads (those of the ST - 2 steps after it stay in flight)
  // and for every wave to be done with the step before it, refill that step's
  // stage, multiply. Past the end the last step is loaded again, so that the count
  // in flight is the same for every step.
  auto turn = [&](int c, f16x8_t *stage, f16x8_t *refill) __attribute__((always_inline)) {
    constexpr int kInFlight = LD * (ST - 2);
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(kInFlight) : "memory");
    load(refill, c + ST - 1 < chunks ? c + ST - 1 : chunks - 1);
    products(stage);
  };
  load(s_0, 0);
  if constexpr (ST > 2) load(s_1, chunks > 1 ? 1 : chunks - 1);
  if constexpr (ST > 3) load(s_2, chunks > 2 ? 2 : chunks - 1);
  // The tile's row words and bias, for the epilogue (they arrive with the first chunks).
  const int64_t n0 = tn * TN, t0 = tt * TT;
  // Bit 0: a row of the tile lost something; bit 1: one takes more than its part of h +
  // 4 c <= k (a quarter for W, whose entries are of a size; three quarters for x).
  int doubt = 0;
  for (int i = tid; i < TN + TT; i += NW * kWave) {
    const bool isn = i < TN;
    const int64_t r = isn ? n0 + i : t0 + (i - TN);
    const uint32_t e = r < (isn ? p.wblocks : p.xblocks) * kSplitRows ? (isn ? p.we : p.xe)[r] : kSplitNoRow;
    doubt |= (split_lost(e) != 0.0f) | (split_share(e) > (isn ? kSplitShare / 4 : kSplitShare / 4 * 3)) << 1;
    if (isn) {
      int64_t col = r;
      if constexpr (EPI == kGemmSwiglu) col = (r / 64) * 32 + r % 32;
      s_we[i] = split_exp(e) - 2 * kSplitExp;
      s_bias[i] = p.bias && col < p.n ? p.bias[EPI == kGemmSwiglu && r / 32 % 2 ? p.glu_off + col : col] : 0.0f;
    } else {
      s_xe[i - TN] = split_exp(e);
    }
  }
  doubt = (__any(doubt & 1) ? 1 : 0) | (__any(doubt & 2) ? 2 : 0);
  if (lane == 0) s_doubt[wave] = doubt;
  int c = 0;
  if constexpr (ST == 2) {
    for (; c + 2 <= chunks; c += 2) {
      turn(c, s_0, s_1);
      turn(c + 1, s_1, s_0);
    }
    if (c < chunks) turn(c, s_0, s_1);
  } else if constexpr (ST == 3) {
    for (; c + 3 <= chunks; c += 3) {
      turn(c, s_0, s_2);
      turn(c + 1, s_1, s_0);
      turn(c + 2, s_2, s_1);
    }
    if (c < chunks) turn(c, s_0, s_2);
    if (c + 1 < chunks) turn(c + 1, s_1, s_0);
  } else {
    for (; c + 4 <= chunks; c += 4) {
      turn(c, s_0, s_3);
      turn(c + 1, s_1, s_0);
      turn(c + 2, s_2, s_1);
      turn(c + 3, s_3, s_2);
    }
    if (c < chunks) turn(c, s_0, s_3);
    if (c + 1 < chunks) turn(c + 1, s_1, s_0);
    if (c + 2 < chunks) turn(c + 2, s_2, s_1);
  }
  // No load into this workgroup's LDS may outlive it.
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // (A step's barrier lies between.) Then, for the sums of token t against the four rows
  // of W from wr: whether one has to be formed again, by what their rows lost (nothing
  // against a row of zeros; an infinity against one is, as NaN).
  doubt = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) doubt |= s_doubt[w];
  const bool exact = doubt == 3;
  auto off = [&](const f32x16_t &acc, int g, int64_t t, int64_t wr) __attribute__((always_inline)) {
    const uint32_t xw = p.xe[t];
    const uint4 w4 = *reinterpret_cast<const uint4 *>(p.we + wr);
    const uint32_t ww[4] = {w4.x, w4.y, w4.z, w4.w};
    bool any = false;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const float lost = split_lost(xw) * (ww[j] & kSplitZero ? 0.0f : 1.0f) +
                         split_lost(ww[j]) * (xw & kSplitZero ? 0.0f : 1.0f);
      any = any || (split_share(xw) + split_share(ww[j]) > kSplitShare && !(fabsf(acc[4 * g + j]) >= lost));
    }
    return any;
  };

  const bool vec = p.ldy % 4 == 0 && reinterpret_cast<uintptr_t>(p.y) % 16 == 0;
  const bool vec_res = EPI == kGemmResidual && p.ldres % 4 == 0 && reinterpret_cast<uintptr_t>(p.res) % 16 == 0;
  static_assert(EPI != kGemmSwiglu || FN % 2 == 0, "a wave holds a gate block with its up block");
#pragma unroll
  for (int a = 0; a < FN; a += STEP)
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int nl = (wn * FN + a) * kSplitRows + 8 * g + 4 * (lane / 32);
      const int4 en = *reinterpret_cast<const int4 *>(s_we + nl);
      const float4 bv = *reinterpret_cast<const float4 *>(s_bias + nl);
      const int64_t n = EPI == kGemmSwiglu ? n0 / 2 + (wn * FN + a) / 2 * kSplitRows + 8 * g + 4 * (lane / 32) : n0 + nl;
#pragma unroll
      for (int b = 0; b < FT; ++b) {
        const int tl = (wt * FT + b) * kSplitRows + lane % 32;
        const int64_t t = t0 + tl;
        const int ex = s_xe[tl];
        float4 v = make_float4(ldexpf(acc[a][b][4 * g], ex + en.x) + bv.x,
                               ldexpf(acc[a][b][4 * g + 1], ex + en.y) + bv.y,
                               ldexpf(acc[a][b][4 * g + 2], ex + en.z) + bv.z,
                               ldexpf(acc[a][b][4 * g + 3], ex + en.w) + bv.w);
        if constexpr (EPI == kGemmSwiglu) {
          const int4 eu = *reinterpret_cast<const int4 *>(s_we + nl + kSplitRows);
          const float4 bu = *reinterpret_cast<const float4 *>(s_bias + nl + kSplitRows);
          const f32x16_t &u = acc[a + 1][b];
          v = make_float4(swiglu_value(v.x, ldexpf(u[4 * g], ex + eu.x) + bu.x),
                          swiglu_value(v.y, ldexpf(u[4 * g + 1], ex + eu.y) + bu.y),
                          swiglu_value(v.z, ldexpf(u[4 * g + 2], ex + eu.z) + bu.z),
                          swiglu_value(v.w, ldexpf(u[4 * g + 3], ex + eu.w) + bu.w));
        }
        bool skip = false;
        if (exact) {
          if (t < p.rows && n < p.n) {
            skip = off(acc[a][b], g, t, n0 + nl);
            if constexpr (EPI == kGemmSwiglu) skip = skip || off(acc[a + 1][b], g, t, n0 + nl + kSplitRows);
          }
          const uint64_t lanes = __ballot(skip);
          if (lane == 0) s_exact[wave][(a / STEP * 4 + g) * FT + b] = lanes;
        }
        if (t < p.rows && !skip) {
          float *out = p.y + t * p.ldy + n;
          if constexpr (EPI == kGemmResidual) {
            const float *res = p.res + t * p.ldres + n;
            if (vec_res && n + 4 <= p.n) {
              const float4 x = *reinterpret_cast<const float4 *>(res);
              v = make_float4(x.x + v.x, x.y + v.y, x.z + v.z, x.w + v.w);
            } else {
              if (n < p.n) v.x = res[0] + v.x;
              if (n + 1 < p.n) v.y = res[1] + v.y;
              if (n + 2 < p.n) v.z = res[2] + v.z;
              if (n + 3 < p.n) v.w = res[3] + v.w;
            }
          }
          if (vec && n + 4 <= p.n) {
            *reinterpret_cast<float4 *>(out) = v;
          } else {
            if (n < p.n) out[0] = v.x;
            if (n + 1 < p.n) out[1] = v.y;
            if (n + 2 < p.n) out[2] = v.z;
            if (n + 3 < p.n) out[3] = v.w;
          }
        }
      }
    }
  // What was left out: the outputs to be formed again, 32 x 32 at a time, each read of
  // res and store of y here and nowhere else (y may be res itself).
  if (!exact) return;
  __syncthreads();
  SplitGemmArgs args = (SplitGemmArgs)__builtin_amdgcn_kernarg_segment_ptr();
#ifdef __OPTIMIZE__
  asm volatile("" : "+s"(args));    // (nothing of this is to be ready, or held, any earlier)
#endif
  auto dots = [&](int64_t t, int64_t w, int64_t w_last) __attribute__((always_inline)) {
    return args->norm_w ? split_exact_block<true>(args, t, w, w_last) : split_exact_block<false>(args, t, w, w_last);
  };
#pragma unroll 1
  for (int i = 0; i < FN / STEP * FT; ++i) {
    const int a = i / FT, b = i % FT;
    bool mine[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) mine[g] = s_exact[wave][(a * 4 + g) * FT + b] >> lane & 1;
    if (!__any(mine[0] || mine[1] || mine[2] || mine[3])) continue;
    const int64_t tq = t0 + (wt * FT + b) * kSplitRows, nq = n0 / STEP + (wn * FN / STEP + a) * kSplitRows;
    const int64_t t = tq + lane % 32, n_end = args->n;
    const f32x16_t sum = dots(tq, nq, n_end - 1);
    f32x16_t up;
    if constexpr (EPI == kGemmSwiglu) up = dots(tq, args->glu_off + nq, args->glu_off + n_end - 1);
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int64_t n = nq + 8 * (j / 4) + 4 * (lane / 32) + j % 4;
      if (!mine[j / 4] || n >= n_end) continue;
      float v = sum[j] + (args->bias ? args->bias[n] : 0.0f);
      if constexpr (EPI == kGemmSwiglu) v = swiglu_value(v, up[j] + (args->bias ? args->bias[args->glu_off + n] : 0.0f));
      if constexpr (EPI == kGemmResidual) v = args->res[t * args->ldres + n] + v;
      args->y[t * args->ldy + n] = v;
    }
  }
}

}  // namespace kla
