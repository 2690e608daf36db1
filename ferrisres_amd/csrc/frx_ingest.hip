// frx_ingest.hip — weight ingest on the device: the CPU 2:4 layout
// (SparseTernaryMatrix, src/model/sparse_ternary.rs:52-70: pattern nibbles,
// sign pairs with bit 1 = +1, groups numbered flat over the matrix) to the
// GPU 5-bit layout (src/compute/kernels/sparse_ternary.rs:254-318: six groups
// per row word, bits[2:0] pattern, bit 3 / bit 4 set = the lower / higher
// nonzero is -1). One thread per GPU word; bit-exact with the host
// transcoder frx_sparse24_cpu_to_gpu. Patterns 6 and 7, which the CPU layout
// can hold but no packer writes, become pattern 0 as in to_ternary
// (sparse_ternary.rs:172-176).
#include "frx_device.hpp"
#include "frx_internal.hpp"

namespace frx {

__global__ __launch_bounds__(256) void sp24_cpu_to_gpu_kernel(const uint8_t *__restrict__ patterns,
                                                              const uint8_t *__restrict__ signs, uint32_t N,
                                                              uint32_t gpr, uint32_t wpr,
                                                              uint32_t *__restrict__ meta) {
  const size_t wid = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (wid >= (size_t)N * wpr) return;
  const size_t r = wid / wpr;
  const uint32_t w = (uint32_t)(wid - r * wpr);
  uint32_t word = 0;
  for (uint32_t q = 0; q < 6; q++) {
    const uint32_t g = w * 6 + q;
    if (g >= gpr) break;
    const size_t gi = r * gpr + g;
    uint32_t pat = (patterns[gi >> 1] >> (4 * (gi & 1))) & 7u;
    if (pat > 5u) pat = 0u;
    const uint32_t sb = (signs[gi >> 2] >> (2 * (gi & 3))) & 3u;
    word |= (pat | (((~sb) & 3u) << 3)) << (5 * q);
  }
  meta[wid] = word;
}

hipError_t launch_sp24_cpu_to_gpu(const uint8_t *patterns, const uint8_t *signs, int N, int K, uint32_t *meta,
                                  hipStream_t stream) {
  const uint32_t gpr = (uint32_t)K / 4, wpr = (gpr + 5) / 6;
  const size_t words = (size_t)N * wpr;
  if (words == 0) return hipSuccess;
  const size_t blocks = (words + 255) / 256;
  hipLaunchKernelGGL(sp24_cpu_to_gpu_kernel, dim3((unsigned)blocks), dim3(256), 0, stream, patterns, signs,
                     (uint32_t)N, gpr, wpr, meta);
  return hipGetLastError();
}

// ---- on-device quantisation: f32 or bf16 weights -> packed codes + scales --
//
// quantize_ternary (src/model/ternary.rs:31-57: alpha = mean|w| /
// ABSMEAN_NORM, 1 for an all-zero input; q = clamp(round(w * (1 / alpha)),
// -1, 1), round half away from zero; used by BitLinear::requantize,
// src/training/shadow_weights.rs:152-160) and the on-the-fly rule of
// BitLinear::forward_ste (shadow_weights.rs:203-231: alpha = mean|w|; q = +1
// where w / alpha > 0.5, -1 where < -0.5, else 0; all 0 when alpha < 1e-10),
// each applied to every row of W [N][K] on its own; a single row of n values
// is the reference's call on a whole tensor. bf16 weights (bf16 shadows) are
// widened exactly, as P::to_f32 does.
// Scale. The reference sums |w| left to right in f32, and that order fixes
// the rounding, so one lane adds its row in exactly that order from LDS while
// the rest of its wave stages the next 1024 values with coalesced loads; one
// workgroup (one wave) per row. Codes: one thread per u32 word, -1 / 0 / +1
// -> codes 0 / 1 / 2, sixteen per word LSB first (pack_ternary with
// pack_ternary_u32's word order, ternary.rs:134-163,1317-1328).
constexpr float QUANT_ABSMEAN_NORM = 0.7978845608f;  // sqrt(2 / pi), ternary.rs:15
constexpr uint32_t QUANT_CHUNK = 1024;               // values per staged chunk

__device__ __forceinline__ float quant_widen(const float *p, size_t i) { return p[i]; }
__device__ __forceinline__ float quant_widen(const uint16_t *p, size_t i) {
  return __uint_as_float((uint32_t)p[i] << 16);
}

// Scale of one block: block b covers values [b * block, min(n, (b + 1) *
// block)) of the flat array (a row of W [N][K] is a block of K; the whole
// tensor is one block of n; quantize_ternary_blocked's blocks are ragged at
// the end). One workgroup (one wave) per block.
template <typename WT>
__global__ __launch_bounds__(64) void quant_scale_kernel(const WT *__restrict__ W, size_t n, size_t block,
                                                        int rule, float *__restrict__ scale) {
  __shared__ __align__(16) float buf[2][QUANT_CHUNK];
  const int lane = threadIdx.x;
  const size_t start = (size_t)blockIdx.x * block;
  const size_t len = min(block, n - start);
  const WT *row = W + start;
  const size_t nch = (len + QUANT_CHUNK - 1) / QUANT_CHUNK;
  float v[QUANT_CHUNK / 64];
  auto load = [&](size_t c) {
#pragma unroll
    for (uint32_t j = 0; j < QUANT_CHUNK / 64; j++) {
      const size_t i = c * QUANT_CHUNK + j * 64 + (uint32_t)lane;
      v[j] = i < len ? quant_widen(row, i) : 0.0f;
    }
  };
  auto store = [&](size_t c) {
#pragma unroll
    for (uint32_t j = 0; j < QUANT_CHUNK / 64; j++) buf[c & 1][j * 64 + lane] = v[j];
  };
  load(0);
  store(0);
  __syncthreads();
  float sum = 0.0f;
  for (size_t c = 0; c < nch; c++) {
    if (c + 1 < nch) load(c + 1);  // in flight during the additions
    if (lane == 0) {
      const uint32_t m = (uint32_t)min((size_t)QUANT_CHUNK, len - c * QUANT_CHUNK);
      const float *b = buf[c & 1];
      for (uint32_t i = 0; i < m; i++) sum = sum + fabsf(b[i]);  // adds only: nothing to contract
    }
    if (c + 1 < nch) store(c + 1);  // the other buffer (read during the previous chunk)
    __syncthreads();
  }
  if (lane == 0) {
    const float mean = sum / (float)len;  // len as f32, as `block.len() as f32`
    // quantize_ternary: sum_abs > 0 (false for NaN) selects the absmean
    scale[blockIdx.x] = rule == 0 ? (sum > 0.0f ? mean / QUANT_ABSMEAN_NORM : 1.0f) : mean;
  }
}

// Codes of 16 consecutive values of the flat array per thread (one u32 word
// of pack_ternary_u32); value i uses the scale of block i / block. Values past
// n are the zero padding bits of pack_ternary (code 0b00).
template <typename WT>
__global__ __launch_bounds__(256) void quant_pack_kernel(const WT *__restrict__ W, size_t n, size_t block, int rule,
                                                        const float *__restrict__ scale,
                                                        uint32_t *__restrict__ packed) {
  const size_t wid = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (wid * 16 >= n) return;
  size_t b_cur = ~(size_t)0;
  float alpha = 1.0f, inv = 1.0f;
  uint32_t word = 0;
#pragma unroll
  for (int j = 0; j < 16; j++) {
    const size_t i = wid * 16 + j;
    if (i >= n) break;
    const size_t b = i / block;
    if (b != b_cur) {
      b_cur = b;
      alpha = scale[b];
      inv = 1.0f / alpha;
    }
    const float w = quant_widen(W, i);
    int q;
    if (rule == 0) {
      // (w * inv).round() as i32, clamped: NaN -> 0, +-inf saturate
      const float r = roundf(w * inv);
      q = r >= 1.0f ? 1 : r <= -1.0f ? -1 : 0;
    } else {
      const float t = w / alpha;  // NaN compares false -> 0
      q = alpha < 1e-10f ? 0 : t > 0.5f ? 1 : t < -0.5f ? -1 : 0;
    }
    word |= (uint32_t)(q + 1) << (2 * j);
  }
  packed[wid] = word;
}

// ---- the same for blocks that 16-byte loads can walk ---------------------------
// (W 16-byte aligned, block and n multiples of the 4 f32 / 8 bf16 values of a
// load.) Every shape of a weight matrix takes these; the kernels above serve
// the unaligned and short-block rest.
//
// Scale. The left-to-right sum is one dependent f32 add per value, about
// 2.6 ns each, but a wave runs 64 of them for the price of one. With a wave
// per row, as above, 11008 rows are 10.75 chains per SIMD that take turns at
// its issue slots and use one lane of 64 each. Here a wave owns R rows, lane r
// adds row r, and the chains of a wave share every instruction. The wave
// loads 16 KB ahead (16 loads, whole lines, in flight during the additions of
// the chunk before) and hands it over through LDS, each row's part shifted by
// 16 bytes so that the R lanes read different banks. Values past a row's end
// are staged as +0, which no sum notices.
// R: as many rows as leave 512 waves (two per CU) to keep HBM busy.
// 11008 x 4096 f32: 104.7 -> 33.7 us (5.4 TB/s). Both kernels, few and short
// rows, us before / now: 64 x 512 bf16 12.7 / 11.3, 512 x 1024 bf16 19.3 / 12.0,
// 512 x 1024 f32 16.5 / 9.0, 1 x 4096 bf16 42 / 28.
template <typename WT, int R>
__global__ __launch_bounds__(64) void quant_scale_rows_kernel(const WT *__restrict__ W, size_t n, size_t block,
                                                             unsigned nb, int rule, float *__restrict__ scale) {
  constexpr int VPL = 16 / (int)sizeof(WT);  // values per 16-byte load
  constexpr int C = 16 / R;                  // loads per row and chunk
  constexpr int CH = C * 64 * VPL;           // values per row and chunk
  constexpr int LS = C * 256 + 4;            // dwords per staged row
  constexpr int G = 8;                       // LDS reads in flight
  __shared__ __align__(16) uint32_t buf[R * LS];
  const int lane = threadIdx.x;
  const unsigned row0 = blockIdx.x * R;
  u32x4 v[16];
  auto len_of = [&](unsigned r) { return min(block, n - (size_t)r * block); };
  auto load = [&](size_t c) {
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const unsigned r = min(row0 + k / C, nb - 1);
      const size_t i = c * CH + (size_t)((k % C) * 64 + lane) * VPL;
      // past the end: the last load of the block, replaced by zeros at staging
      v[k] = *reinterpret_cast<const u32x4 *>(W + (size_t)r * block + min(i, len_of(r) - VPL));
    }
  };
  const size_t nch = (block + CH - 1) / CH;
  load(0);
  float sum = 0.0f;
  const uint32_t *mine = buf + (lane & (R - 1)) * LS;
  for (size_t c = 0; c < nch; c++) {
#pragma unroll
    for (int k = 0; k < 16; k++) {
      const unsigned r = min(row0 + k / C, nb - 1);
      const size_t i = c * CH + (size_t)((k % C) * 64 + lane) * VPL;
      const bool ok = i < len_of(r);
      u32x4 t = v[k];
#pragma unroll
      for (int e = 0; e < 4; e++) t[e] = ok ? t[e] : 0u;
      *reinterpret_cast<u32x4 *>(buf + (k / C) * LS + ((k % C) * 64 + lane) * 4) = t;
    }
    __syncthreads();
    if (c + 1 < nch) load(c + 1);
    // two sets of G reads: one is added while the other is on its way
    u32x4 a[2][G];
    auto read = [&](u32x4(&d)[G], int g) {
#pragma unroll
      for (int j = 0; j < G; j++) d[j] = *reinterpret_cast<const u32x4 *>(mine + (g * G + j) * 4);
    };
    auto add = [&](const u32x4(&d)[G]) {
#pragma unroll
      for (int j = 0; j < G; j++)
#pragma unroll
        for (int e = 0; e < 4; e++) {
          if constexpr (sizeof(WT) == 4) {
            sum = sum + fabsf(__uint_as_float(d[j][e]));  // adds only: nothing to contract
          } else {
            sum = sum + fabsf(__uint_as_float(d[j][e] << 16));
            sum = sum + fabsf(__uint_as_float(d[j][e] & 0xFFFF0000u));
          }
        }
    };
    auto sums = [&](int ng) __attribute__((always_inline)) {
      read(a[0], 0);
      for (int g = 0; g < ng; g += 2) {
        read(a[1], g + 1);
        __builtin_amdgcn_sched_barrier(0);
        add(a[0]);
        if (g + 2 < ng) read(a[0], g + 2);
        __builtin_amdgcn_sched_barrier(0);
        add(a[1]);
      }
    };
    // a last chunk ends with the rows (in pairs of sets): the zeros staged past
    // them cost as much as values. Whole chunks keep the constant count: over a
    // variable one 2048 x 4096 f32 went from 24.0 to 28.0 us.
    constexpr int NG = C * 64 / G;  // even
    const size_t rest = block - c * CH;
    if (rest >= CH) sums(NG);
    else sums(2 * (int)((rest + 2 * G * VPL - 1) / (2 * G * VPL)));
    __syncthreads();
  }
  const unsigned r = row0 + lane;
  if (lane < R && r < nb) {
    const float mean = sum / (float)len_of(r);
    scale[r] = rule == 0 ? (sum > 0.0f ? mean / QUANT_ABSMEAN_NORM : 1.0f) : mean;
  }
}

// Codes: a wave takes 4 x 64 loads of one block (whole lines; a thread per
// word, as above, put 64 bytes between the lanes of each load), every lane
// makes the bits of its own values, and the lanes of a word join theirs with
// DPP. Bound by the read of W: 11008 x 4096 f32 102.4 -> 28.2 us (the second
// read of W hits the Infinity Cache in part).
// The rules without a division per value, to the same codes:
//  - roundf(p) >= 1 exactly when p >= 0.5 (halves round away from zero);
//  - fl(w / alpha) > 0.5 exactly when w > alpha / 2: the quotient exceeds 0.5
//    after rounding when it exceeds the midpoint 0.5 (1 + 2^-24) (the midpoint
//    itself rounds to the even 0.5), alpha / 2 is exact from 1e-10 up, and the
//    next float above alpha / 2 lies above it by more than 2^-24 of itself.
//    Infinite and NaN alpha or w compare false on both sides.
template <typename WT>
__global__ __launch_bounds__(256) void quant_pack_rows_kernel(const WT *__restrict__ W, size_t n, size_t block,
                                                             unsigned units, unsigned per_block, int rule,
                                                             const float *__restrict__ scale,
                                                             uint32_t *__restrict__ packed) {
  constexpr int VPL = 16 / (int)sizeof(WT);
  constexpr int LPW = 16 / VPL;   // lanes per word
  constexpr int WPL = 64 / LPW;   // words per load of the wave
  const int lane = threadIdx.x & 63;
  const unsigned unit = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (unit >= units) return;
  const unsigned b = unit / per_block;
  const size_t i0 = (size_t)(unit - b * per_block) * (4 * 64 * VPL);
  const size_t start = (size_t)b * block, len = min(block, n - start);
  u32x4 v[4];
#pragma unroll
  for (int j = 0; j < 4; j++)
    v[j] = *reinterpret_cast<const u32x4 *>(W + start + min(i0 + (size_t)(j * 64 + lane) * VPL, len - VPL));
  const float alpha = scale[b];
  const float inv = 1.0f / alpha;
  const float thr = alpha < 1e-10f ? __builtin_inff() : 0.5f * alpha;
  uint32_t word[4];
#pragma unroll
  for (int j = 0; j < 4; j++) {
    uint32_t bits = 0;
#pragma unroll
    for (int e = 0; e < VPL; e++) {
      const float w = VPL == 4   ? __uint_as_float(v[j][e & 3])
                      : (e & 1) ? __uint_as_float(v[j][e >> 1] & 0xFFFF0000u)
                                : __uint_as_float(v[j][e >> 1] << 16);
      const float p = w * inv;
      const bool up = rule == 0 ? p >= 0.5f : w > thr;
      const bool dn = rule == 0 ? p <= -0.5f : w < -thr;
      bits |= (up ? 2u : dn ? 0u : 1u) << (2 * e);
    }
    bits <<= 2 * VPL * (lane & (LPW - 1));
    bits |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits, 0xB1, 0xF, 0xF, true);  // lane ^ 1
    if (LPW == 4) bits |= (uint32_t)__builtin_amdgcn_update_dpp(0, (int)bits, 0x4E, 0xF, 0xF, true);  // lane ^ 2
    word[j] = bits;
  }
  // lane k of a word's lanes stores the words of loads k, k + LPW, ...
#pragma unroll
  for (int h = 0; h < 4 / LPW; h++) {
    const int k = lane & (LPW - 1);
    uint32_t out = word[h * LPW];
#pragma unroll
    for (int q = 1; q < LPW; q++) out = k == q ? word[h * LPW + q] : out;
    const size_t wi = i0 / 16 + (size_t)(h * LPW + k) * WPL + lane / LPW;
    if (wi * 16 < len) packed[start / 16 + wi] = out;
  }
}

template <typename WT>
static hipError_t launch_quantize_t(const WT *w, size_t n, size_t block, int rule, uint32_t *packed, float *scale,
                                    hipStream_t stream) {
  constexpr size_t VPL = 16 / sizeof(WT);
  const size_t nb = (n + block - 1) / block;
  const bool al = (reinterpret_cast<uintptr_t>(w) & 15) == 0;
  // a block shorter than a wave's load is better off a lane per value
  if (al && block % VPL == 0 && n % VPL == 0 && block >= 64 * VPL && nb < ((size_t)1 << 31)) {
    const unsigned rows = (unsigned)nb;
#define FRX_QS(R)                                                                                             \
  hipLaunchKernelGGL((quant_scale_rows_kernel<WT, R>), dim3((rows + R - 1) / R), dim3(64), 0, stream, w, n, block, \
                     rows, rule, scale)
    if (rows >= 16 * 512) FRX_QS(16);
    else if (rows >= 8 * 512) FRX_QS(8);
    else if (rows >= 4 * 512) FRX_QS(4);
    else if (rows >= 2 * 512) FRX_QS(2);
    else FRX_QS(1);
#undef FRX_QS
  } else {
    hipLaunchKernelGGL(quant_scale_kernel<WT>, dim3((unsigned)nb), dim3(64), 0, stream, w, n, block, rule, scale);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess || !packed) return e;
  const size_t per = (block + 4 * 64 * VPL - 1) / (4 * 64 * VPL);
  // whole words per block, and blocks that fill most of a wave's loads
  if (al && block % 16 == 0 && n % 16 == 0 && block >= 2 * 64 * VPL && nb * per < ((size_t)1 << 31)) {
    hipLaunchKernelGGL(quant_pack_rows_kernel<WT>, dim3((unsigned)((nb * per + 3) / 4)), dim3(256), 0, stream, w, n,
                       block, (unsigned)(nb * per), (unsigned)per, rule, scale, packed);
  } else {
    const size_t words = (n + 15) / 16;
    hipLaunchKernelGGL(quant_pack_kernel<WT>, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream, w, n, block,
                       rule, scale, packed);
  }
  return hipGetLastError();
}

hipError_t launch_quantize_flat(const void *w, int wt_bf16, size_t n, size_t block, int rule, uint32_t *packed,
                                float *scale, hipStream_t stream) {
  if (n == 0) return hipSuccess;
  if (wt_bf16) return launch_quantize_t(reinterpret_cast<const uint16_t *>(w), n, block, rule, packed, scale, stream);
  return launch_quantize_t(reinterpret_cast<const float *>(w), n, block, rule, packed, scale, stream);
}

hipError_t launch_quantize(const void *w, int wt_bf16, int N, int K, int rule, uint32_t *packed, float *scale,
                           hipStream_t stream) {
  return launch_quantize_flat(w, wt_bf16, (size_t)N * (size_t)K, (size_t)K, rule, packed, scale, stream);
}

// ---- dequantize_ternary_blocked (ternary.rs:113-128) ------------------------
// out[i] = scales[i / block] * dec(code i) over the flat packed codes
// (alpha * {-1, 0, +1}, one IEEE product: exact). Codes 0b01 and 0b11 are 0
// (TERNARY_DECODE, ternary.rs:136-140).
__global__ __launch_bounds__(256) void dequant_kernel(const uint32_t *__restrict__ packed,
                                                     const float *__restrict__ scales, size_t n, size_t block,
                                                     float *__restrict__ out) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  const uint32_t c = (packed[i >> 4] >> (2 * (i & 15))) & 3u;
  const float d = c == 0 ? -1.0f : c == 2 ? 1.0f : 0.0f;
  out[i] = scales[i / block] * d;
}

hipError_t launch_dequantize(const uint32_t *packed, const float *scales, size_t n, size_t block, float *out,
                             hipStream_t stream) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(dequant_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, stream, packed, scales, n,
                     block, out);
  return hipGetLastError();
}

// ---- prune_fp32_to_sparse_ternary (sparse_ternary.rs:598-663) -----------------
// One group of four values: the two largest |v| by the reference's stable
// sort_by (an insertion sort on four elements: a value moves left only past
// a strictly smaller |v|, so ties keep the lower position and a NaN moves
// past nothing). pat = pattern of the ordered positions; s0 / s1 = 1 when the
// LARGEST / second largest value is >= 0: the reference packs the sign bits
// in magnitude order (:642-644) while decoding reads bit 0 as the lower
// position's sign, and this keeps that.
__device__ __forceinline__ void prune_group(const float v[4], uint32_t &pat, uint32_t &s0, uint32_t &s1) {
  int idx[4] = {0, 1, 2, 3};
#pragma unroll
  for (int i = 1; i < 4; i++) {
#pragma unroll
    for (int j = i; j > 0; j--) {
      // adjacent swap while the later element is strictly larger in |v|
      if (fabsf(v[idx[j]]) > fabsf(v[idx[j - 1]])) {
        const int t = idx[j];
        idx[j] = idx[j - 1];
        idx[j - 1] = t;
      } else {
        break;
      }
    }
  }
  const int a = idx[0], b = idx[1];
  const int p0 = min(a, b), p1 = max(a, b);
  // SPARSE_PATTERN (sparse_ternary.rs:27-34): (0,1)(0,2)(0,3)(1,2)(1,3)(2,3)
  pat = p0 == 0 ? (uint32_t)(p1 - 1) : p0 == 1 ? (uint32_t)(p1 + 1) : 5u;
  s0 = v[a] >= 0.0f ? 1u : 0u;
  s1 = v[b] >= 0.0f ? 1u : 0u;
}

template <typename WT>
__device__ __forceinline__ void load_group(const WT *w, size_t g, float v[4]) {
#pragma unroll
  for (int j = 0; j < 4; j++) v[j] = quant_widen(w, 4 * g + j);
}

// CPU layout: thread t owns flat groups 4t .. 4t+3, i.e. pattern bytes 2t
// and 2t+1 and sign byte t, so no byte is shared between threads.
template <typename WT>
__global__ __launch_bounds__(256) void prune_cpu_kernel(const WT *__restrict__ w, size_t ng,
                                                       uint8_t *__restrict__ patterns,
                                                       uint8_t *__restrict__ signs) {
  const size_t t = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (4 * t >= ng) return;
  uint32_t pb[2] = {0, 0}, sb = 0;
#pragma unroll
  for (int q = 0; q < 4; q++) {
    const size_t g = 4 * t + q;
    if (g >= ng) break;
    float v[4];
    load_group(w, g, v);
    uint32_t pat, s0, s1;
    prune_group(v, pat, s0, s1);
    pb[q >> 1] |= pat << (4 * (q & 1));
    sb |= (s0 | (s1 << 1)) << (2 * q);
  }
  patterns[2 * t] = (uint8_t)pb[0];
  if (2 * t + 1 < (ng + 1) / 2) patterns[2 * t + 1] = (uint8_t)pb[1];
  signs[t] = (uint8_t)sb;
}

// GPU layout: one thread per row word (six groups, bit 3 / bit 4 set when
// the lower / higher position decodes to -1), the same bits the transcoder
// writes from the CPU layout.
template <typename WT>
__global__ __launch_bounds__(256) void prune_gpu_kernel(const WT *__restrict__ w, uint32_t N, uint32_t gpr,
                                                       uint32_t wpr, uint32_t *__restrict__ meta) {
  const size_t wid = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (wid >= (size_t)N * wpr) return;
  const size_t r = wid / wpr;
  const uint32_t j = (uint32_t)(wid - r * wpr);
  uint32_t word = 0;
  for (uint32_t q = 0; q < 6; q++) {
    const uint32_t g = j * 6 + q;
    if (g >= gpr) break;
    float v[4];
    load_group(w, r * gpr + g, v);
    uint32_t pat, s0, s1;
    prune_group(v, pat, s0, s1);
    word |= (pat | ((s0 ^ 1u) << 3) | ((s1 ^ 1u) << 4)) << (5 * q);
  }
  meta[wid] = word;
}

__global__ void broadcast_first_kernel(float *__restrict__ v, uint32_t n) {
  const uint32_t i = blockIdx.x * 256 + threadIdx.x + 1;
  if (i < n) v[i] = v[0];
}

template <typename WT>
static hipError_t launch_prune_t(const WT *w, int N, int K, int per_row, uint8_t *patterns, uint8_t *signs,
                                 uint32_t *meta, float *scale, hipStream_t stream) {
  const size_t n = (size_t)N * (size_t)K;
  if (n == 0) return hipSuccess;
  const size_t ng = n / 4;
  if (patterns) {
    const size_t threads = (ng + 3) / 4;
    hipLaunchKernelGGL(prune_cpu_kernel<WT>, dim3((unsigned)((threads + 255) / 256)), dim3(256), 0, stream, w, ng,
                       patterns, signs);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  if (meta) {
    const uint32_t gpr = (uint32_t)K / 4, wpr = (gpr + 5) / 6;
    const size_t words = (size_t)N * wpr;
    hipLaunchKernelGGL(prune_gpu_kernel<WT>, dim3((unsigned)((words + 255) / 256)), dim3(256), 0, stream, w,
                       (uint32_t)N, gpr, wpr, meta);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
  // the reference's per-tensor absmean (rule 0 of the quantiser), or one
  // per row; the tensor scale is then copied to every row
  hipError_t e = launch_quantize_flat(w, sizeof(WT) == 2, n, per_row ? (size_t)K : n, 0, nullptr, scale, stream);
  if (e != hipSuccess || per_row || N <= 1) return e;
  hipLaunchKernelGGL(broadcast_first_kernel, dim3((unsigned)((N - 1 + 255) / 256)), dim3(256), 0, stream, scale,
                     (uint32_t)N);
  return hipGetLastError();
}

hipError_t launch_prune_sparse24(const void *w, int wt_bf16, int N, int K, int per_row, uint8_t *patterns,
                                 uint8_t *signs, uint32_t *meta, float *scale, hipStream_t stream) {
  if (wt_bf16)
    return launch_prune_t(reinterpret_cast<const uint16_t *>(w), N, K, per_row, patterns, signs, meta, scale,
                          stream);
  return launch_prune_t(reinterpret_cast<const float *>(w), N, K, per_row, patterns, signs, meta, scale, stream);
}

}  // namespace frx
