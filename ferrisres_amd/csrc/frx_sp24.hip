// frx_sp24.hip — 2:4 ternary GEMV for a decode batch on the sparse matrix pipe.
//
// Semantics of sparse_ternary_matmul_main (src/compute/kernels/
// sparse_ternary.rs:54-112): y[m][n] = scale[n] * sum over the groups of row n
// of its two signed columns of x[m], metadata in the 5-bit GPU layout or in
// the prepared form of frx_sparse24_prepare.
//
// What bounds a small batch. The metadata of 11008 x 4096 is 7.5 MB, under 2
// us of HBM; the tile engine that served 3 tokens and more multiplies 64
// token rows in a pipeline three 64-column steps deep, wants f32 activations
// split into planes by a launch of their own and its K parts added by another
// (8 f32 tokens: 2.4 + 24 + 4 us). Here, as in the dense split-K GEMV
// (frx_gemv_sk.hip), a workgroup owns 128 rows and a slice of the columns: it
// stages the slice's activations once in LDS (f32 split on the way), every
// wave has the slice's metadata of its 16 rows in flight before that, and the
// last slice of a row tile to arrive adds the partial tiles in slice order.
//
// Operands. v_smfmac_f32_16x16x64_bf16 takes 4 groups (16 columns) of row i
// from lane (i = l % 16, kg = l / 16), and from the B lane of token t the
// columns 8 kg .. 8 kg + 7 and 32 + 8 kg .. of its 64. Which 64 columns of the
// matrix those are is free as long as both sides agree, so a lane loads 16
// bytes of its row, 24 groups of the 5-bit layout (96 columns; 16 groups of
// the prepared form) wherever they start, and multiplies them in 6 (4) steps
// of its own 16 columns: no window that straddles the lanes, one funnel shift
// per two steps for the groups that straddle words. Columns past K are staged
// as zeros and cancel whatever the words there hold, so any K % 4 == 0 and any
// N run here (K % 64 != 0 used to take the register-staged engine).
// The 16 columns of B are 16 bf16 tokens, 8 f32 tokens' hi planes and the same
// tokens' lo planes, or up to 4 f32 tokens in three planes each, added across
// lanes at the end; SETS of them share the decoded operand. Three planes hold
// every bit of an f32 value: the few-token calls, which the columns have room
// for, keep full fp32 products as a VALU kernel would (1-4 tokens over 4096 x
// 11008, 8.4-9.2 us with two planes and with three).
#include <type_traits>

#include "frx_device.hpp"
#include "frx_gemm2.hpp"
#include "frx_internal.hpp"

namespace frx {

constexpr int SPR_WAVES = 8;                 // waves per workgroup, 16 rows each
constexpr int SPR_ROWS = SPR_WAVES * 16;     // rows per workgroup
constexpr int SPR_NC = 4;                    // 16-byte loads per lane and slice at most
constexpr int SPR_CG = 16;                   // partial slices loaded before they are added
constexpr uint32_t SPR_OOB = 0x80000000u;    // past every range the plan admits

constexpr int spr_chunk(bool prep) { return prep ? 256 : 384; }  // columns of a wave's 16-byte loads
// bf16 per staged row: nc chunks and 16 bytes that put the 16 rows of an operand
// read on different banks
constexpr int spr_stride(bool prep, int nc) { return nc * spr_chunk(prep) + 8; }

// Step j of a lane's 16 bytes as a sparse A operand.
template <bool PREP>
__device__ __forceinline__ void spr_operand(const u32x4 &w, int j, u32x4 &a, uint32_t &idx) {
  if constexpr (PREP) {
    sp24p_operand(w[j], a, idx);
  } else {
    // groups 4 j .. 4 j + 3 of 24, six to a word
    const int k = j / 3 * 2;
    const uint32_t F = j % 3 == 0 ? w[k] & 0xFFFFFu
                       : j % 3 == 1 ? (__builtin_amdgcn_ubfe(w[k], 20, 10) | (w[k + 1] << 10)) & 0xFFFFFu
                                    : __builtin_amdgcn_ubfe(w[k + 1], 10, 20);
    sp24_operand(F, a, idx);
  }
}

__device__ __forceinline__ f32x4 spr_mul(const f32x4 &acc, const u32x4 &a, const u32x4 &b0, const u32x4 &b1,
                                         uint32_t idx) {
  typedef __bf16 bf16x8v __attribute__((ext_vector_type(8)));
  typedef __bf16 bf16x16v __attribute__((ext_vector_type(16)));
  const u32x8 b = {b0.x, b0.y, b0.z, b0.w, b1.x, b1.y, b1.z, b1.w};
  return __builtin_amdgcn_smfmac_f32_16x16x64_bf16(__builtin_bit_cast(bf16x8v, a), __builtin_bit_cast(bf16x16v, b), acc,
                                                   (int)idx, 0, 0);
}

// grid (ceil(N / 128), S): rows of the tile over chunks s ncs .. of the
// columns; part [S][M][Np]. PL: planes of a token, f32 2 or 3, bf16 1.
// NC: most chunks of a slice (2 or 4; the smaller one keeps more workgroups on a
// compute unit).
template <typename XT, typename YT, int SETS, bool PREP, int NC, int PL>
__global__ __launch_bounds__(SPR_WAVES * 64) void sp24_rows_kernel(const uint32_t *__restrict__ W,
                                                                  const float *__restrict__ scale,
                                                                  const XT *__restrict__ X, float *__restrict__ part,
                                                                  unsigned *__restrict__ counters, YT *__restrict__ Y,
                                                                  int M, int K, int N, int Np, int wpr, int ncs, int S) {
  constexpr bool F32 = sizeof(XT) == 4;
  constexpr int CH = spr_chunk(PREP), NJ = CH / 64, STRIDE = spr_stride(PREP, NC);
  static_assert(F32 ? PL == 2 || PL == 3 : PL == 1, "planes by type");
  constexpr int TPS = PL == 1 ? 16 : PL == 2 ? 8 : 4;  // tokens per set, plane p at columns p TPS ..
  constexpr int PPT = NC * CH / 8, PCS = TPS * PPT, XR = (PCS + SPR_WAVES * 64 - 1) / (SPR_WAVES * 64), XL = F32 ? 2 : 1;
  extern __shared__ __align__(16) uint16_t xs[];  // [16 SETS][STRIDE]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int nch = (K + CH - 1) / CH;
  const int s = blockIdx.y, c0 = s * ncs, nc = min(ncs, nch - c0), k0 = c0 * CH;
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(X, (uint32_t)M * (uint32_t)K * (uint32_t)sizeof(XT));
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(W, (uint32_t)N * (uint32_t)wpr * 4u);
  // 8-column pieces of a set's tokens, zeros past M and K and past the slice
  // (pieces past the set repeat the last one)
  u32x4 xv[SETS][XR][XL];
  auto xload = [&](int set) {
#pragma unroll
    for (int r = 0; r < XR; r++) {
      const int pc = min(tid + r * SPR_WAVES * 64, PCS - 1), t = set * TPS + pc / PPT, o = pc % PPT * 8, col = k0 + o;
      const bool ok = t < M && col < K && o < nc * CH;
      const uint32_t e = ((uint32_t)t * (uint32_t)K + (uint32_t)col) * (uint32_t)sizeof(XT);
#pragma unroll
      for (int l = 0; l < XL; l++)
        xv[set][r][l] = __builtin_amdgcn_raw_buffer_load_b128(xr, ok && (!l || col + 4 < K) ? e + 16u * l : SPR_OOB, 0, 0);
    }
  };
  auto xstore = [&](int set) {
#pragma unroll
    for (int r = 0; r < XR; r++) {
      const int pc = min(tid + r * SPR_WAVES * 64, PCS - 1), row = set * 16 + pc / PPT, o = pc % PPT * 8;
      u32x4 v[PL];
      if constexpr (F32) {
#pragma unroll
        for (int q = 0; q < 4; q++) {
          const float a = __uint_as_float(xv[set][r][q >> 1][2 * (q & 1)]);
          const float b = __uint_as_float(xv[set][r][q >> 1][2 * (q & 1) + 1]);
          uint32_t h, m, l;
          if constexpr (PL == 3) {
            split3_bf16(a, b, h, m, l);
            v[1][q] = m;
          } else {
            split2_bf16(a, b, h, l);
          }
          v[0][q] = h;
          v[PL - 1][q] = l;
        }
      } else {
        v[0] = xv[set][r][0];
        // K % 8 == 4: the second half of the last piece is the next row's
        const uint32_t keep = k0 + o + 4 < K ? 0xFFFFFFFFu : 0u;
        v[0].z &= keep;
        v[0].w &= keep;
      }
#pragma unroll
      for (int p = 0; p < PL; p++) *reinterpret_cast<u32x4 *>(xs + (row + p * TPS) * STRIDE + o) = v[p];
    }
  };
  // activations first (vector loads complete in issue order), then the wave's
  // metadata, every chunk of the slice
#pragma unroll
  for (int set = 0; set < SETS; set++) xload(set);
  __builtin_amdgcn_sched_barrier(0);
  const int i = lane & 15, g = lane >> 4;
  const int row = blockIdx.x * SPR_ROWS + wave * 16 + i;
  u32x4 wv[NC];
#pragma unroll
  for (int c = 0; c < NC; c++)
    wv[c] = __builtin_amdgcn_raw_buffer_load_b128(
        wr,
        c < nc && row < N ? ((uint32_t)row * (uint32_t)wpr + (uint32_t)(c0 + c) * 16u + 4u * g) * 4u : SPR_OOB, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int set = 0; set < SETS; set++) xstore(set);
  __syncthreads();
  f32x4 acc[SETS][2];
#pragma unroll
  for (int t = 0; t < SETS; t++) acc[t][0] = acc[t][1] = (f32x4){0.f, 0.f, 0.f, 0.f};
  // B operand of lane (token i, g): 8 columns of A lane group g / 2 and 8 of
  // group 2 + g / 2 (half g % 2 of their 16)
  const uint16_t *xb = xs + i * STRIDE + (g >> 1) * (CH / 4) + (g & 1) * 8;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (c < nc) {  // workgroup-uniform
#pragma unroll
      for (int j = 0; j < NJ; j++) {
        u32x4 a;
        uint32_t idx;
        spr_operand<PREP>(wv[c], j, a, idx);
#pragma unroll
        for (int t = 0; t < SETS; t++) {
          const uint16_t *p = xb + t * 16 * STRIDE + c * CH + 16 * j;
          acc[t][j & 1] = spr_mul(acc[t][j & 1], a, *reinterpret_cast<const u32x4 *>(p),
                                  *reinterpret_cast<const u32x4 *>(p + CH / 2), idx);
        }
      }
    }
  }
  // partial tile: lane (column j = l % 16, g) holds rows 4 g .. 4 g + 3 of the
  // wave's 16 (unscaled), stored at the point of coherence of all XCDs
  constexpr int SC1 = 16;
  const __amdgpu_buffer_rsrc_t pr = buffer_rsrc(part, (uint32_t)S * (uint32_t)M * (uint32_t)Np * 4u);
#pragma unroll
  for (int t = 0; t < SETS; t++) {
    f32x4 v = acc[t][0] + acc[t][1];
    if constexpr (PL == 2) {
#pragma unroll
      for (int q = 0; q < 4; q++)  // the other plane, 8 columns away (row_ror:8)
        v[q] += __uint_as_float(
            (uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v[q]), 0x128, 0xF, 0xF, true));
    } else if constexpr (PL == 3) {
#pragma unroll
      for (int q = 0; q < 4; q++) {  // mid 4 columns on (row_ror:12), lo 8 (row_ror:8), the small ones first
        const int u = (int)__float_as_uint(v[q]);
        v[q] += __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, u, 0x12C, 0xF, 0xF, true)) +
                __uint_as_float((uint32_t)__builtin_amdgcn_update_dpp(0, u, 0x128, 0xF, 0xF, true));
      }
    }
    const int tok = t * TPS + i, r0 = blockIdx.x * SPR_ROWS + wave * 16 + 4 * g;
    const uint32_t off = i < TPS && tok < M && r0 < Np
                             ? (((uint32_t)s * (uint32_t)M + (uint32_t)tok) * (uint32_t)Np + (uint32_t)r0) * 4u
                             : SPR_OOB;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), pr, off, 0, SC1);
  }
  // the last slice of this row tile adds all of them in slice order (a
  // per-tile counter, reset for the next launch)
  __shared__ int last;
  wait_vmcnt<0>();  // this wave's partial stores are complete
  __syncthreads();
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(counters + blockIdx.x, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    last = old == (unsigned)S - 1u;
    if (last) __hip_atomic_store(counters + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;  // workgroup-uniform
  for (int u = tid; u < M * (SPR_ROWS / 4); u += SPR_WAVES * 64) {
    const int t = u / (SPR_ROWS / 4), n = blockIdx.x * SPR_ROWS + (u % (SPR_ROWS / 4)) * 4;
    if (n >= N) continue;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < S; s0 += SPR_CG) {
      f32x4 v[SPR_CG];
#pragma unroll
      for (int k = 0; k < SPR_CG; k++)
        v[k] = __builtin_bit_cast(
            f32x4,
            __builtin_amdgcn_raw_buffer_load_b128(
                pr,
                s0 + k < S ? (((uint32_t)(s0 + k) * (uint32_t)M + (uint32_t)t) * (uint32_t)Np + (uint32_t)n) * 4u
                           : SPR_OOB,
                0, SC1));
#pragma unroll
      for (int k = 0; k < SPR_CG; k++)
        if (s0 + k < S) sum = (s0 + k == 0) ? v[k] : sum + v[k];
    }
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) o[e] = sum[e] * (0.5f * scale[min(n + e, N - 1)]);  // 0.5 undoes the +-2 values
    YStore<YT>::store4(Y + (size_t)t * N + n, o, min(4, N - n));
  }
}

// Chunks per slice: the fewest that keep the grid within three workgroups per
// compute unit (13824 rows of 5120, 16 f32 / 32 bf16 tokens: 17.2 / 18.2 us
// within two, 14.7 / 15.5 within three; the prepared form decodes faster and
// keeps to two: 11008 rows of 4096, 8 / 32 tokens 8.5 / 14.5 against 9.4 / 17.0) and
// the slices within one batch of the last workgroup's loads (1024 prepared rows
// of 14336, 16 tokens: 15.0 us in 56 slices, 8.0 in 14).
// Against what served these calls before (graph replays, 11008 rows of 4096
// columns): f32 x, 2 / 4 tokens in the table GEMV 10.7 / 19.1 -> 8.8 / 9.0 us, 8 /
// 16 / 24 in the tile engine 28.0 / 29.3 / 30.7 -> 9.8 / 12.9 / 16.1; bf16 8 / 16 /
// 32 tokens 17.2 / 18.8 / 22.1 -> 9.3 / 10.7 / 15.2, prepared 14.4 / 15.7 / 18.6
// -> 7.3 / 8.0 / 12.5. At 48 bf16 tokens (a third column set) the tile engine is
// level or ahead.
bool sp24_rows_plan(int M, int K, int N, int xt_bf16, int prepared, int cus, int *ncs, int *S) {
  if (M < 1 || K % 4 != 0 || M > (xt_bf16 ? SP24_ROWS_MAX_BF16 : SP24_ROWS_MAX_F32)) return false;
  const size_t wpr = prepared ? (size_t)K / 16 : ((size_t)K / 4 + 5) / 6;
  const size_t tiles = ((size_t)N + SPR_ROWS - 1) / SPR_ROWS;
  if (tiles > GEMV_SK_MAX_TILES || (size_t)N * wpr * 4 >= SPR_OOB || (size_t)M * K * 4 >= SPR_OOB) return false;
  const int ch = spr_chunk(prepared), nch = (K + ch - 1) / ch;
  int n = 1;
  while (n < SPR_NC && (tiles * ((nch + n - 1) / n) > (size_t)(prepared ? 2 : 3) * cus || (nch + n - 1) / n > SPR_CG)) n++;
  *ncs = n;
  *S = (nch + n - 1) / n;
  // prepared rows past 24 tokens in many short slices: with tiles that are no
  // multiple of 4 a tile's slices lie on up to eight XCDs, each of which fetches
  // the lines they share, and the tile engine is level or ahead (rows x columns, 32
  // tokens, engine / here: 7296 x 1920 12.1 / 14.2 us, 3904 x 2752 12.2 / 13.3, 11008
  // x 1024 11.5 / 12.2; but 6632 x 4096, 52 tiles, 27 tokens 13.1 / 10.4). Keeping
  // them on one XCD gained 7-14% there and lost as much on others (28 tokens, 3328 x
  // 3392 11.5 -> 12.7, 11008 x 4096 11.0 -> 12.9).
  if (prepared && M > 24 && tiles % 4 != 0 && n <= 2 && 10 * tiles * (size_t)*S > 13 * (size_t)cus) return false;
  return sp24_rows_workspace_bytes(M, N, *S) < SPR_OOB;
}

size_t sp24_rows_workspace_bytes(int M, int N, int S) { return (size_t)S * M * ((size_t)(N + 3) / 4 * 4) * 4; }

template <typename XT, typename YT, int SETS, bool PREP, int NC, int PL>
static hipError_t launch_sp24_rows_nc(const uint32_t *w, const float *scale, const void *x, void *y, int M, int K,
                                      int N, int ncs, int S, float *part, unsigned *counters, hipStream_t stream) {
  const size_t lds = (size_t)16 * SETS * spr_stride(PREP, NC) * 2;
  static std::atomic<uint64_t> done;
  const hipError_t e =
      opt_in_lds(reinterpret_cast<const void *>(&sp24_rows_kernel<XT, YT, SETS, PREP, NC, PL>), (int)lds, done);
  if (e != hipSuccess) return e;
  const int wpr = PREP ? K / 16 : (K / 4 + 5) / 6;
  hipLaunchKernelGGL((sp24_rows_kernel<XT, YT, SETS, PREP, NC, PL>), dim3((N + SPR_ROWS - 1) / SPR_ROWS, S),
                     dim3(SPR_WAVES * 64), lds, stream, w, scale, reinterpret_cast<const XT *>(x), part, counters,
                     reinterpret_cast<YT *>(y), M, K, N, (N + 3) / 4 * 4, wpr, ncs, S);
  return hipGetLastError();
}

template <typename XT, int SETS, bool PREP, int PL = sizeof(XT) == 4 ? 2 : 1>
static hipError_t launch_sp24_rows_t(const uint32_t *w, const float *scale, const void *x, void *y, int yt_bf16, int M,
                                     int K, int N, int ncs, int S, float *part, unsigned *counters,
                                     hipStream_t stream) {
  auto run = [&](auto yp) {
    using YT = std::remove_pointer_t<decltype(yp)>;
    return ncs <= 2 ? launch_sp24_rows_nc<XT, YT, SETS, PREP, 2, PL>(w, scale, x, y, M, K, N, ncs, S, part, counters,
                                                                     stream)
                    : launch_sp24_rows_nc<XT, YT, SETS, PREP, SPR_NC, PL>(w, scale, x, y, M, K, N, ncs, S, part,
                                                                          counters, stream);
  };
  return yt_bf16 ? run((uint16_t *)nullptr) : run((float *)nullptr);
}

hipError_t launch_sp24_rows(const uint32_t *w, int prepared, const float *scale, const void *x, int xt_bf16, void *y,
                            int yt_bf16, int M, int K, int N, int ncs, int S, float *part, unsigned *counters,
                            hipStream_t stream) {
  const int sets = (M + (xt_bf16 ? 15 : 7)) / (xt_bf16 ? 16 : 8);
  auto run = [&](auto f) { return f(w, scale, x, y, yt_bf16, M, K, N, ncs, S, part, counters, stream); };
  if (prepared) return sets == 1 ? run(launch_sp24_rows_t<uint16_t, 1, true>) : run(launch_sp24_rows_t<uint16_t, 2, true>);
  if (xt_bf16) return sets == 1 ? run(launch_sp24_rows_t<uint16_t, 1, false>) : run(launch_sp24_rows_t<uint16_t, 2, false>);
  if (M <= SP24_EXACT_MAX_F32) return run(launch_sp24_rows_t<float, 1, false, 3>);
  return sets == 1   ? run(launch_sp24_rows_t<float, 1, false>)
         : sets == 2 ? run(launch_sp24_rows_t<float, 2, false>)
                     : run(launch_sp24_rows_t<float, 3, false>);
}

}  // namespace frx
