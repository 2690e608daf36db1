// frx_gemv_sk.hip — decode ternary GEMV for 2-16 tokens with K split over
// workgroups (tall row tiles, short column slices) and an ordered combine.
//
// Same semantics as the WGSL entry ternary_matmul_main
// (src/compute/kernels/ternary_matmul.rs:32-75): y[m][n] = scale[n] *
// sum_k dec(W[n][k]) x[m][k].
//
// Why a split. At 16 tokens the activations outweigh the weights a compute
// unit reads: a 16-row tile over the whole of K = 11008 multiplies 44 KB of
// weights against 16 x 11008 activations (352 KB as bf16, 704 KB as f32),
// and every tile of the launch streams all of them through its L1 and LDS.
// Here a workgroup owns 128 rows (eight waves of 16) and a slice of at most
// SK_NC 256-column chunks (gemv_sk_chunks): the activations of the slice are
// staged once in LDS for all 128 rows, which cuts the activation stream per
// weight byte by 8x; the slices of a row tile run on other compute units and
// write fp32 partial tiles part[s][B][Np] with device-coherent stores. The last slice of a row
// tile to finish (a per-tile counter, agent-scope atomic) adds the slices of
// each output in slice order (deterministic whatever the arrival order),
// applies the row scale (and bias) and converts; no second launch and no
// workgroup waits for another.
//
// Operands. Lane (i = l % 16, g = l / 16) of a wave loads 16 bytes (words
// 4g .. 4g + 3, 64 codes) of its row i per chunk; they decode in K-interleaved
// pairs (unpack32_kil), and the activations are staged to match (stage_kil).
// The 16 columns of B are 16 bf16 tokens, or 8 tokens of an fp32 activation as
// hi planes and the same 8 tokens' lo planes (|x - hi - lo| <= 2^-17 |x|;
// split at staging, or given as planes: the FFN's h), whose sums are added
// across lanes at the end, so that up to 8 such tokens cost the MFMAs and
// operand reads of one plane. 9-16 of them take a column set per plane, into
// the same sums. Columns past K and tokens past B are staged as zeros, which
// cancel whatever the weight words hold there.
#include <type_traits>

#include "frx_device.hpp"
#include "frx_gemm2.hpp"
#include "frx_internal.hpp"

namespace frx {

constexpr int SK_WAVES = 8;                  // waves per workgroup, 16 rows each
constexpr int SK_ROWS = SK_WAVES * 16;       // rows per workgroup
constexpr int SK_NC = 4;                     // 256-column chunks per slice at most

constexpr int SK_CPOL_SC1 = 16;  // cache policy: performed at the point of coherence of all XCDs
constexpr int SK_CG = 16;        // partial slices loaded before they are added

// XS: 0 bf16 x; 1 f32 x (split into planes); 2 bf16 planes (X hi, X2 lo).
// SETS: 16-column sets (2: one per plane of up to 16 tokens). NC: most chunks of a slice (the smaller LDS area of 2
// keeps more workgroups on a compute unit).
template <typename YT, int XS, int SETS, int NC>
__global__ __launch_bounds__(SK_WAVES * 64) void gemv_sk_kernel(const uint32_t *__restrict__ W,
                                                                const float *__restrict__ scale,
                                                                const float *__restrict__ bias,
                                                                const void *__restrict__ X,
                                                                const void *__restrict__ X2,
                                                                float *__restrict__ part,
                                                                unsigned *__restrict__ counters,
                                                                YT *__restrict__ Y, int B, int K, int N,
                                                                int Np, int ncs, int S) {
  constexpr int P = XS == 0 ? 1 : 2;
  static_assert(SETS == 1 || (SETS == 2 && P == 2), "a set per plane");
  constexpr int TPS = 16 * SETS / P;           // tokens
  constexpr int STRIDE = NC * 256 + 8;         // bf16 per staged row (16-byte pad)
  constexpr int PPT = NC * 32;                 // 8-column pieces per token
  constexpr int XR = TPS * PPT / (SK_WAVES * 64);
  static_assert(XR * SK_WAVES * 64 == TPS * PPT, "whole rounds of pieces");
  extern __shared__ __align__(16) uint16_t xs[];  // [16 SETS][STRIDE]
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int s = blockIdx.y;
  const int nch = (K + 255) >> 8;
  const int c0 = s * ncs, nc = min(ncs, nch - c0);
  const int k0 = c0 * 256;
  const int kw = K >> 4;
  constexpr uint32_t OOB = 0x80000000u;  // past every range this kernel takes
  // 1. activation pieces of the slice (token t, 8 columns), zero past B or K or
  //    the slice; issued before the weights, since vector loads complete in
  //    issue order
  const __amdgpu_buffer_rsrc_t xr = buffer_rsrc(X, (uint32_t)B * (uint32_t)K * (XS == 1 ? 4u : 2u));
  const __amdgpu_buffer_rsrc_t xr2 = buffer_rsrc(XS == 2 ? X2 : X, (uint32_t)B * (uint32_t)K * 2u);
  u32x4 xv[XR][P];
#pragma unroll
  for (int r = 0; r < XR; r++) {
    const int pc = tid + r * SK_WAVES * 64;
    const int t = pc / PPT, o = pc % PPT * 8, col = k0 + o;
    const bool ok = t < B && col < K && o < nc * 256;
    const uint32_t e = (uint32_t)t * (uint32_t)K + (uint32_t)col;  // element index
    if constexpr (XS == 1) {
#pragma unroll
      for (int l = 0; l < 2; l++) xv[r][l] = __builtin_amdgcn_raw_buffer_load_b128(xr, ok ? e * 4u + 16u * l : OOB, 0, 0);
    } else {
      xv[r][0] = __builtin_amdgcn_raw_buffer_load_b128(xr, ok ? e * 2u : OOB, 0, 0);
      if constexpr (XS == 2) xv[r][1] = __builtin_amdgcn_raw_buffer_load_b128(xr2, ok ? e * 2u : OOB, 0, 0);
    }
  }
  __builtin_amdgcn_sched_barrier(0);
  // 2. the wave's weight words, every chunk of the slice (rows past N and
  //    chunks past the slice read zeros)
  const int i = lane & 15, g = lane >> 4;
  const int row = blockIdx.x * SK_ROWS + wave * 16 + i;
  const __amdgpu_buffer_rsrc_t wr = buffer_rsrc(W, (uint32_t)N * (uint32_t)kw * 4u);
  u32x4 wv[NC];
#pragma unroll
  for (int c = 0; c < NC; c++) {
    const uint32_t off =
        (c < nc && row < N) ? ((uint32_t)row * (uint32_t)kw + (uint32_t)(c0 + c) * 16u + 4u * g) * 4u : OOB;
    wv[c] = __builtin_amdgcn_raw_buffer_load_b128(wr, off, 0, 0);
  }
  __builtin_amdgcn_sched_barrier(0);
  // 3. stage (f32 split into planes)
#pragma unroll
  for (int r = 0; r < XR; r++) {
    const int pc = tid + r * SK_WAVES * 64;
    uint16_t *dst = xs + pc / PPT * STRIDE + pc % PPT * 8;
    u32x4 v[P];
    if constexpr (XS == 1) {
#pragma unroll
      for (int q = 0; q < 4; q++) {
        uint32_t h, l;
        split2_bf16(__uint_as_float(xv[r][q >> 1][2 * (q & 1)]), __uint_as_float(xv[r][q >> 1][2 * (q & 1) + 1]), h, l);
        v[0][q] = h;
        v[P - 1][q] = l;
      }
    } else {
#pragma unroll
      for (int p = 0; p < P; p++) v[p] = xv[r][p];
    }
#pragma unroll
    for (int p = 0; p < P; p++) *reinterpret_cast<u32x4 *>(dst + p * TPS * STRIDE) = stage_kil(v[p], tid);
  }
  __syncthreads();
  // 4. chunks in order as their words land: 8 MFMAs per set each
  f32x4 acc[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
  // B operand of lane (column i, g): the column's staged row at 64 g
  const uint16_t *xb = xs + i * STRIDE + 64 * g;
#pragma unroll
  for (int c = 0; c < NC; c++) {
    if (c < nc) {  // workgroup-uniform
#pragma unroll
      for (int q = 0; q < 4; q += 2) {
        u32x4 a[4];
        unpack32_kil(wv[c][q], wv[c][q + 1], a[0], a[1], a[2], a[3]);
#pragma unroll
        for (int t = 0; t < SETS; t++)
#pragma unroll
          for (int k = 0; k < 4; k++)
            acc[k & 1] = mfma16(
                a[k], *reinterpret_cast<const u32x4 *>(xb + t * 16 * STRIDE + c * 256 + 16 * q + 8 * k), acc[k & 1]);
      }
    }
  }
  // 5. partial tile: lane (column j = l % 16, g) holds rows 4g .. 4g + 3 of
  //    the wave's 16 (unscaled, 2 * the dot product), stored device-coherent
  //    so that the workgroup that adds the slices (on any XCD) reads them from
  //    the point of coherence, not from its own L2
  const __amdgpu_buffer_rsrc_t pr = buffer_rsrc(part, (uint32_t)S * (uint32_t)B * (uint32_t)Np * 4u);
  {
    f32x4 v = acc[0] + acc[1];
    if constexpr (P > SETS) {
#pragma unroll
      for (int q = 0; q < 4; q++)  // the other plane, 8 columns away (row_ror:8)
        v[q] += __uint_as_float(
            (uint32_t)__builtin_amdgcn_update_dpp(0, (int)__float_as_uint(v[q]), 0x128, 0xF, 0xF, true));
    }
    const int r0 = blockIdx.x * SK_ROWS + wave * 16 + 4 * g;
    const uint32_t off = i < TPS && i < B && r0 < Np
                             ? (((uint32_t)s * (uint32_t)B + (uint32_t)i) * (uint32_t)Np + (uint32_t)r0) * 4u
                             : OOB;
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, v), pr, off, 0, SK_CPOL_SC1);
  }
  // 6. the last slice of this row tile to arrive adds all slices in slice
  //    order (a per-tile counter, reset by that workgroup for the next launch)
  __shared__ int last;
  wait_vmcnt<0>();  // this wave's partial stores are complete
  __syncthreads();
  if (tid == 0) {
    const unsigned old = __hip_atomic_fetch_add(counters + blockIdx.x, 1u, __ATOMIC_RELAXED,
                                                __HIP_MEMORY_SCOPE_AGENT);
    last = old == (unsigned)S - 1u;
    if (last) __hip_atomic_store(counters + blockIdx.x, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  }
  __syncthreads();
  if (!last) return;  // workgroup-uniform
  // unit u = (token t, rows 4c .. 4c + 3 of the tile): 32 units per token
  for (int u = tid; u < B * (SK_ROWS / 4); u += SK_WAVES * 64) {
    const int t = u / (SK_ROWS / 4), n = blockIdx.x * SK_ROWS + (u % (SK_ROWS / 4)) * 4;
    if (n >= N) continue;
    f32x4 sum = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < S; s0 += SK_CG) {
      f32x4 v[SK_CG];
#pragma unroll
      for (int k = 0; k < SK_CG; k++) {
        const uint32_t off = s0 + k < S ? (((uint32_t)(s0 + k) * (uint32_t)B + (uint32_t)t) * (uint32_t)Np + (uint32_t)n) * 4u
                                        : OOB;
        v[k] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(pr, off, 0, SK_CPOL_SC1));
      }
#pragma unroll
      for (int k = 0; k < SK_CG; k++)
        if (s0 + k < S) sum = (s0 + k == 0) ? v[k] : sum + v[k];
    }
    const int nok = min(4, N - n);
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; e++) {
      const int nn = min(n + e, N - 1);
      o[e] = sum[e] * (0.5f * scale[nn]);  // 0.5 undoes the 2*dec(c) encoding
      if (bias) o[e] = add_bias(o[e], bias[nn]);
    }
    YStore<YT>::store4(Y + (size_t)t * N + n, o, nok);
  }
}

// Chunks per slice: the fewest that keep the grid within three workgroups per
// compute unit (two where two column sets double the LDS area) and the slices
// within one batch of the last workgroup's loads, at most SK_NC.
static int gemv_sk_chunks(int K, int N, int cus, int sets) {
  const int nch = (K + 255) / 256, tiles = (N + SK_ROWS - 1) / SK_ROWS;
  int n = 1;
  while (n < SK_NC && ((size_t)tiles * ((nch + n - 1) / n) > (size_t)(4 - sets) * cus || (nch + n - 1) / n > SK_CG))
    n++;
  return n;
}

// Enough for any token count and activation source.
size_t gemv_sk_workspace_bytes(int K, int N, int cus) {
  const int ncs = gemv_sk_chunks(K, N, cus, 1);
  const int S = ((K + 255) / 256 + ncs - 1) / ncs;
  const size_t Np = (size_t)(N + 3) / 4 * 4;
  return (size_t)S * 16 * Np * 4;
}

template <typename YT, int XS, int SETS, int NC>
static hipError_t launch_gemv_sk_t(const uint32_t *w, const float *scale, const void *x, const void *x2, void *y, int B,
                                   int K, int N, float *part, unsigned *counters, const float *bias, int ncs,
                                   hipStream_t stream) {
  const size_t lds = (size_t)16 * SETS * (NC * 256 + 8) * 2;
  static std::atomic<uint64_t> done;
  const hipError_t e = opt_in_lds(reinterpret_cast<const void *>(&gemv_sk_kernel<YT, XS, SETS, NC>), (int)lds, done);
  if (e != hipSuccess) return e;
  const int S = ((K + 255) / 256 + ncs - 1) / ncs;
  hipLaunchKernelGGL((gemv_sk_kernel<YT, XS, SETS, NC>), dim3((unsigned)((N + SK_ROWS - 1) / SK_ROWS), (unsigned)S),
                     dim3(SK_WAVES * 64), lds, stream, w, scale, bias, x, x2, part, counters, reinterpret_cast<YT *>(y),
                     B, K, N, (N + 3) / 4 * 4, ncs, S);
  return hipGetLastError();
}

hipError_t launch_gemv_sk(const uint32_t *w, const float *scale, const void *x, const void *x2, int xs,
                          void *y, int yt_bf16, int B, int K, int N, float *part, unsigned *counters,
                          const float *bias, int cus, hipStream_t stream) {
  const int ncs = gemv_sk_chunks(K, N, cus, xs != 0 && B > 8 ? 2 : 1);
  auto run = [&](auto yp, auto xsc, auto sets) {
    using YT = std::remove_pointer_t<decltype(yp)>;
    constexpr int XS = decltype(xsc)::value, SETS = decltype(sets)::value;
    return ncs <= 2 ? launch_gemv_sk_t<YT, XS, SETS, 2>(w, scale, x, x2, y, B, K, N, part, counters, bias, ncs, stream)
                    : launch_gemv_sk_t<YT, XS, SETS, SK_NC>(w, scale, x, x2, y, B, K, N, part, counters, bias, ncs,
                                                            stream);
  };
  using one = std::integral_constant<int, 1>;
  using two = std::integral_constant<int, 2>;
  auto runx = [&](auto yp) {
    if (xs == 0) return run(yp, std::integral_constant<int, 0>(), one());
    if (xs == 1) return B <= 8 ? run(yp, one(), one()) : run(yp, one(), two());
    return B <= 8 ? run(yp, two(), one()) : run(yp, two(), two());
  };
  return yt_bf16 ? runx((uint16_t *)nullptr) : runx((float *)nullptr);
}

}  // namespace frx
