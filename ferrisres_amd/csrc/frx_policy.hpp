// frx_policy.hpp — host-side rules: the sizes of the context workspaces and
// the kernels of the decode FFN, kept free of HIP so that a CPU build can check
// them.
#pragma once
#include <stddef.h>

namespace frx {

// Size to allocate when a workspace of `have` bytes must hold `need`:
// at least 1.5x the old size (rounded to 256 bytes), so that a run of rising
// requests makes O(log(max / first)) allocations and the buffers it retires
// sum to less than twice the final size.
inline size_t grow_bytes(size_t have, size_t need) {
  const size_t a = (need + 255) & ~(size_t)255;
  if (need <= have) return have;
  const size_t g = have + have / 2;
  const size_t b = (g + 255) & ~(size_t)255;
  return b > a ? b : a;
}

// ---- the FFN of 1-16 tokens: gate and up over K columns and N rows each, then
// the down projection (times are of the whole FFN, hidden / intermediate) -------

// bf16 tokens from which gate and up leave the kernel with operand loads for the
// staged one (gemv_xs_kernel), 8 where it is not ahead from 5 or 6. Writing h as
// planes (the FFN): over 2048 to 4096 columns past 4096 rows (4096 / 14336, 5 / 7
// tokens 25.9 / 27.4 us with operand loads, 24.4 / 23.7 staged; 2560 / 8192 15.9 / 16.7
// and 15.4 / 15.6; over fewer rows the FFN is level). Writing fp32 h
// (frx_ternary_glu): past 8192 rows, and below where the columns fill its waves'
// quads (2816 / 12288 8.1 / 8.5 and 7.6 / 7.6, 4096 / 5632 7.6 / 7.9 and 7.1 / 7.1; but
// 3328 / 5632 6.4 / 6.6 and 7.0 / 6.9, 2432 / 5632 5.8 / 6.0 and 6.9 / 6.9). Below 2048
// columns a workgroup's few quads leave its waves idle (FFN 1024 / 2048, 5 tokens
// 8.8 against 9.3). Above 4096 its x outweighs its rows (FFN 5120 / 4096, 5 / 7 tokens
// 16.1 / 14.0 against 17.1 / 14.6, 5120 / 13824 28.3 / 30.5 against 29.8 / 30.2) but
// where the FFN gives each unit two tiles of them (5120 / 5632, 5 / 6 / 7 tokens 17.9 /
// 18.5 / 18.9 against 18.0 / 17.9 / 17.9, 5120 / 8192 20.0 / 20.7 / 21.2 against 20.2 /
// 20.6 / 20.5). fp32 h leaves the operand loads there only where rows that are no
// multiple of 16 bytes narrow them (5 / 7 tokens: 4432 / 5632 11.3 / 12.3 against 9.6 /
// 9.5, 5136 / 8192 12.6 / 14.6 against 10.0 / 10.1; 4416 / 5632 7.8 / 8.7 against 9.5 /
// 9.5, 5120 / 5632 8.8 / 9.8 against 9.7 / 9.7).
constexpr int glu_staged_min_tokens(int K, int N, bool planes) {
  if (K < 2048) return 8;
  if (K > 4096 && (N <= 4096 || N > 8192)) return 8;
  if (K > 4096) return planes ? 6 : K % 64 != 0 ? 5 : 8;
  if (planes) return N > 4096 ? 5 : 8;
  return N > 8192 || (K > 3840 && N > 4096) ? 5 : 8;
}

// Whether one f32 token takes the staged kernel: not over more than 4096
// columns (5120 / 13824 31.8 us with the 16-row tiles, 35.9 staged) nor, where
// short rows make a workgroup's start its time, over more than 4096 rows (1024 /
// 5632 8.7 and 9.7, 1024 / 13824 12.1 and 13.7; but 1024 / 4096 7.7 and 7.6, 3072 /
// 11008 18.0 and 16.6).
constexpr bool glu_staged_one_f32(int K, int N) { return K <= 4096 && (K > 2048 || N <= 4096); }

// Most 16-row tiles of both matrices in a workgroup of the staged kernel (its
// weight registers allow 4 up to 4096 columns, 2 up to 8192, 1 above). bf16 x:
// not so many that the fullest compute unit gets more of them, and where three
// do not hold a unit's rows, two workgroups of two on it (their loads overlap)
// before one of four. 5 / 16 tokens: 5120 / 11008, one tile 24.9 / 28.3 us, two
// (344 workgroups, four tiles on the units that have two) 29.4 / 31.3; 5120 / 5632
// 18.4 / 20.5 against 18.0 / 20.3; 4096 / 13824, two 21.7 / 24.8, four 22.1 / 25.6;
// 4096 / 11008, two 20.8 / 23.9, three 19.3 / 22.2. f32 x has one workgroup per
// unit anyway (LDS) and keeps the most tiles (2048 / 13824, 5 tokens 17.5 us with
// four, 20.2 with two).
constexpr int glu_staged_tiles(int K, int N, bool bf16, int cus) {
  if (K > 8192) return 1;
  if (K > 4096) {
    const int one = ((N + 15) / 16 + cus - 1) / cus, two = 2 * (((N + 31) / 32 + cus - 1) / cus);
    return bf16 && two > one ? 1 : 2;
  }
  return bf16 && N > 48 * cus ? 2 : 4;
}

// Intermediate from which the down projection of `tokens` is split over K. Up to
// 8 tokens, whose planes share the 16 columns (whole rows / split: 4096 / 5632, 5 / 8
// tokens 18.3 / 15.9 and 14.9 / 15.1 us; 2048 / 5632 16.5 / 14.0 and 13.1 / 13.3),
// and above over H output rows whose 16-row tiles are few or past one round of
// the compute units (12 / 16 tokens: 1024 / 5632 14.1 / 14.5 and 12.8 / 13.6, 5120 /
// 5632 20.4 / 20.8 and 19.4 / 20.3; but 3072 / 5632 16.2 / 16.6 and 17.3 / 18.4, 4096 /
// 5632 16.3 / 16.9 and 16.3 / 17.0, 2048 / 5632 14.5 / 14.8 and 14.4 / 15.0).
constexpr int ffn_down_split_min(int tokens, int H, int cus) {
  return tokens <= 8 || H < 2048 || H > 16 * cus ? 4097 : 8192;
}

// ---- the staged kernel over one matrix, 2-16 tokens ----------------------------

// Most 16-row tiles of a workgroup, by its weight registers (planes: 2 for f32 x).
constexpr int linear_staged_tiles(int K, int planes) {
  return planes == 1 ? (K <= 8192 ? 4 : 2) : K <= 4096 ? 4 : K <= 8192 ? 2 : 1;
}

// Rounds of workgroups, one to a compute unit, over `tiles` 16-row tiles: a
// workgroup per unit while it holds them, else as many as hold them.
constexpr int staged_rounds(int tiles, int tmax, int cus) {
  return tiles <= tmax * cus ? 1 : ((tiles + tmax - 1) / tmax + cus - 1) / cus;
}

// Whether one launch over the tiles of a group's matrices takes fewer rounds
// than a launch for each: above 8192 columns a workgroup holds two tiles, and
// two launches of one round are ahead of one of two (5 / 16 bf16 tokens, us, apart /
// one launch: 5504 and 2752 rows of 9216 15.4 / 15.9 and 16.9 / 17.3, 8192 and
// 4096 rows of 11008 17.6 / 18.5 and 18.9 / 19.3; but 3 x 5440 of 11008 30.3 / 31.5
// and 21.0 / 21.4, 2 x 4096 of 11008 15.0 / 15.4 and 10.2 / 10.6).
constexpr bool group_fewer_rounds(int count, const int *n, int K, int planes, int cus) {
  const int tmax = linear_staged_tiles(K, planes);
  int tiles = 0, apart = 0;
  for (int i = 0; i < count; i++) {
    tiles += (n[i] + 15) / 16;
    apart += staged_rounds((n[i] + 15) / 16, tmax, cus);
  }
  return staged_rounds(tiles, tmax, cus) < apart;
}

}  // namespace frx
