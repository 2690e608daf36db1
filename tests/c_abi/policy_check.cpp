// Host check of the workspace growth rule (frx::grow_bytes): rising
// requests make O(log) allocations and the retired buffers stay below twice
// the final size; and of the decode FFN's kernel rules. Built with g++ by
// tests/test_c_abi.py; no GPU.
#include <stdio.h>

#include "frx_policy.hpp"

static int check(size_t first, size_t last, size_t step) {
  size_t have = 0, retired = 0;
  unsigned allocs = 0;
  for (size_t need = first; need <= last; need += step) {
    const size_t b = frx::grow_bytes(have, need);
    if (b < need || b % 256 != 0) {
      printf("grow_bytes(%zu, %zu) = %zu\n", have, need, b);
      return 1;
    }
    if (b != have) {
      retired += have;
      have = b;
      allocs++;
    }
  }
  // 1.5x growth: at most log_1.5(last / first) + 2 allocations
  unsigned bound = 2;
  for (double r = (double)last / (double)first; r > 1.0; r /= 1.5) bound++;
  if (allocs > bound || retired >= 2 * have) {
    printf("first %zu last %zu step %zu: %u allocations (bound %u), retired %zu of %zu\n", first, last, step, allocs,
           bound, retired, have);
    return 1;
  }
  return 0;
}

// 16-row tiles on the fullest of `cus` units when workgroups hold up to t of
// them (a workgroup per unit while the rows fit, as gemv_xs_grid).
static int fullest(int N, int t, int cus) {
  const int tiles = (N + 15) / 16;
  int G = tiles < cus ? tiles : cus;
  if ((N + G - 1) / G > 16 * t) G = (N + 16 * t - 1) / (16 * t);
  const int rows = (N + G - 1) / G, per = (rows + 15) / 16;
  return (G + cus - 1) / cus * per;
}

static int check_ffn_rules() {
  const int units[] = {64, 228, 256, 304};
  for (int cus : units)
    for (int N = 16; N <= 40000; N += 16)
      for (int K = 64; K <= 12288; K += 64)
        for (int bf16 = 0; bf16 < 2; bf16++) {
          const int t = frx::glu_staged_tiles(K, N, bf16, cus), most = K <= 4096 ? 4 : K <= 8192 ? 2 : 1;
          bool ok = t >= 1 && t <= most && (bf16 || t == most);
          // bf16: no fewer tiles would leave the fullest unit with fewer of them
          if (bf16 && K > 4096) ok = ok && fullest(N, t, cus) <= fullest(N, 1, cus) + (t == 2 && N <= 32 * cus);
          if (bf16 && K <= 4096 && N <= 64 * cus) ok = ok && fullest(N, t, cus) <= fullest(N, 2, cus);
          if (!ok) {
            printf("glu_staged_tiles(%d, %d, %d, %d) = %d\n", K, N, bf16, cus, t);
            return 1;
          }
        }
  // the measured sides of each line (hidden, intermediate)
  const bool ok = frx::glu_staged_tiles(5120, 11008, true, 256) == 1 && frx::glu_staged_tiles(5120, 13824, true, 256) == 2 &&
                  frx::glu_staged_tiles(5120, 11008, false, 256) == 2 && frx::glu_staged_tiles(4096, 11008, true, 256) == 4 &&
                  frx::glu_staged_tiles(4096, 13824, true, 256) == 2 && frx::glu_staged_tiles(2048, 13824, false, 256) == 4 &&
                  frx::glu_staged_min_tokens(5120, 4096, true) == 8 && frx::glu_staged_min_tokens(4096, 11008, true) == 5 &&
                  frx::glu_staged_min_tokens(4096, 4096, true) == 8 && frx::glu_staged_min_tokens(1024, 2048, true) == 8 &&
                  frx::glu_staged_min_tokens(2560, 8192, true) == 5 && frx::glu_staged_min_tokens(5120, 5632, true) == 6 &&
                  frx::glu_staged_min_tokens(2816, 12288, false) == 5 && frx::glu_staged_min_tokens(2816, 5632, false) == 8 &&
                  frx::glu_staged_min_tokens(4096, 5632, false) == 5 && frx::glu_staged_min_tokens(4432, 7328, false) == 5 &&
                  frx::glu_staged_min_tokens(5120, 5632, false) == 8 && frx::glu_staged_min_tokens(4416, 8192, false) == 8 &&
                  !frx::glu_staged_one_f32(1024, 13824) && frx::glu_staged_one_f32(1024, 4096) &&
                  frx::glu_staged_one_f32(3072, 11008) && !frx::glu_staged_one_f32(5120, 13824) &&
                  frx::ffn_down_split_min(8, 3072, 256) <= 5632 &&
                  frx::ffn_down_split_min(9, 3072, 256) > 5632 && frx::ffn_down_split_min(16, 3072, 256) <= 8192 &&
                  frx::ffn_down_split_min(12, 1024, 256) <= 5632 && frx::ffn_down_split_min(12, 5120, 256) <= 5632;
  if (!ok) printf("measured lines of the FFN rules\n");
  return !ok;
}

// Groups of one round are always fewer than apart; more rounds, only if so.
static int check_group_rule() {
  const int qkv[] = {4096, 4096, 4096}, two[] = {5504, 2752}, wide[] = {8192, 4096}, three[] = {5440, 5440, 5440};
  const int even[] = {4096, 4096}, one[] = {512};
  const bool ok = frx::group_fewer_rounds(3, qkv, 4096, 1, 256) && frx::group_fewer_rounds(3, qkv, 4096, 2, 256) &&
                  !frx::group_fewer_rounds(2, two, 9216, 1, 256) && frx::group_fewer_rounds(2, two, 8192, 1, 256) &&
                  !frx::group_fewer_rounds(2, wide, 11008, 1, 256) && frx::group_fewer_rounds(3, three, 11008, 1, 256) &&
                  frx::group_fewer_rounds(2, even, 11008, 1, 256) && !frx::group_fewer_rounds(2, even, 8256, 2, 256) &&
                  !frx::group_fewer_rounds(1, one, 4096, 1, 256);
  if (!ok) printf("measured lines of the group rule\n");
  return !ok;
}

int main() {
  int bad = check_ffn_rules() | check_group_rule();
  // prefill M = 17..2048 at I = 11008 (fp32 h rows), and byte-sized steps
  bad |= check(17 * 11008 * 4, 2048 * 11008 * 4, 11008 * 4);
  bad |= check(1, 1 << 20, 1);
  bad |= check(256, 256 << 20, 4096);
  if (frx::grow_bytes(1000, 10) != 1000 || frx::grow_bytes(0, 1) != 256 || frx::grow_bytes(1024, 1025) != 1536) {
    printf("closed cases\n");
    bad = 1;
  }
  if (!bad) printf("policy_check ok\n");
  return bad;
}
