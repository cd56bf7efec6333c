// Which real products with a narrow side narrow.hip takes, and how it shares
// them out over the chip.  Host arithmetic on sizes and layouts alone.
#pragma once
#include <algorithm>
#include <cstdint>

namespace cumpsgemm_amd {

constexpr uint32_t kNarrowMax = 32;  // largest narrow side
constexpr uint32_t kNarrowRows = 32; // rows of the large operand per workgroup

constexpr uint32_t kNarrowMinWide = 1024; // smallest wide side

struct NarrowPlan {
  uint32_t waves;           // per workgroup: 8 or 16
  uint32_t chunks;          // parts of K, added into C with atomics; 0: not a product for this kernel
  uint32_t steps_per_chunk; // whole 32-wide K-steps of a part
};

// Whether the product is served faster here than by the tiled kernels.  Every line lies where a sweep of both put it:
// 1024 - 2^20 rows x {1, 8, 16, 17, 24, 32} x K = 1 - 16384, four layouts, operands from memory and from the caches;
// the figures are narrow / tiled times, the worst over the narrow sides, from memory and from the caches.
// `groups`: workgroups, one per kNarrowRows rows and part of K.
inline bool narrow_is_faster(bool bf16x3, bool big_kc, bool small_kc, uint32_t wide, uint32_t groups, uint32_t few,
                             uint32_t k, uint32_t cus) {
  const uint32_t tiles = (wide + kNarrowRows - 1) / kNarrowRows;
  const bool two = few > 16; // two blocks of narrow rows: more registers, more products per byte
  const bool both_kc = big_kc && small_kc, whole = k % 32 == 0;
  // More workgroups than the CUs hold at once (two of 8 waves, three with one narrow block).  Every workgroup adds up
  // its waves' sums, idle ones included, so a short K loses most: 2^20 rows, K = 4, FP16TCEC 1.7 - 2.1, two blocks 3.8.
  // (Means of the two times over 4500 shapes of 16384 - 2^20 rows.)
  if (tiles > (two ? 2 : 3) * cus) {
    // Rows in thousands of cache lines: the tiled kernels' tiles fit exactly, this one's loads fall on few channels
    // (2^20 x 32 x 128 bf16x3 NN 1.4, 2^18 x 16 x 256 FP16TCEC NN 1.3, 32768 x 32 x 512 1.2 - 1.4).
    if (wide % 4096 == 0 && ((tiles > 6 * cus && (two || !bf16x3)) || (two && !bf16x3))) return false;
    // (K < 32: one block 0.86, up to 4 * cus tiles 1.06, two blocks 1.1 - 1.5; K >= 32: 0.42 - 0.94)
    if (bf16x3) return k >= 32 || (!two && tiles > 4 * cus);
    // (up to 4 * cus, K = 128 - 1024: 0.84 - 0.97, up to 6 * cus, K < 384: 0.87 - 0.98; K < 128 1.0 - 2.4; else 1.1 - 1.35)
    if (two)
      return k >= 128 && (tiles <= 4 * cus ? k <= 1024 && !(both_kc && whole && k > 256) : tiles <= 6 * cus && k < 384);
    // (K = 32 - 383: 0.70 - 0.85; up to 6 * cus, K = 384 - 1535: 0.84 - 0.92, longer, K-contiguous: 0.82 - 1.0;
    // K < 32 1.0 - 1.3, a long K on more workgroups 1.0 - 1.1)
    return k >= 32 && (tiles <= 6 * cus ? k < 1536 || big_kc : k < 384);
  }
  if (!bf16x3) {
    if (two) {
      // K = 1024: up to 4096 rows 1.0 - 1.8, 5000 - 8192 rows 0.68 - 0.9; beyond that TN 1.1 - 1.3 (K = 512 1.0 - 1.4),
      // others 0.8 - 1.04.  Long K: 5000 x 20 x 5000 27 -> 30 us, 16384 x 32 x 8192 NN 95 -> 128.
      if (k > 1024 || (k >= 896 && tiles <= cus / 2)) return false;
      return !(both_kc && whole && k > 256 && tiles > cus);
    }
    if (k < 1024) return true; // (0.47 - 1.0; 12000 x 30 x 777 17 -> 14 us, 1024 x 32 x 256 9.3 -> 6.0)
    // Few workgroups with a long K, which the tiled kernels split over more of them: TN 1024 rows, K = 1024 1.37 - 1.53,
    // 2048 1.9 - 2.1; 4096 rows 1.0 - 1.3.  Row-contiguous: K = 1024 0.73 - 0.98, longer only with a workgroup per CU
    // (2048 x 8192 0.88, 4096 x 4096 0.86, where 1024 x 4096 takes 1.4).
    if (tiles <= cus / 2)
      return (k < 1536 && (!big_kc || (!small_kc && !whole))) || (!big_kc && groups >= cus);
    // About one workgroup per CU: K up to 2560 0.65 - 0.97, longer ones where it is nearly exactly one
    // (8192 rows 0.83 - 1.07, 6500 rows 1.0 - 1.28) or the narrow operand is row-contiguous (0.83 - 1.0).
    if (tiles <= cus)
      return k <= 2560 || (whole && tiles >= cus * 15 / 16) || (!small_kc && (big_kc || k <= 4096));
    // Two or three: K = 1024, 1300 0.85 - 1.04, longer 1.0 - 1.5 except K-contiguous from nearly two on
    // (16384 rows, K = 4096 0.8 - 1.1, 8192 0.8).
    return k < 1536 || (big_kc && whole && k >= 4096 && tiles >= cus * 15 / 8);
  }
  // bf16x3, whose tiled kernels are bound by the split: everything but a long K on few workgroups.  K = 1024 on 32 of
  // them 1.2 - 1.5 TN, on 94 0.9 - 1.0; K = 2048 on 32 1.7 - 2.0, on 94 0.95 - 1.3, on 128 0.9 - 1.0 (two blocks
  // 1.1 - 1.2); 2048 x 4096 on 2 x 64 1.04 - 1.14; row-contiguous with one block K = 1024 0.9 - 0.96 on any number.
  if (k < 1024) return true;
  if (two) return groups >= (k < 2048 ? cus / 3 : cus / 2 + 1);
  if (!big_kc) return k < 2048 || groups >= cus / 3;
  return groups >= (k < 2048 ? cus / 3 : tiles >= cus / 2 ? cus / 2 : cus / 2 + 1);
}

// wide x k times k x few (or its mirror image), FP16TCEC or bf16x3; big_kc / small_kc: operand stored K-contiguous
inline NarrowPlan plan_narrow(bool bf16x3, bool big_kc, bool small_kc, uint32_t wide, uint32_t few, uint32_t k,
                              uint32_t num_cus) {
  const NarrowPlan none{0, 0, 0};
  if (few > kNarrowMax || wide < kNarrowMinWide) return none;
  // Waves on a CU are what keeps loads in flight: 16 a workgroup while there is at most one per CU, 8 beyond (16 fill a
  // CU, and 257 - 511 workgroups of them run as two rounds, the second mostly empty: 10000 x 16 TN, us,
  // 16 -> 8 waves: K = 256 6.5 -> 5.8, K = 777 16.8 -> 14.3); K is split over workgroups where there are fewer of them than CUs, as long as every wave has a few steps.
  const uint32_t tiles = (wide + kNarrowRows - 1) / kNarrowRows, steps = k / 32;
  NarrowPlan p{tiles > num_cus ? 8u : 16u, 1, 0};
  // (a launch holds fewer than 2^32 threads along one axis; the tiled kernels need an eighth of these)
  if ((uint64_t)tiles * p.waves * 64 >= (1ull << 32)) return none;
  while (tiles * p.chunks * 2 <= num_cus * 3 / 2 && steps / (p.chunks * 2) >= 4 * p.waves) p.chunks *= 2;
  // (FP16TCEC, chunks that leave the second round of workgroups mostly empty: 3000 x 3 x 12345 TN 29.3 -> 32.4)
  if (!bf16x3 && p.chunks > 1 && tiles * p.chunks > num_cus) return none;
  if (!narrow_is_faster(bf16x3, big_kc, small_kc, wide, tiles * p.chunks, few, k, num_cus)) return none;
  p.steps_per_chunk = (steps + p.chunks - 1) / p.chunks;
  if (p.steps_per_chunk != 0) p.chunks = std::max(1u, (steps + p.steps_per_chunk - 1) / p.steps_per_chunk);
  return p;
}
} // namespace cumpsgemm_amd
