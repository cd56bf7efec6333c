// Which real products with a narrow side narrow.hip takes, and how it shares
// them out over the chip.  Host arithmetic on sizes alone.
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

// wide x k times k x few (or its mirror image), FP16TCEC or bf16x3
inline NarrowPlan plan_narrow(bool bf16x3, uint32_t wide, uint32_t few, uint32_t k, uint32_t num_cus) {
  const NarrowPlan none{0, 0, 0};
  // Measured, tiled -> this kernel, us.  bf16x3, whose tiled kernels are bound by the split: every shape tried,
  // 8192 x 16 x 8192 65 - 83 -> 44 - 51, 16384 x 32 x 8192 144 - 180 -> 119 - 131, 1024 x 32 x 256 9.3 -> 5.7.
  // FP16TCEC: 16 rows or columns at any K, 16384 x 1 x 1000 16.5 -> 12.5, 1024 x 16 x 16384 18.9 -> 17.0,
  // 2048 x 8 x 8192 17 - 24 -> 15.5 - 17; more of them while K is short, 12000 x 30 x 777 17 -> 14,
  // 1024 x 32 x 256 9.3 -> 6.0 (long K loses: 5000 x 20 x 5000 27 -> 30, 16384 x 32 x 8192 NN 95 -> 128).
  if (few > kNarrowMax || wide < kNarrowMinWide) return none;
  if (!bf16x3 && few > 16 && k > 1024) return none;
  // Waves on a CU are what keeps loads in flight: 8 a workgroup where there are
  // two workgroups per CU, 16 below, and K split over workgroups where there
  // are fewer of them than CUs, as long as every wave has a few steps.
  const uint32_t tiles = (wide + kNarrowRows - 1) / kNarrowRows, steps = k / 32;
  NarrowPlan p{tiles >= 2 * num_cus ? 8u : 16u, 1, 0};
  // (a launch holds fewer than 2^32 threads along one axis; the tiled kernels need an eighth of these)
  if ((uint64_t)tiles * p.waves * 64 >= (1ull << 32)) return none;
  while (tiles * p.chunks * 2 <= num_cus * 3 / 2 && steps / (p.chunks * 2) >= 4 * p.waves) p.chunks *= 2;
  // (FP16TCEC, chunks that leave the second round of workgroups mostly empty: 3000 x 3 x 12345 TN 29.3 -> 32.4)
  if (!bf16x3 && p.chunks > 1 && tiles * p.chunks > num_cus) return none;
  p.steps_per_chunk = (steps + p.chunks - 1) / p.chunks;
  if (p.steps_per_chunk != 0) p.chunks = std::max(1u, (steps + p.steps_per_chunk - 1) / p.steps_per_chunk);
  return p;
}
} // namespace cumpsgemm_amd
