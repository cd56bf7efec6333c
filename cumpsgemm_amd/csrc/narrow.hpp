// Real products with one narrow side (C has at most kNarrowMax rows or columns):
// one pass over the large operand, see narrow.hip.
#pragma once
#include "gemm_table.hpp"
#include "narrow_rule.hpp"

namespace cumpsgemm_amd {

// what used_kernel_module_id reports for it: the number behind the table's classes (+ 100: K split, as there)
constexpr int kNarrowModuleId = kNumTileClasses;

struct NarrowArgs {
  const float *big, *small; // op(big): wide x k, op(small): few x k
  float *c;
  uint64_t ld_big, ld_small, ldc;
  uint32_t wide, few, k;
  uint32_t steps_per_chunk; // whole 32-wide K-steps per blockIdx.z
  uint32_t few_is_n;        // C is wide x few (else few x wide)
  uint32_t atomic_out;      // K is split over blockIdx.z: C += alpha * x
  float alpha, beta;
};

// whether every 32-bit offset the kernel forms fits
bool narrow_offsets_fit(uint64_t ld_big, uint64_t ld_small);
// p: FP16TCEC or BF16X3; big_kc / small_kc: stored K-contiguous; `waves`: 8 or 16 per workgroup
void launch_narrow(const NarrowArgs &args, Prec p, bool big_kc, bool small_kc, uint32_t waves, uint32_t chunks,
                   hipStream_t stream);
} // namespace cumpsgemm_amd
