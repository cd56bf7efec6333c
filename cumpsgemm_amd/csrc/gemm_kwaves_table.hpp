// Instances of the small-product kernel (gemm_kwaves.hpp): per precision and real /
// complex, [layout][form]; layout as in gemm_table.hpp.
#pragma once
#include "gemm_table.hpp"
#include "kwaves_rule.hpp"

namespace cumpsgemm_amd {

struct KWavesEntry {
  void (*launch)(const GemmArgs &, dim3 grid, hipStream_t stream); // nullptr: no such form
  void (*launch_scaled)(const GemmArgs &, dim3 grid, hipStream_t stream); // (FP16TCEC only, else nullptr)
};

#define CUMPSGEMM_DECLARE_KWAVES(name) extern KWavesEntry g_kwaves_##name[4][kKWavesForms];
CUMPSGEMM_DECLARE_KWAVES(fp16tcec_s)
CUMPSGEMM_DECLARE_KWAVES(fp16tcec_c)
CUMPSGEMM_DECLARE_KWAVES(fp16tc_s)
CUMPSGEMM_DECLARE_KWAVES(fp16tc_c)
CUMPSGEMM_DECLARE_KWAVES(bf16x3_s)
CUMPSGEMM_DECLARE_KWAVES(bf16x3_c)
CUMPSGEMM_DECLARE_KWAVES(bf16x2_s)
CUMPSGEMM_DECLARE_KWAVES(bf16x2_c)
#undef CUMPSGEMM_DECLARE_KWAVES
} // namespace cumpsgemm_amd
