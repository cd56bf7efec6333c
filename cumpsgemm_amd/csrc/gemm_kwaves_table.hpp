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

// AUTO: bf16x3 or FP16TCEC with fused scaling, by the launch flag; [layout][form], nullptr: no such form.
typedef void (*kwaves_either_t)(const GemmArgs &, uint32_t accept_bf16, uint32_t accept_fp16, dim3 grid, hipStream_t stream);
extern kwaves_either_t g_kwaves_either_s[4][kKWavesForms];
extern kwaves_either_t g_kwaves_either_c[4][kKWavesForms];
} // namespace cumpsgemm_amd
