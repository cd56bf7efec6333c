// Small-product kernels of FP16TCEC, real and complex.
#include "gemm_kwaves_inst.hpp"
namespace cumpsgemm_amd {
#define ROW(A, B) \
  { kwaves_entry<Prec::FP16TCEC, false, A, B, 64, 64, 4, 2>(), kwaves_entry<Prec::FP16TCEC, false, A, B, 32, 32, 8, 4>(), \
    kwaves_entry<Prec::FP16TCEC, false, A, B, 32, 32, 4, 4>(), kwaves_entry<Prec::FP16TCEC, false, A, B, 32, 32, 1, 4>(), \
    kwaves_entry<Prec::FP16TCEC, false, A, B, 64, 64, 4, 1>() }
CUMPSGEMM_KWAVES_TABLE(fp16tcec_s, ROW)
#undef ROW
#define ROW(A, B) \
  { kwaves_entry<Prec::FP16TCEC, true, A, B, 32, 32, 4, 2>(), kwaves_entry<Prec::FP16TCEC, true, A, B, 32, 32, 8, 2>(), KWavesEntry{}, KWavesEntry{}, \
    kwaves_entry<Prec::FP16TCEC, true, A, B, 64, 32, 4, 1>() }
CUMPSGEMM_KWAVES_TABLE(fp16tcec_c, ROW)
#undef ROW
} // namespace cumpsgemm_amd
