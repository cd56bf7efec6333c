// Small-product kernels of BF16X3, real and complex.
#include "gemm_kwaves_inst.hpp"
namespace cumpsgemm_amd {
#define ROW(A, B) \
  { kwaves_entry<Prec::BF16X3, false, A, B, 64, 64, 4, 1>(), kwaves_entry<Prec::BF16X3, false, A, B, 32, 32, 8, 3>(), \
    kwaves_entry<Prec::BF16X3, false, A, B, 32, 32, 4, 3>(), kwaves_entry<Prec::BF16X3, false, A, B, 32, 32, 1, 3>() }
CUMPSGEMM_KWAVES_TABLE(bf16x3_s, ROW)
#undef ROW
#define ROW(A, B) \
  { kwaves_entry<Prec::BF16X3, true, A, B, 32, 32, 4, 1>(), KWavesEntry{}, KWavesEntry{}, KWavesEntry{} }
CUMPSGEMM_KWAVES_TABLE(bf16x3_c, ROW)
#undef ROW
} // namespace cumpsgemm_amd
