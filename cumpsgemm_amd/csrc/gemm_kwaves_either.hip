// Small products under AUTO: both candidates in one kernel (gemm_kwaves.hpp).
#include "gemm_kwaves_inst.hpp"
namespace cumpsgemm_amd {
namespace {
template <class CfgA, class CfgB>
void launch_either(const GemmArgs &args, uint32_t accept_a, uint32_t accept_b, dim3 grid, hipStream_t stream) {
  constexpr int LDS_BYTES = CfgA::LDS_BYTES > CfgB::LDS_BYTES ? CfgA::LDS_BYTES : CfgB::LDS_BYTES;
  static device_flags_t done = {};
  allow_dynamic_lds(reinterpret_cast<const void *>(&kwaves_either_gemm_tcec_kernel<CfgA, CfgB>), LDS_BYTES, done);
  hipLaunchKernelGGL((kwaves_either_gemm_tcec_kernel<CfgA, CfgB>), grid, dim3(CfgA::NT), LDS_BYTES, stream, args, accept_a,
                     accept_b);
}
// (OCC_A, OCC_B: as in the tables of the two precisions)
template <bool CPLX, bool AKC, bool BKC, int BM, int BN, int W, int OCC_A, int OCC_B> constexpr kwaves_either_t either() {
  return &launch_either<KWavesCfg<Prec::BF16X3, CPLX, AKC, BKC, BM, BN, W, OCC_A>,
                        KWavesCfg<Prec::FP16TCEC, CPLX, AKC, BKC, BM, BN, W, OCC_B, true>>;
}
} // namespace
#define ROW(A, B) \
  { either<false, A, B, 64, 64, 4, 1, 2>(), either<false, A, B, 32, 32, 8, 3, 4>(), either<false, A, B, 32, 32, 4, 3, 4>(), \
    either<false, A, B, 32, 32, 1, 3, 4>(), nullptr }
kwaves_either_t g_kwaves_either_s[4][kKWavesForms] = {ROW(false, false), ROW(true, false), ROW(false, true), ROW(true, true)};
#undef ROW
#define ROW(A, B) \
  { either<true, A, B, 32, 32, 4, 1, 2>(), nullptr, nullptr, nullptr, nullptr }
kwaves_either_t g_kwaves_either_c[4][kKWavesForms] = {ROW(false, false), ROW(true, false), ROW(false, true), ROW(true, true)};
#undef ROW
} // namespace cumpsgemm_amd
