// Building blocks of the gemm_kwaves_*.hip tables.
#pragma once
#include "gemm_kwaves.hpp"
#include "gemm_kwaves_table.hpp"

namespace cumpsgemm_amd {

template <class Cfg> void launch_kwaves(const GemmArgs &args, dim3 grid, hipStream_t stream) {
  static device_flags_t done = {};
  allow_dynamic_lds(reinterpret_cast<const void *>(&kwaves_gemm_tcec_kernel<Cfg>), Cfg::LDS_BYTES, done);
  hipLaunchKernelGGL(kwaves_gemm_tcec_kernel<Cfg>, grid, dim3(Cfg::NT), Cfg::LDS_BYTES, stream, args);
}

// (tile and waves as in kwaves_rule.hpp; OCC: waves per SIMD that the registers allow)
template <Prec P, bool CPLX, bool AKC, bool BKC, int BM, int BN, int W, int OCC> constexpr KWavesEntry kwaves_entry() {
  KWavesEntry e{};
  e.launch = &launch_kwaves<KWavesCfg<P, CPLX, AKC, BKC, BM, BN, W, OCC>>;
  if constexpr (P == Prec::FP16TCEC) e.launch_scaled = &launch_kwaves<KWavesCfg<P, CPLX, AKC, BKC, BM, BN, W, OCC, true>>;
  return e;
}
#define CUMPSGEMM_KWAVES_TABLE(name, ROW) \
  KWavesEntry g_kwaves_##name[4][kKWavesForms] = {ROW(false, false), ROW(true, false), ROW(false, true), ROW(true, true)};
} // namespace cumpsgemm_amd
