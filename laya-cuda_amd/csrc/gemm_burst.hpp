// The few-row GEMM (gemm_burst.hip): its tile menu and launcher.
#pragma once

#include <type_traits>

#include "kernels.hpp"

namespace laya {

// LAYA_BURST(variant, BM, BN, WM, WN, KG, 64-deep slabs per stage, stages): WM x WN x KG waves.
// The 32x32 tile's 64 KB of LDS let two workgroups share a CU; the others have a CU each.
#define LAYA_BURST_TILES               \
  LAYA_BURST(0, 32, 32, 1, 2, 4, 2, 4) \
  LAYA_BURST(1, 48, 32, 1, 2, 4, 4, 3) \
  LAYA_BURST(2, 64, 32, 2, 1, 4, 4, 3) \
  LAYA_BURST(3, 32, 64, 1, 2, 4, 4, 3) \
  LAYA_BURST(4, 64, 64, 2, 2, 2, 2, 4) \
  LAYA_BURST(5, 64, 64, 2, 2, 4, 2, 4) \
  LAYA_BURST(6, 64, 96, 2, 2, 2, 2, 3) \
  LAYA_BURST(7, 128, 64, 4, 2, 1, 1, 4)

hipError_t burst_prepare();  // dynamic LDS limits, once per device
// `a` as launch_gemm checks it; N a multiple of the variant's BN.
hipError_t launch_burst(const GemmArgs& a, Epi epi, DType t, int variant, hipStream_t stream);

}  // namespace laya
