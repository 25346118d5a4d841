// Launch of the even forms of the persistent grouped GEMM (persistent_even.hip).
#pragma once

#include "persistent_body.h"

// (results stored non-temporal without the SwiGLU, cached with it, whatever their size: the 256 x 256 tiles store results beyond
// 192 MB non-temporal, here it is the same within 0.3 %: 8 experts, 4096 / 14336, layer of 3600 / 4250 / 5000 tokens cached 1984 / 2423 /
// 2571 us, non-temporal 1981 / 2418 / 2566)
template <typename T, int FORM, int NB, int BM, bool SCANNED = false> __device__ __forceinline__ void even_body(const GemmArgs& a, const PgRows& experts) {
  constexpr bool GLU = FORM == PG_SWIGLU || FORM == PG_SWIGLU_KEEP;
  persistent_body<T, GLU, FORM == PG_WEIGHT_KN, FORM == PG_SWIGLU_KEEP, !GLU, NB, true, BM, SCANNED>(a, experts);
}

template <typename T, int FORM, int NB, int BM>
__global__ __launch_bounds__(256, 1) void grouped_gemm_even_kernel(GemmArgs a) {
  pg_fetch_arguments(a);
  even_body<T, FORM, NB, BM>(a, pg_rows(a.expert_offsets, a.L, a.E));
}

template <typename T, int FORM, int NB, int BM> static int launch_even(GemmArgs a, hipStream_t s) {
  constexpr int BN = (FORM == PG_SWIGLU || FORM == PG_SWIGLU_KEEP ? 16 : 32) * NB;
  constexpr int LDS = 3 * (BM + 32 * NB) * 128 <= PG_LDS ? 3 * (BM + 32 * NB) * 128 : PG_LDS;
  auto kern = grouped_gemm_even_kernel<T, FORM, NB, BM>;
  static std::atomic<uint64_t> lds_ok{0};
  int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), LDS, lds_ok), grid = 0;
  if (rc != MI_MOE_OK || (rc = persistent_prepare(a, BM, BN, &grid)) != MI_MOE_OK) return rc;
  a.ws = nullptr;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), LDS, s, a);
  return mi_launch_status();
}

template <typename T, int FORM> static int launch_even_tile(const GemmArgs& a, int tile, hipStream_t s) {
  switch (tile) {
    case EVEN_160x256: return launch_even<T, FORM, 8, 160>(a, s);
    case EVEN_256x256: return launch_even<T, FORM, 8, 256>(a, s);
  }
  if constexpr (FORM != PG_WEIGHT_KN) {
    switch (tile) {
      case EVEN_256x128: return launch_even<T, FORM, 4, 256>(a, s);
      case EVEN_224x192: return launch_even<T, FORM, 6, 224>(a, s);
    }
  }
  return MI_MOE_EUNSUPPORTED;
}
