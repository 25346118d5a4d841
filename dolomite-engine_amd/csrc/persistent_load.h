// The persistent grouped GEMM with the tiles that the load on hand wants: every workgroup counts the row tiles that each form would
// have, out of the experts' ends, and runs the form that persist_time finds the fastest (pg_form_by_load).  The host knows the
// average of the experts' rows only, and that says little about how many tiles there are: a form picked for rows that scatter
// around it goes into a second, nearly empty round as soon as a few experts have more of them.
//
// us of 256 x 256 tiles / the form for the average / this kernel, where the largest expert has so many times the average:
//                                          2.5 - 4.5 (logits lowered by 0.49 ln(rank))   1.4 - 1.7 (by 0.12)
//   40 experts, 1536 -> 512 SwiGLU,   700 tokens  39.2 / 51.7 / 37.7
//                                    1000         41.1 / 54.1 / 41.1                     40.9 / 55.8 / 41.5
//               512 -> 1536           700                                                20.6 / 26.7 / 21.1
//               with pre-activation  1400         47.0 / 63.2 / 47.6                     46.8 / 61.7 / 48.0
//   32 experts, 1024 -> 512 SwiGLU,   509 tokens  26.6 / 32.4 / 25.4
//                                    1000         28.5 / 38.2 / 29.3                     28.6 / 39.6 / 29.6
//   16 experts, 2048 -> 1024 SwiGLU, 2048 tokens  50.7 / 64.9 / 48.9                     49.9 / 73.0 / 49.5
//               transposed weights   2048         50.0 / 66.0 / 49.0                     48.4 / 70.8 / 48.6
//   8 experts, 14336 -> 4096,        1000 tokens   315 /  396 /  313
// 219 problems of 64 to 8192 tokens in 8 to 64 experts, all forms, against the form for the average: 0.996 of its time where the load
// is even, 0.964 and 0.953 in the two columns' loads.
#pragma once

#include "persistent_even.h"

template <typename T, int FORM, bool NT> __device__ __forceinline__ void whole_body(const GemmArgs& a, const PgRows& experts) {
  constexpr bool GLU = FORM == PG_SWIGLU || FORM == PG_SWIGLU_KEEP;
  persistent_body<T, GLU, FORM == PG_WEIGHT_KN, FORM == PG_SWIGLU_KEEP, NT, 8, false, 256, true>(a, experts);
}

template <typename T, int FORM> __global__ __launch_bounds__(256, 1) void grouped_gemm_by_load_kernel(GemmArgs a) {
  constexpr bool GLU = FORM == PG_SWIGLU || FORM == PG_SWIGLU_KEEP;
  pg_fetch_arguments(a);
  PgRows experts = pg_rows(a.expert_offsets, a.L, a.E);
  const int i = pg_form_by_load(a, experts, FORM, gridDim.x);
  if (i == 0) {
    if constexpr (FORM == PG_SWIGLU) {
      if (a.out_nt) whole_body<T, FORM, true>(a, experts);
      else whole_body<T, FORM, false>(a, experts);
    } else {
      whole_body<T, FORM, !GLU>(a, experts);
    }
    return;
  }
  a.ws = nullptr;
  auto as = [&](auto itag) __attribute__((always_inline)) {
    constexpr int I = decltype(itag)::value, NB = persist_form_blocks(I);
    if constexpr (FORM != PG_WEIGHT_KN || NB == 8) {
      persistent_columns(a, (GLU ? 16 : 32) * NB);
      even_body<T, FORM, NB, persist_form_rows(I), true>(a, experts);
    }
  };
  if (i == 1) as(std::integral_constant<int, 1>{});
  else if (i == 2) as(std::integral_constant<int, 2>{});
  else if (i == 3) as(std::integral_constant<int, 3>{});
  else as(std::integral_constant<int, 4>{});
}

template <typename T, int FORM> static int launch_by_load(GemmArgs a, hipStream_t s) {
  auto kern = grouped_gemm_by_load_kernel<T, FORM>;
  static std::atomic<uint64_t> lds_ok{0};
  int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), PG_LDS, lds_ok), grid = 0;
  if (rc != MI_MOE_OK || (rc = by_load_prepare(a, FORM, &grid)) != MI_MOE_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), PG_LDS, s, a);
  if ((rc = mi_launch_status()) != MI_MOE_OK || a.ws == nullptr) return rc;
  return mi_gemm_split_finish(a, std::is_same<T, bf16_t>::value ? MI_MOE_BF16 : MI_MOE_F16, FORM, grid / 8, true, s);
}
