// persistent_load.h for inference: plain and SwiGLU.
#include "persistent_load.h"

int mi_gemm_by_load(const GemmArgs& a, int dtype, int form, hipStream_t s) {
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  const bool bf = dtype == MI_MOE_BF16;
  switch (form) {
    case PG_PLAIN: return bf ? launch_by_load<bf16_t, PG_PLAIN>(a, s) : launch_by_load<f16_t, PG_PLAIN>(a, s);
    case PG_SWIGLU: return bf ? launch_by_load<bf16_t, PG_SWIGLU>(a, s) : launch_by_load<f16_t, PG_SWIGLU>(a, s);
  }
  return mi_gemm_by_load_train(a, dtype, form, s);
}
