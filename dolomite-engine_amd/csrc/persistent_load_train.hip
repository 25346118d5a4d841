// persistent_load.h for training: with the pre-activation, and with the weights as they lie for the data gradients.
#include "persistent_load.h"

int mi_gemm_by_load_train(const GemmArgs& a, int dtype, int form, hipStream_t s) {
  const bool bf = dtype == MI_MOE_BF16;
  switch (form) {
    case PG_SWIGLU_KEEP: return bf ? launch_by_load<bf16_t, PG_SWIGLU_KEEP>(a, s) : launch_by_load<f16_t, PG_SWIGLU_KEEP>(a, s);
    case PG_WEIGHT_KN: return bf ? launch_by_load<bf16_t, PG_WEIGHT_KN>(a, s) : launch_by_load<f16_t, PG_WEIGHT_KN>(a, s);
  }
  return MI_MOE_EUNSUPPORTED;
}
