// The even forms of the persistent grouped GEMM (persistent_even.hip) for training: with the pre-activation, and with the weights
// as they lie for the data gradients.
#include "persistent_even.h"

int mi_gemm_even_train(const GemmArgs& a, int dtype, int form, int tile, hipStream_t s) {
  const bool bf = dtype == MI_MOE_BF16;
  switch (form) {
    case PG_SWIGLU_KEEP:
      return bf ? launch_even_tile<bf16_t, PG_SWIGLU_KEEP>(a, tile, s) : launch_even_tile<f16_t, PG_SWIGLU_KEEP>(a, tile, s);
    case PG_WEIGHT_KN:
      return bf ? launch_even_tile<bf16_t, PG_WEIGHT_KN>(a, tile, s) : launch_even_tile<f16_t, PG_WEIGHT_KN>(a, tile, s);
  }
  return MI_MOE_EUNSUPPORTED;
}
