// The whole inference forward of the layer behind one call (moe.py:212-290 of
// lm_engine/hf_models/modeling_utils/mlp_blocks): router (with the block's RMSNorm) -> sort -> up-projection + SwiGLU ->
// down-projection -> [shared experts] -> combine with the block's tail.  Host code only: it picks the same entry points in
// the same order as the callers of the single stages, with every intermediate in one workspace.  A small batch is bound
// by the host: five launches through five calls with their own argument conversion and a dozen allocations took
// 60 - 68 us a pass whatever the kernels did.
#include "gemm_common.h"

// router_fused.hip
bool mi_rmsnorm_router_sorts(int T, int H, int E);
int mi_rmsnorm_router(const void* h, const void* ln_weight, float eps, const void* gate_w, const float* bias, int T, int H, int E,
                      int k, int dtype, void* x_norm_out, void* logits_out, void* gates_out, int32_t* idx_out,
                      int32_t* sorted_expert, int32_t* sorted_scattered, int32_t* expert_offsets, mi_moe_stream_t stream);

namespace {

struct LayerSpace {
  size_t gates, experts, sorted_expert, sorted_scattered, offsets, router, x_norm, act, o, shared_act, shared_out, bytes;
};

size_t take(size_t& at, size_t n) {
  const size_t p = at;
  at += (n + 255) / 256 * 256;
  return p;
}

LayerSpace layer_space(int T, int H, int E, int k, int I, int S, int elt, bool norm) {
  LayerSpace w = {};
  const size_t L = (size_t)T * k;
  size_t at = 0;
  w.gates = take(at, L * elt);
  w.experts = take(at, L * 4);
  w.sorted_expert = take(at, L * 4);
  w.sorted_scattered = take(at, L * 4);
  w.offsets = take(at, (size_t)E * 4);
  // one after the other: the router's, then the sort's
  size_t r = mi_moe_router_fused_sort_workspace_bytes(T, H, E, k);
  const size_t r1 = mi_moe_router_fused_workspace_bytes(T, H, E), r2 = mi_moe_sort_bin_workspace_bytes((int)L, E);
  r = r > r1 ? r : r1;
  r = r > r2 ? r : r2;
  w.router = take(at, r + 16);
  w.x_norm = take(at, norm ? (size_t)T * H * elt : 0);
  w.act = take(at, L * I * elt);
  w.o = take(at, L * H * elt);
  w.shared_act = take(at, (size_t)T * S * elt);
  w.shared_out = take(at, S > 0 ? (size_t)T * H * elt : 0);
  w.bytes = at;
  return w;
}

}  // namespace

extern "C" size_t mi_moe_layer_workspace_bytes(int T, int H, int E, int k, int I, int S, int dtype, int has_norm) {
  if (T < 1 || H < 1 || E < 1 || k < 1 || I < 1 || S < 0 || (long)T * k > 0x7fffffffL) return 0;
  return layer_space(T, H, E, k, I, S, dtype == MI_MOE_F32 ? 4 : 2, has_norm != 0).bytes;
}

extern "C" int mi_moe_layer_forward(const void* x, const void* norm_w, float norm_eps, int has_norm, const void* gate_w,
                                    const float* gate_bias, const void* logits, const void* w_fc, const float* fc_scale,
                                    const void* w_proj, const float* proj_scale, int w_tiled, const void* shared_fc,
                                    const void* shared_proj, const void* residual, float residual_scale, int has_scale, void* y,
                                    int T, int H, int E, int k, int I, int S, int dtype, void* ws, size_t ws_bytes,
                                    void* gemm_ws, size_t gemm_ws_bytes, mi_moe_stream_t stream) {
  if (T < 1 || H < 1 || E < 1 || k < 1 || k > E || I < 1 || S < 0 || (long)T * k > 0x7fffffffL) return MI_MOE_ESHAPE;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16 && dtype != MI_MOE_F32) return MI_MOE_EDTYPE;
  if (!x || !w_fc || !w_proj || !y || !ws || (!gate_w && !logits) || (S > 0 && (!shared_fc || !shared_proj))) return MI_MOE_ENULL;
  const int elt = dtype == MI_MOE_F32 ? 4 : 2;
  const LayerSpace w = layer_space(T, H, E, k, I, S, elt, has_norm != 0);
  if (ws_bytes < w.bytes) return MI_MOE_EWORKSPACE;
  unsigned char* b = static_cast<unsigned char*>(ws);
  const int L = T * k;
  void* gates = b + w.gates;
  int32_t* experts = reinterpret_cast<int32_t*>(b + w.experts);
  int32_t* se = reinterpret_cast<int32_t*>(b + w.sorted_expert);
  int32_t* ss = reinterpret_cast<int32_t*>(b + w.sorted_scattered);
  int32_t* off = reinterpret_cast<int32_t*>(b + w.offsets);
  void* rws = b + w.router;
  int rc;

  // router and sort: the forms and the order of the single calls, so that the routing does not depend on the caller
  bool sorted = false;
  if (has_norm) {
    if (logits) return MI_MOE_EUNSUPPORTED;
    void* xn = b + w.x_norm;
    sorted = mi_rmsnorm_router_sorts(T, H, E);
    if ((rc = mi_rmsnorm_router(x, norm_w, norm_eps, gate_w, gate_bias, T, H, E, k, dtype, xn, nullptr, gates, experts,
                                sorted ? se : nullptr, ss, off, stream)) != MI_MOE_OK)
      return rc;
    x = xn;
  } else if (logits) {
    if ((rc = mi_moe_router_topk_softmax(logits, T, E, k, dtype, gates, experts, stream)) != MI_MOE_OK) return rc;
  } else {
    const bool streaming = dtype != MI_MOE_F32 && E <= 64 && k <= 8 && H % 16 == 0;
    const size_t need = streaming ? mi_moe_router_fused_sort_workspace_bytes(T, H, E, k) : 0;
    if (need > 0) {
      rc = mi_moe_router_fused_sort(x, gate_w, gate_bias, T, H, E, k, dtype, nullptr, gates, experts, se, ss, off, rws, need, stream);
      sorted = true;
    } else {
      const size_t n = streaming || E > 64 ? mi_moe_router_fused_workspace_bytes(T, H, E) : 0;
      rc = mi_moe_router_fused(x, gate_w, gate_bias, T, H, E, k, dtype, nullptr, gates, experts, n ? rws : nullptr, n, stream);
    }
    if (rc != MI_MOE_OK) return rc;
  }
  if (!sorted) {
    const size_t n = mi_moe_sort_bin_workspace_bytes(L, E);
    if ((rc = mi_moe_sort_bin(experts, T, k, E, se, ss, off, rws, n < 16 ? 16 : n, stream)) != MI_MOE_OK) return rc;
  }

  // experts
  void* act = b + w.act;
  void* o = b + w.o;
  if (fc_scale) {
    if ((rc = mi_moe_up_swiglu_fp8(x, w_fc, fc_scale, act, ss, off, L, H, I, E, k, dtype, w_tiled & 1, stream)) != MI_MOE_OK) return rc;
    if ((rc = mi_moe_down_fp8(act, w_proj, proj_scale, o, ss, off, L, I, H, E, dtype, (w_tiled >> 1) & 1, stream)) != MI_MOE_OK) return rc;
  } else {
    void* up_ws = gemm_ws && mi_moe_grouped_gemm_splits(H, dtype) ? gemm_ws : nullptr;
    void* down_ws = gemm_ws && mi_moe_grouped_gemm_splits(I, dtype) ? gemm_ws : nullptr;
    if ((rc = mi_moe_up_swiglu_ws(x, w_fc, act, ss, off, L, H, I, E, k, dtype, -1, up_ws, gemm_ws_bytes, stream)) != MI_MOE_OK) return rc;
    if ((rc = mi_moe_scattered_gemm_ws(act, w_proj, o, ss, off, L, I, H, E, 1, 1, 0, dtype, -1, down_ws, gemm_ws_bytes, stream)) != MI_MOE_OK)
      return rc;
  }

  // shared experts: one expert that owns every token, rows in place
  void* shared = nullptr;
  if (S > 0) {
    void* sact = b + w.shared_act;
    shared = b + w.shared_out;
    if ((rc = mi_gemm_one_expert(x, shared_fc, sact, T, H, S, true, dtype, stream)) != MI_MOE_OK) return rc;
    if ((rc = mi_gemm_one_expert(sact, shared_proj, shared, T, S, H, false, dtype, stream)) != MI_MOE_OK) return rc;
  }
  if (!shared && !residual && !has_scale) return mi_moe_combine(o, gates, y, T, k, H, dtype, stream);
  return mi_moe_combine_block_tail(o, gates, shared, residual, residual_scale, has_scale, y, T, k, H, dtype, stream);
}
