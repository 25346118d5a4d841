// The whole inference forward of the layer behind one call (moe.py:212-290 of
// lm_engine/hf_models/modeling_utils/mlp_blocks): router (with the block's RMSNorm) -> sort -> up-projection + SwiGLU ->
// down-projection -> [shared experts] -> combine with the block's tail.  Host code only: it picks the same entry points in
// the same order as the callers of the single stages, with every intermediate in one workspace.  A small batch is bound
// by the host: five launches through five calls with their own argument conversion and a dozen allocations took
// 60 - 68 us a pass whatever the kernels did.
#include "gemm_common.h"

#include <initializer_list>

// router_fused.hip
bool mi_rmsnorm_router_sorts(int T, int H, int E);
int mi_rmsnorm_router(const void* h, const void* ln_weight, float eps, const void* gate_w, const float* bias, int T, int H, int E,
                      int k, int dtype, void* x_norm_out, void* logits_out, void* gates_out, int32_t* idx_out,
                      int32_t* sorted_expert, int32_t* sorted_scattered, int32_t* expert_offsets, int32_t* hist,
                      mi_moe_stream_t stream);
size_t mi_rmsnorm_router_sort_bytes(int T, int H, int E, int k);

// combine.hip, backward.hip, aux_loss.hip, grouped_wgrad.hip
int mi_combine_sum(const void* o, const void* add, void* y, int T, int k, int H, int dtype, mi_moe_stream_t stream);
int mi_swiglu_backward(const void* h, const void* d_act, const void* gates, const int32_t* sorted_scattered, void* d_h, void* act_g,
                       void* d_gates, int32_t* tokens, int L, int I, int k, int dtype, mi_moe_stream_t stream);
int mi_aux_loss(const void* logits, const int32_t* topk_idx, float* loss_w, void* loss_out, void* workspace, size_t workspace_bytes,
                int T, int E, int k, int dtype, mi_moe_stream_t stream);
int mi_router_dlogits_aux(const void* logits, const int32_t* idx, const void* d_gates, const float* loss_w, const void* grad,
                          void* d_logits, int T, int E, int k, int dtype, hipStream_t s);
int mi_grouped_wgrad(const void* a, const int32_t* a_idx, const void* b, const int32_t* b_idx, const int32_t* expert_offsets, void* dw,
                     void* workspace, size_t workspace_bytes, int L, int a_rows, int b_rows, int M, int N, int E, int dtype,
                     mi_moe_stream_t stream, bool entry);
size_t mi_grouped_wgrad_bytes(int L, int a_rows, int b_rows, int M, int N, int E);

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
  const size_t r3 = norm ? mi_rmsnorm_router_sort_bytes(T, H, E, k) : 0;
  r = r > r3 ? r : r3;
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
    const bool counts = mi_rmsnorm_router_sort_bytes(T, H, E, k) > 0;
    sorted = counts || mi_rmsnorm_router_sorts(T, H, E);
    if ((rc = mi_rmsnorm_router(x, norm_w, norm_eps, gate_w, gate_bias, T, H, E, k, dtype, xn, nullptr, gates, experts,
                                sorted ? se : nullptr, ss, off, counts ? static_cast<int32_t*>(rws) : nullptr, stream)) != MI_MOE_OK)
      return rc;
    x = xn;
  } else if (logits) {
    if ((rc = mi_moe_router_topk_softmax(logits, T, E, k, dtype, gates, experts, stream)) != MI_MOE_OK) return rc;
  } else {
    const bool streaming = dtype != MI_MOE_F32 && E <= 64 && k <= 8 && H % 16 == 0;
    const size_t need = streaming ? mi_moe_router_fused_sort_workspace_bytes(T, H, E, k) : 0;
    if (dtype != MI_MOE_F32 && H % 16 != 0) {
      rc = mi_moe_router_ragged(x, gate_w, gate_bias, T, H, E, k, dtype, nullptr, gates, experts, stream);
    } else if (need > 0) {
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

// ---- a training step's routed experts, forward and backward ----------------------------------------------------------------
// The launches of autograd.FusedRouter, SwitchAuxLoss and ScatteredSwiGLUExperts (16-bit, pre-activation kept), one call each
// way.  Behind one call the router's gradient of x is added where the k rows of a token are summed, instead of in a pass of its own
// over both (32768 tokens of 1536: 46 us; with shared experts it is handed back apart, see autograd.RoutedExperts), the rows' tokens come out of the SwiGLU's backward, and the loss and its gradient stay
// in the logits' type (three small launches).
namespace {

struct TrainSpace {
  size_t h, logits, gates, experts, sorted_scattered, offsets, loss_w, saved;  // kept for the backward
  size_t router, aux, sorted_expert, act, o, forward;                          // the forward's workspace
  size_t a, act_g, d_h, d_gates, tokens, d_logits, dx_router, backward;        // the backward's
};

size_t larger(size_t a, size_t b) { return a > b ? a : b; }

TrainSpace train_space(int T, int H, int E, int k, int I) {
  TrainSpace w = {};
  const size_t L = (size_t)T * k, elt = 2;
  size_t at = 0;
  w.h = take(at, L * 2 * I * elt);
  w.logits = take(at, (size_t)T * E * elt);
  w.gates = take(at, L * elt);
  w.experts = take(at, L * 4);
  w.sorted_scattered = take(at, L * 4);
  w.offsets = take(at, (size_t)E * 4);
  w.loss_w = take(at, ((size_t)E + 1) * 4);
  w.saved = at;
  at = 0;
  const size_t r = larger(mi_moe_router_fused_sort_workspace_bytes(T, H, E, k), mi_moe_router_fused_workspace_bytes(T, H, E));
  w.router = take(at, larger(r, mi_moe_sort_bin_workspace_bytes((int)L, E)) + 16);
  w.aux = take(at, mi_moe_aux_loss_workspace_bytes(T, E));
  w.sorted_expert = take(at, L * 4);
  w.act = take(at, L * I * elt);
  w.o = take(at, L * H * elt);
  w.forward = at;
  at = 0;
  // one after the other: the gradient of the activation with the gated activation behind it, the workspace of the down-projection's
  // weight gradient in place of the former, the slots' gradient of x, the other weight gradients' workspace
  const size_t wg = larger(mi_grouped_wgrad_bytes((int)L, (int)L, T, 2 * I, H, E), mi_grouped_wgrad_bytes(T, T, T, E, H, 1));
  const size_t front = (larger(L * I * elt, mi_grouped_wgrad_bytes((int)L, T, (int)L, H, I, E)) + 255) / 256 * 256;
  w.a = take(at, larger(larger(front + L * I * elt, L * H * elt), wg));
  w.act_g = w.a + front;
  w.d_h = take(at, L * 2 * I * elt);
  w.d_gates = take(at, L * elt);
  w.tokens = take(at, L * 4);
  w.d_logits = take(at, (size_t)T * E * elt);
  w.dx_router = take(at, (size_t)T * H * elt);
  w.backward = at;
  return w;
}

}  // namespace

// Everything that a call of the two below needs to be taken by every launch, but for the alignment of its pointers.
static bool train_ok(int T, int H, int E, int k, int I, int dtype) {
  if (T < 1 || H < 1 || E < 1 || k < 1 || k > E || I < 1) return false;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return false;
  if (E > 64 || k > 8 || E % 8 != 0 || H % 16 != 0 || I % 8 != 0) return false;
  const double L = (double)T * k, most = 2147483648.0;
  return L * H < most && L * 2 * I < most && (double)E * 2 * I * H < most;
}

extern "C" int mi_moe_layer_train_sizes(int T, int H, int E, int k, int I, int dtype, size_t* saved, size_t* forward_ws, size_t* backward_ws) {
  if (!saved || !forward_ws || !backward_ws) return MI_MOE_ENULL;
  if (!train_ok(T, H, E, k, I, dtype)) return MI_MOE_EUNSUPPORTED;
  const TrainSpace w = train_space(T, H, E, k, I);
  *saved = w.saved;
  *forward_ws = w.forward;
  *backward_ws = w.backward;
  return MI_MOE_OK;
}

extern "C" int mi_moe_layer_train_forward(const void* x, const void* gate_w, const float* gate_bias, const void* w_fc, const void* w_proj,
                                          void* y, void* aux_loss, void* saved, size_t saved_bytes, int T, int H, int E, int k, int I,
                                          int dtype, void* ws, size_t ws_bytes, void* gemm_ws, size_t gemm_ws_bytes, mi_moe_stream_t stream) {
  if (!train_ok(T, H, E, k, I, dtype)) return MI_MOE_EUNSUPPORTED;
  if (!x || !gate_w || !w_fc || !w_proj || !y || !aux_loss || !saved || !ws) return MI_MOE_ENULL;
  for (const void* p : {x, gate_w, w_fc, w_proj, static_cast<const void*>(y), static_cast<const void*>(saved), static_cast<const void*>(ws)})
    if (!mi_aligned(p, 16)) return MI_MOE_EALIGN;
  const TrainSpace w = train_space(T, H, E, k, I);
  if (saved_bytes < w.saved || ws_bytes < w.forward) return MI_MOE_EWORKSPACE;
  unsigned char *k0 = static_cast<unsigned char*>(saved), *b = static_cast<unsigned char*>(ws);
  const int L = T * k;
  void *h = k0 + w.h, *logits = k0 + w.logits, *gates = k0 + w.gates;
  int32_t* experts = reinterpret_cast<int32_t*>(k0 + w.experts);
  int32_t* ss = reinterpret_cast<int32_t*>(k0 + w.sorted_scattered);
  int32_t* off = reinterpret_cast<int32_t*>(k0 + w.offsets);
  int32_t* se = reinterpret_cast<int32_t*>(b + w.sorted_expert);
  float* loss_w = reinterpret_cast<float*>(k0 + w.loss_w);
  void *rws = b + w.router, *act = b + w.act, *o = b + w.o;
  int rc;
  const size_t need = mi_moe_router_fused_sort_workspace_bytes(T, H, E, k);
  if (need > 0) {
    rc = mi_moe_router_fused_sort(x, gate_w, gate_bias, T, H, E, k, dtype, logits, gates, experts, se, ss, off, rws, need, stream);
  } else {
    const size_t n = mi_moe_router_fused_workspace_bytes(T, H, E), m = mi_moe_sort_bin_workspace_bytes(L, E);
    rc = mi_moe_router_fused(x, gate_w, gate_bias, T, H, E, k, dtype, logits, gates, experts, n ? rws : nullptr, n, stream);
    if (rc == MI_MOE_OK) rc = mi_moe_sort_bin(experts, T, k, E, se, ss, off, rws, m < 16 ? 16 : m, stream);
  }
  if (rc != MI_MOE_OK) return rc;
  rc = mi_aux_loss(logits, experts, loss_w, aux_loss, b + w.aux, mi_moe_aux_loss_workspace_bytes(T, E), T, E, k, dtype, stream);
  if (rc != MI_MOE_OK) return rc;
  rc = mi_moe_up_swiglu_keep(x, w_fc, act, h, ss, off, L, H, I, E, k, dtype, stream);
  if (rc == MI_MOE_EUNSUPPORTED) {
    // few rows per expert: the product and the activation apart
    void* up_ws = gemm_ws && mi_moe_grouped_gemm_splits(H, dtype) ? gemm_ws : nullptr;
    rc = mi_moe_scattered_gemm_ws(x, w_fc, h, ss, off, L, H, 2 * I, E, k, 0, 1, dtype, -1, up_ws, gemm_ws_bytes, stream);
    if (rc == MI_MOE_OK) rc = mi_moe_swiglu_forward(h, act, L, I, dtype, stream);
  }
  if (rc != MI_MOE_OK) return rc;
  void* down_ws = gemm_ws && mi_moe_grouped_gemm_splits(I, dtype) ? gemm_ws : nullptr;
  rc = mi_moe_scattered_gemm_ws(act, w_proj, o, ss, off, L, I, H, E, 1, 1, 0, dtype, -1, down_ws, gemm_ws_bytes, stream);
  return rc != MI_MOE_OK ? rc : mi_moe_combine(o, gates, y, T, k, H, dtype, stream);
}

extern "C" int mi_moe_layer_train_backward_parts(const void* x, const void* gate_w, const void* w_fc, const void* w_proj, const void* saved,
                                                 size_t saved_bytes, const void* dy, const void* d_aux, void* dx, void* dx_router_out,
                                                 void* d_gate_w, void* d_w_fc, void* d_w_proj, int T, int H, int E, int k, int I, int dtype,
                                                 void* ws, size_t ws_bytes, void* gemm_ws, size_t gemm_ws_bytes, mi_moe_stream_t stream) {
  if (!train_ok(T, H, E, k, I, dtype)) return MI_MOE_EUNSUPPORTED;
  if (!x || !gate_w || !w_fc || !w_proj || !saved || !ws || (!dy && !d_aux) || (!dy && (d_w_fc || d_w_proj || (dx && dx_router_out)))) return MI_MOE_ENULL;
  for (const void* p : {x, gate_w, w_fc, w_proj, saved, dy, static_cast<const void*>(dx), static_cast<const void*>(dx_router_out), static_cast<const void*>(d_gate_w),
                        static_cast<const void*>(d_w_fc), static_cast<const void*>(d_w_proj), static_cast<const void*>(ws)})
    if (!mi_aligned(p, 16)) return MI_MOE_EALIGN;
  const TrainSpace w = train_space(T, H, E, k, I);
  if (saved_bytes < w.saved || ws_bytes < w.backward) return MI_MOE_EWORKSPACE;
  const unsigned char* k0 = static_cast<const unsigned char*>(saved);
  unsigned char* b = static_cast<unsigned char*>(ws);
  const int L = T * k;
  const void *h = k0 + w.h, *logits = k0 + w.logits, *gates = k0 + w.gates;
  const int32_t* experts = reinterpret_cast<const int32_t*>(k0 + w.experts);
  const int32_t* ss = reinterpret_cast<const int32_t*>(k0 + w.sorted_scattered);
  const int32_t* off = reinterpret_cast<const int32_t*>(k0 + w.offsets);
  const float* loss_w = reinterpret_cast<const float*>(k0 + w.loss_w);
  void *a = b + w.a, *d_h = b + w.d_h, *act_g = b + w.act_g, *d_logits = b + w.d_logits;
  void* d_gates = dy ? b + w.d_gates : nullptr;
  int32_t* tokens = reinterpret_cast<int32_t*>(b + w.tokens);
  // the router's gradient of x: on its own, or all of dx, or what the sum over a token's rows adds
  void* dx_router = dx_router_out ? dx_router_out : !dx ? nullptr : dy ? b + w.dx_router : dx;
  const bool router = dx_router || d_gate_w;
  auto split = [&](int K) { return gemm_ws && mi_moe_grouped_gemm_splits(K, dtype) ? gemm_ws : nullptr; };
  auto wgrad = [&](const void* ga, const int32_t* ai, const void* gb, const int32_t* bi, const int32_t* offsets, void* dw, int rows, int a_rows,
                   int b_rows, int M, int N, int experts_) {
    return mi_grouped_wgrad(ga, ai, gb, bi, offsets, dw, a, mi_grouped_wgrad_bytes(rows, a_rows, b_rows, M, N, experts_), rows, a_rows, b_rows, M, N,
                            experts_, dtype, stream, false);
  };
  int rc;
  if (dy) {
    // gradient of the activation, in sorted order and before the router weight; then d h, gate times activation, and d gates
    if ((rc = mi_moe_scattered_gemm_wt_ws(dy, w_proj, a, ss, off, L, H, I, E, k, 0, 1, dtype, split(H), gemm_ws_bytes, stream)) != MI_MOE_OK) return rc;
    if ((rc = mi_swiglu_backward(h, a, gates, ss, d_h, act_g, d_gates, tokens, L, I, k, dtype, stream)) != MI_MOE_OK) return rc;
    if (d_w_proj && (rc = wgrad(dy, tokens, act_g, nullptr, off, d_w_proj, L, T, L, H, I, E)) != MI_MOE_OK) return rc;
  }
  if (router) {
    if ((rc = mi_router_dlogits_aux(logits, experts, d_gates, loss_w, d_aux, d_logits, T, E, k, dtype, static_cast<hipStream_t>(stream))) != MI_MOE_OK)
      return rc;
    if (dx_router && (rc = mi_gemm_one_expert_wt(d_logits, gate_w, dx_router, T, E, H, dtype, stream)) != MI_MOE_OK) return rc;
  }
  if (dy && dx) {
    if ((rc = mi_moe_scattered_gemm_wt_ws(d_h, w_fc, a, ss, off, L, 2 * I, H, E, 1, 1, 0, dtype, split(2 * I), gemm_ws_bytes, stream)) != MI_MOE_OK)
      return rc;
    if ((rc = mi_combine_sum(a, dx_router_out ? nullptr : dx_router, dx, T, k, H, dtype, stream)) != MI_MOE_OK) return rc;
  }
  if (d_w_fc && (rc = wgrad(d_h, nullptr, x, tokens, off, d_w_fc, L, L, T, 2 * I, H, E)) != MI_MOE_OK) return rc;
  if (d_gate_w && (rc = wgrad(d_logits, nullptr, x, nullptr, nullptr, d_gate_w, T, T, T, E, H, 1)) != MI_MOE_OK) return rc;
  return MI_MOE_OK;
}

extern "C" int mi_moe_layer_train_backward(const void* x, const void* gate_w, const void* w_fc, const void* w_proj, const void* saved,
                                           size_t saved_bytes, const void* dy, const void* d_aux, void* dx, void* d_gate_w, void* d_w_fc,
                                           void* d_w_proj, int T, int H, int E, int k, int I, int dtype, void* ws, size_t ws_bytes,
                                           void* gemm_ws, size_t gemm_ws_bytes, mi_moe_stream_t stream) {
  return mi_moe_layer_train_backward_parts(x, gate_w, w_fc, w_proj, saved, saved_bytes, dy, d_aux, dx, nullptr, d_gate_w, d_w_fc, d_w_proj, T, H,
                                           E, k, I, dtype, ws, ws_bytes, gemm_ws, gemm_ws_bytes, stream);
}
