// Training-mode auxiliary loss of the router (lm_engine/hf_models/modeling_utils/mlp_blocks/moe.py:346-369,
// single data-parallel rank) and its gradient with respect to the logits:
//
//   loss = E * sum_e  A_e / max(sum A, eps) * f_e / max(sum f, eps)  +  0.1 * mean_t( logsumexp(logits[t])^2 )
//   A_e = sum_t softmax(logits[t])_e,  f_e = number of (token, slot) pairs routed to expert e,  eps = 1e-12
//
// Forward: one pass over the (T, E) logits -- a wave per row computes the row's logsumexp and probabilities
// and keeps per-lane sums; a workgroup writes one partial per column [A (E) | f (E) | sum lse^2]; a second kernel
// adds each column's partials in a fixed order (deterministic) and a third, one workgroup, forms the loss and
// w_e = d loss / d A_e.
// Backward: d logits[t, j] = g * p_tj * ( w_j - sum_e p_te w_e  +  0.2 / T * lse_t ), one more pass.
// All arithmetic in fp32 from the logits as stored; the eager module rounds its intermediates to the model
// dtype instead, so the two agree to that dtype's rounding, not bit for bit.
#include "common.h"
#include "topk_row.h"

#define AUX_MAX_E 256
#define AUX_ROWS_PER_BLOCK 32

// (backward) lane holds experts lane, lane + 64, ... (at most 4 of them); returns the row's logsumexp and
// leaves the probabilities in p[]
template <typename T>
__device__ __forceinline__ float aux_row_softmax(const T* __restrict__ row, int E, int lane, float (&p)[4]) {
  float x[4];
  float mx = -INFINITY;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane + 64 * i;
    x[i] = e < E ? Elt<T>::load(row + e) : -INFINITY;
    mx = fmaxf(mx, x[i]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) mx = fmaxf(mx, __shfl_xor(mx, off, MI_WAVE));
  float sum = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    p[i] = lane + 64 * i < E ? __expf(x[i] - mx) : 0.f;
    sum += p[i];
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) sum += __shfl_xor(sum, off, MI_WAVE);
  const float inv = 1.0f / sum;
#pragma unroll
  for (int i = 0; i < 4; ++i) p[i] *= inv;
  return mx + __logf(sum);
}

// A wave has eight rows, NE columns a lane.  It is a chain of latencies (a load, two butterflies and two transcendentals a
// row; 509 tokens are 16 blocks), so the loads of all rows are issued at once and the rows' butterflies run side by
// side; the sums take the rows in order.  509 tokens of 32 experts: 12.5 -> 7.2 us.
template <typename T, int NE>
__global__ __launch_bounds__(256) void aux_loss_partial_kernel(const T* __restrict__ logits, const int32_t* __restrict__ topk_idx,
                                                               float* __restrict__ partial, int Trows, int E, int k) {
  constexpr int R = AUX_ROWS_PER_BLOCK / 4;
  __shared__ float acc[4][AUX_MAX_E];
  __shared__ int cnt[AUX_MAX_E];
  __shared__ float zsum[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row0 = (long)blockIdx.x * AUX_ROWS_PER_BLOCK + wave;  // rows row0 + 4 r
  float x[R][NE], mx[R], sum[R];
  int id[R];
#pragma unroll
  for (int r = 0; r < R; ++r) {
    const long t = row0 + 4 * r;
    const bool in = t < Trows;
#pragma unroll
    for (int i = 0; i < NE; ++i) x[r][i] = in && lane + 64 * i < E ? Elt<T>::load(logits + t * E + lane + 64 * i) : -INFINITY;
    id[r] = in && lane < k ? topk_idx[t * k + lane] : -1;
  }
  for (int e = threadIdx.x; e < E; e += 256) cnt[e] = 0;
  __syncthreads();
#pragma unroll
  for (int r = 0; r < R; ++r) {
    mx[r] = x[r][0];
#pragma unroll
    for (int i = 1; i < NE; ++i) mx[r] = fmaxf(mx[r], x[r][i]);
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r) mx[r] = fmaxf(mx[r], __shfl_xor(mx[r], off, MI_WAVE));
#pragma unroll
  for (int r = 0; r < R; ++r) {
    sum[r] = 0.f;
#pragma unroll
    for (int i = 0; i < NE; ++i) {
      x[r][i] = lane + 64 * i < E ? __expf(x[r][i] - mx[r]) : 0.f;
      sum[r] += x[r][i];
    }
  }
#pragma unroll
  for (int off = 32; off > 0; off >>= 1)
#pragma unroll
    for (int r = 0; r < R; ++r) sum[r] += __shfl_xor(sum[r], off, MI_WAVE);
  float a[NE] = {};
  float z = 0.f;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (row0 + 4 * r >= Trows) continue;
    const float inv = 1.0f / sum[r], lse = mx[r] + __logf(sum[r]);
#pragma unroll
    for (int i = 0; i < NE; ++i) a[i] += x[r][i] * inv;
    z = fmaf(lse, lse, z);
    if (id[r] >= 0 && id[r] < E) atomicAdd(&cnt[id[r]], 1);  // integer: the order does not matter
    for (int j = lane + 64; j < k; j += 64) {
      const int e = topk_idx[(row0 + 4 * r) * k + j];
      if (e >= 0 && e < E) atomicAdd(&cnt[e], 1);
    }
  }
#pragma unroll
  for (int i = 0; i < NE; ++i)
    if (lane + 64 * i < E) acc[wave][lane + 64 * i] = a[i];
  if (lane == 0) zsum[wave] = z;
  __syncthreads();
  // partial[column][block], columns = [A (E) | f (E) | sum lse^2]
  float* out = partial + blockIdx.x;
  const size_t nb = gridDim.x;
  for (int e = threadIdx.x; e < E; e += 256) {
    out[e * nb] = ((acc[0][e] + acc[1][e]) + acc[2][e]) + acc[3][e];
    out[(E + e) * nb] = (float)cnt[e];
  }
  if (threadIdx.x == 0) out[2 * E * nb] = ((zsum[0] + zsum[1]) + zsum[2]) + zsum[3];
}

// column sums of the partials: a wave per column, lanes stride over the blocks, then a fixed butterfly -- the same
// order every run
__global__ __launch_bounds__(256) void aux_loss_colsum_kernel(const float* __restrict__ partial, float* __restrict__ colsum,
                                                              int nblocks, int ncols) {
  const int lane = threadIdx.x & 63;
  const int c = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (c >= ncols) return;
  float s = 0.f;
  for (int b = lane; b < nblocks; b += 64) s += partial[(size_t)c * nblocks + b];
#pragma unroll
  for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, MI_WAVE);
  if (lane == 0) colsum[c] = s;
}

// loss_w[0] = loss, loss_w[1 + e] = d loss / d A_e; loss_out (or null): the loss in the logits' type.  The column sums are taken here,
// as aux_loss_colsum_kernel takes them, while a column is few blocks; else `partial` holds them already (nblocks = 1).
template <typename T>
__global__ __launch_bounds__(1024) void aux_loss_finish_kernel(const float* __restrict__ partial, int nblocks,
                                                               float* __restrict__ loss_w, T* __restrict__ loss_out, int Trows, int E) {
  __shared__ float A[AUX_MAX_E], F[AUX_MAX_E];
  __shared__ float scal[4];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll 4
  for (int c = wave; c < 2 * E + 1; c += 16) {
    float v = lane < nblocks ? partial[(size_t)c * nblocks + lane] : 0.f;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) v += __shfl_xor(v, off, MI_WAVE);
    if (lane == 0) (c < E ? A[c] : c < 2 * E ? F[c - E] : scal[3]) = v;
  }
  __syncthreads();
  if (wave == 0) {
    // lane l has experts l, 64 + l, ...; fixed butterflies (one thread's walk over 32 experts and its divisions took 3 us)
    float av[AUX_MAX_E / 64], fv[AUX_MAX_E / 64], sa = 0.f, sf = 0.f, dot = 0.f;
#pragma unroll
    for (int i = 0; i < AUX_MAX_E / 64; ++i) {
      const int e = lane + 64 * i;
      av[i] = e < E ? A[e] : 0.f;
      fv[i] = e < E ? F[e] : 0.f;
      sa += av[i];
      sf += fv[i];
    }
    sa = fmaxf(wave_sum_f32(sa), 1e-12f);
    sf = fmaxf(wave_sum_f32(sf), 1e-12f);
#pragma unroll
    for (int i = 0; i < AUX_MAX_E / 64; ++i) dot = fmaf(av[i] / sa, fv[i] / sf, dot);
    const float sw = (float)E * wave_sum_f32(dot);
    if (lane == 0) {
      scal[0] = sa;
      scal[1] = sf;
      scal[2] = sw;
      const float loss = sw + 0.1f * (scal[3] / (float)Trows);
      loss_w[0] = loss;
      if (loss_out != nullptr) Elt<T>::store(loss_out, loss);
    }
  }
  __syncthreads();
  // d/dA_e [ sum_e' A_e' c_e' / S ] = (c_e - switch) / S  with c_e = E f_e / sum f  (S = sum A above its floor)
  for (int e = threadIdx.x; e < E; e += 1024) loss_w[1 + e] = ((float)E * F[e] / scal[1] - scal[2]) / scal[0];
}

template <typename T>
__global__ __launch_bounds__(256) void aux_loss_backward_kernel(const T* __restrict__ logits, const float* __restrict__ loss_w,
                                                                const float* __restrict__ grad, T* __restrict__ d_logits,
                                                                int Trows, int E) {
  const int lane = threadIdx.x & 63;
  const float g = grad[0];
  const float zc = 0.2f / (float)Trows;
  float w[4];
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = lane + 64 * i < E ? loss_w[1 + lane + 64 * i] : 0.f;
  for (int t = blockIdx.x * 4 + (threadIdx.x >> 6); t < Trows; t += gridDim.x * 4) {
    float p[4];
    const float lse = aux_row_softmax<T>(logits + (size_t)t * E, E, lane, p);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s = fmaf(p[i], w[i], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, MI_WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int e = lane + 64 * i;
      if (e < E) Elt<T>::store(d_logits + (size_t)t * E + e, g * p[i] * ((w[i] - s) + zc * lse));
    }
  }
}

static int aux_blocks(int T) { return mi_ceil_div(T, AUX_ROWS_PER_BLOCK); }

extern "C" size_t mi_moe_aux_loss_workspace_bytes(int T, int E) {
  if (T < 1 || E < 1) return 0;
  // [partials: (2E + 1) columns x blocks][column sums: 2E + 1]
  return ((size_t)aux_blocks(T) + 1) * (2 * (size_t)E + 1) * sizeof(float);
}

template <typename T>
static void aux_forward_launch(const void* logits, const int32_t* idx, float* ws, float* loss_w, void* loss_out, int Trows, int E,
                               int k, hipStream_t s) {
  const int nb = aux_blocks(Trows);
  auto kern = E <= 64 ? aux_loss_partial_kernel<T, 1> : aux_loss_partial_kernel<T, AUX_MAX_E / 64>;
  hipLaunchKernelGGL(kern, dim3(nb), dim3(256), 0, s, static_cast<const T*>(logits), idx, ws, Trows, E, k);
  const int ncols = 2 * E + 1;
  float* colsum = ws + (size_t)nb * ncols;
  if (nb > 64) hipLaunchKernelGGL(aux_loss_colsum_kernel, dim3(mi_ceil_div(ncols, 4)), dim3(256), 0, s, ws, colsum, nb, ncols);
  hipLaunchKernelGGL((aux_loss_finish_kernel<T>), dim3(1), dim3(1024), 0, s, nb > 64 ? colsum : ws, nb > 64 ? 1 : nb, loss_w,
                     static_cast<T*>(loss_out), Trows, E);
}

// loss_out (or null): the loss in `dtype` as well
int mi_aux_loss(const void* logits, const int32_t* topk_idx, float* loss_w, void* loss_out, void* workspace, size_t workspace_bytes,
                int T, int E, int k, int dtype, mi_moe_stream_t stream) {
  if (T < 1 || E < 1 || k < 1) return MI_MOE_ESHAPE;
  if (E > AUX_MAX_E) return MI_MOE_EUNSUPPORTED;
  if (!logits || !topk_idx || !loss_w) return MI_MOE_ENULL;
  if (!workspace || workspace_bytes < mi_moe_aux_loss_workspace_bytes(T, E)) return MI_MOE_EWORKSPACE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  float* ws = static_cast<float*>(workspace);
  switch (dtype) {
    case MI_MOE_F32: aux_forward_launch<float>(logits, topk_idx, ws, loss_w, loss_out, T, E, k, s); break;
    case MI_MOE_F16: aux_forward_launch<f16_t>(logits, topk_idx, ws, loss_w, loss_out, T, E, k, s); break;
    case MI_MOE_BF16: aux_forward_launch<bf16_t>(logits, topk_idx, ws, loss_w, loss_out, T, E, k, s); break;
    default: return MI_MOE_EDTYPE;
  }
  return mi_launch_status();
}

extern "C" int mi_moe_aux_loss(const void* logits, const int32_t* topk_idx, float* loss_w, void* workspace,
                               size_t workspace_bytes, int T, int E, int k, int dtype, mi_moe_stream_t stream) {
  return mi_aux_loss(logits, topk_idx, loss_w, nullptr, workspace, workspace_bytes, T, E, k, dtype, stream);
}

extern "C" int mi_moe_aux_loss_backward(const void* logits, const float* loss_w, const float* grad, void* d_logits, int T,
                                        int E, int dtype, mi_moe_stream_t stream) {
  if (T < 1 || E < 1) return MI_MOE_ESHAPE;
  if (E > AUX_MAX_E) return MI_MOE_EUNSUPPORTED;
  if (!logits || !loss_w || !grad || !d_logits) return MI_MOE_ENULL;
  hipStream_t s = static_cast<hipStream_t>(stream);
  long blocks = ((long)T + 3) / 4;
  if (blocks > 256L * 16) blocks = 256L * 16;
  switch (dtype) {
    case MI_MOE_F32:
      hipLaunchKernelGGL((aux_loss_backward_kernel<float>), dim3((unsigned)blocks), dim3(256), 0, s,
                         static_cast<const float*>(logits), loss_w, grad, static_cast<float*>(d_logits), T, E);
      break;
    case MI_MOE_F16:
      hipLaunchKernelGGL((aux_loss_backward_kernel<f16_t>), dim3((unsigned)blocks), dim3(256), 0, s,
                         static_cast<const f16_t*>(logits), loss_w, grad, static_cast<f16_t*>(d_logits), T, E);
      break;
    case MI_MOE_BF16:
      hipLaunchKernelGGL((aux_loss_backward_kernel<bf16_t>), dim3((unsigned)blocks), dim3(256), 0, s,
                         static_cast<const bf16_t*>(logits), loss_w, grad, static_cast<bf16_t*>(d_logits), T, E);
      break;
    default: return MI_MOE_EDTYPE;
  }
  return mi_launch_status();
}

// d logits of a training step in one pass: the auxiliary loss's part as above, rounded, and the gates' part of
// router_dlogits_kernel (router_general.hip) on top of it, with the same roundings.  grad (or null: no such part) is the loss's
// upstream gradient in the logits' type, d_gates (or null) the gates'.
template <typename T>
__global__ __launch_bounds__(256) void router_dlogits_aux_kernel(const T* __restrict__ logits, const int32_t* __restrict__ idx,
                                                                 const T* __restrict__ d_gates, const float* __restrict__ loss_w,
                                                                 const T* __restrict__ grad, T* __restrict__ d_logits, int Trows, int E,
                                                                 int k) {
  const int lane = threadIdx.x & 63;
  const int t = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (t >= Trows) return;
  const float gl = grad != nullptr ? Elt<T>::load(grad) : 0.f;
  const float zc = 0.2f / (float)Trows;
  float w[4], base[4] = {};
#pragma unroll
  for (int i = 0; i < 4; ++i) w[i] = grad != nullptr && lane + 64 * i < E ? loss_w[1 + lane + 64 * i] : 0.f;
  // picked logit, its expert and the incoming gradient of slot j = lane (k <= 64)
  int e_j = 0;
  float z = -INFINITY, g = 0.f;
  if (d_gates != nullptr && lane < k) {
    e_j = idx[(size_t)t * k + lane];
    z = Elt<T>::load(logits + (size_t)t * E + e_j);
    g = Elt<T>::load(d_gates + (size_t)t * k + lane);
  }
  if (grad != nullptr) {
    float p[4];
    const float lse = aux_row_softmax<T>(logits + (size_t)t * E, E, lane, p);
    float s = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) s = fmaf(p[i], w[i], s);
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) s += __shfl_xor(s, off, MI_WAVE);
#pragma unroll
    for (int i = 0; i < 4; ++i) base[i] = Elt<T>::round(gl * p[i] * ((w[i] - s) + zc * lse));
  }
  float dz = 0.f;
  if (d_gates != nullptr) {
    float zmax = z;
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) zmax = fmaxf(zmax, __shfl_xor(zmax, off, MI_WAVE));
    float p = lane < k ? expf(z - zmax) : 0.f;
    p /= wave_sum_f32(p);
    const float dot = wave_sum_f32(p * g);
    dz = Elt<T>::round(p * (g - dot));
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int e = lane + 64 * i;
    if (64 * i >= E) break;
    float val = base[i];
    if (d_gates != nullptr) {
      for (int j = 0; j < k; ++j) {
        const int ej = __shfl(e_j, j, MI_WAVE);
        const float dzj = __shfl(dz, j, MI_WAVE);
        if (ej == e) val = grad != nullptr ? Elt<T>::round(dzj + base[i]) : dzj;
      }
    }
    if (e < E) Elt<T>::store(d_logits + (size_t)t * E + e, val);
  }
}

int mi_router_dlogits_aux(const void* logits, const int32_t* idx, const void* d_gates, const float* loss_w, const void* grad,
                          void* d_logits, int T, int E, int k, int dtype, hipStream_t s) {
  const dim3 grid(mi_ceil_div(T, 4)), block(256);
  if (E > AUX_MAX_E || k > 64) return MI_MOE_EUNSUPPORTED;
  if (dtype == MI_MOE_BF16)
    hipLaunchKernelGGL((router_dlogits_aux_kernel<bf16_t>), grid, block, 0, s, static_cast<const bf16_t*>(logits), idx,
                       static_cast<const bf16_t*>(d_gates), loss_w, static_cast<const bf16_t*>(grad), static_cast<bf16_t*>(d_logits), T, E, k);
  else if (dtype == MI_MOE_F16)
    hipLaunchKernelGGL((router_dlogits_aux_kernel<f16_t>), grid, block, 0, s, static_cast<const f16_t*>(logits), idx,
                       static_cast<const f16_t*>(d_gates), loss_w, static_cast<const f16_t*>(grad), static_cast<f16_t*>(d_logits), T, E, k);
  else return MI_MOE_EDTYPE;
  return mi_launch_status();
}
