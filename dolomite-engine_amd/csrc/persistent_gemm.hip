// Persistent grouped GEMM for large expert loads: one workgroup per CU walks a list of 256 x 256 tiles.
//
//   out[orow(i), :] = in[irow(i), :] @ W[e_i]^T     for every row i of the expert-sorted order
//
// (the scattered_experts op called at lm_engine/hf_models/modeling_utils/mlp_blocks/moe.py:91-101), with the SwiGLU of
// activations/glu.py:42-43 in the epilogue (GLU), with the pre-activation written next to it for training (KEEP), or
// with the weights stored (E, K, N) as both data gradients of the backward need them (WT).
//
// What bounds it and why it looks like this
//   * Four waves, ONE per SIMD, each owning a 128 x 128 piece of the tile: 256 accumulators per lane, the whole AGPR
//     half of the register file.  A K slice of 64 then costs a wave 32 fragment reads for its 128 matrix instructions
//     (eight waves of 64 x 128 need 48 per 128), the LDS is busy for three quarters of the matrix time and not all of
//     it, and the chip -- which runs these kernels against its power limit -- spends the difference on clock.
//   * Operands come to LDS by DMA in whole 128-byte lines (64 values of a row): the same bytes in 64-byte halves
//     doubled the L2 requests and lost 6 % of the rate.  The DMA is spread evenly over the slice, one instruction per
//     eight matrix instructions; in two bursts per slice it costs 5 %, in one burst 12 %: an instruction whose
//     queue is full holds the wave, and with one wave per SIMD that idles the matrix pipe.
//   * The LDS ring has five units of 32 KB -- the rows of one operand for one slice -- which is all of the LDS: while
//     slice k is multiplied, slice k + 1 is complete or landing, the weights of slice k + 2 arrive in the fifth unit, and
//     its activations replace slice k once everybody has read it.  One barrier per slice.  Weights first: they come from
//     memory, activations from a cache, and whoever is requested first has half a slice more time (the other way round:
//     40 experts, 1536 -> 512 SwiGLU, 2048 tokens 75.9 -> 73.4 us, 4096 tokens 109.9 -> 106.9; 32 experts, 512 -> 1024,
//     16384 tokens 147.5 -> 142.8; loads of thousands of rows per expert the same within 1 %).
//   * Fragments are read one half slice ahead into a second register set; every LDS read, DMA instruction and scalar
//     step sits alone between two matrix instructions (a matrix instruction leaves three free issue slots).
//   * The accumulators are addressed by number (mfma_core.h).
//   * A tile boundary has no barrier.  SwiGLU results go from registers to memory: the weight rows are dealt to the matrix
//     instruction so that a lane ends up with eight neighbouring columns of a row (the staging before, per half of a training
//     tile once more, and its waits: 40 experts, 1536 -> 512, 2048 tokens 55.4 -> 53 us, with the pre-activation 63 -> 57.5;
//     32 experts, 1024 -> 512, 16384 tokens 219 -> 214 and 268 -> 255; 32768 tokens, which the stores bound, 690 -> 683 with the
//     pre-activation).  The plain form stages them through the eight 1 KB pieces of the free ring unit that the wave's own DMA
//     fills next.  The stores stay in flight under the next tile's first slice (they are counted, vmcnt retires in issue
//     order).  The tile list of a workgroup is decoded once, a lane per tile.
//   * What a boundary costs (40 experts, 32768 tokens, uneven; without the stores' traffic / without the epilogue): SwiGLU 1536 ->
//     512 629 us (602 / 563), plain 512 -> 1536 396 (338 / 286), pre-activation kept 703 (632 / 535).  Starting the workgroups
//     of an XCD a half or a quarter of a tile apart changes nothing: they are out of step by themselves.
// Measured (8192 x 8192 x 8192, one expert): the loop runs at 0.94 of the matrix pipe's cycles without DMA; the form it
// replaces -- eight waves in two groups that alternated between a memory and a matrix phase, 64-byte rows -- reached
// 0.80 with DMA.
#include "persistent_body.h"

// Splitting the last round along K.  A workgroup's tiles all take the same time, so when the tiles of an XCD do not
// fill its last round, the workgroups without a tile wait for one tile time.  With a workspace, the `rem` tiles of
// that round are cut into `parts` = min(slots / rem, PERSIST_SPLIT_MAX) ranges of K slices, one per workgroup; a
// part writes its fp32 accumulators to the workspace instead of running the epilogue, and a second, small launch
// (grouped_gemm_split_finish_kernel) adds the parts of every split tile in part order and runs the epilogue, so
// the result does not depend on timing.  A round is only split if that shortens it by at least
// PERSIST_SPLIT_MIN_SAVED (persistent_tiles.h) slices, for the partial tiles' trip through memory and the second launch.
// Whole / cut, us: 8 experts, 14336 -> 4096, 2048 tokens 562 / 413, 4096 tokens 841 / 742, 8192 tokens 1443 / 1356; 16 experts,
// 8192 -> 2048, 2500 tokens 354 / 304; 8 experts, 5632 -> 1024, 8192 tokens 220 / 174; 5120 -> 1024 SwiGLU, 4096 tokens 204 / 158.
// Where the plan then cuts nothing the second launch is 2 - 4 us (5120 -> 2048, 2048 tokens 112 / 115).  With the line at 16 slices
// contractions of 2048 and 4096 are cut as well: 4096 -> 14336, 1024 tokens 575 -> 540, 4096 tokens 1442 -> 1451, 6000 tokens 1984 ->
// 1995; 2048 -> 5120, 2048 and 3000 tokens 182 -> 187 and 204 -> 209.
// whether a contraction of length K can be shortened by PERSIST_SPLIT_MIN_SAVED slices at all (launch_persistent
// applies the same rule, plus one on the grid)
static bool persistent_may_split(int K) {
  const int nk = K / PG_BK;
  return nk - nk / PERSIST_SPLIT_MAX >= PERSIST_SPLIT_MIN_SAVED;
}

template <typename T, bool GLU, bool WT, bool KEEP>
__global__ __launch_bounds__(256, 1) void grouped_gemm_persistent_kernel(GemmArgs a) {
  pg_fetch_arguments(a);
  const PgRows experts = pg_rows(a.expert_offsets, a.L, a.E);
  if constexpr (!GLU) {
    persistent_body<T, GLU, WT, KEEP, true>(a, experts);
  } else if constexpr (KEEP) {
    persistent_body<T, GLU, WT, KEEP, false>(a, experts);  // (the backward reads both again)
  } else {
    if (a.out_nt) persistent_body<T, GLU, WT, KEEP, true>(a, experts);
    else persistent_body<T, GLU, WT, KEEP, false>(a, experts);
  }
}

// The tiles the persistent kernel cut along K (see PERSIST_SPLIT_MAX): one workgroup per (XCD, tile of its last round)
// and quarter of the accumulator blocks recomputes the same plan, adds the tile's partial accumulators in part order
// and writes them the way the persistent kernel's epilogue does (same arithmetic, same rounding; thread t holds what
// thread t of a part held).  Workgroups whose tile does not exist or was not split return at once.
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void grouped_gemm_split_finish_kernel(GemmArgs a, int nslot, int by_load_form) {
  constexpr int BM = 256, BN = GLU ? 128 : 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 1, wn = wave >> 1;
  PgRows experts = pg_rows(a.expert_offsets, a.L, a.E);
  if (by_load_form >= 0 && pg_form_by_load(a, experts, by_load_form, 8 * nslot) != 0) return;
  PgTable tb;
  pg_table<BM>(experts, a.E, tb);
  // contiguous: workgroup b adds up tile b / 8 of XCD b % 8's last round; interleaved: tile b of the chip's last round
  const bool interleave = (a.remap & PERSIST_REMAP_INTERLEAVE) != 0;
  const int xcd = interleave ? 0 : (int)(blockIdx.x & 7), j = interleave ? (int)blockIdx.x : (int)(blockIdx.x >> 3);
  const SplitPlan sp = persist_split_plan(tb.total * a.n_tiles, xcd, 0, nslot, (a.K + PG_BK - 1) / PG_BK, true, interleave);
  if (sp.parts == 1 || j >= sp.rem) return;
  const PgTile t = pg_locate<BM>(tb, a.E, a.n_tiles, sp.rem_base + j);

  constexpr int MBS = 2;  // row blocks of this workgroup: 2 q, 2 q + 1
  const int q = blockIdx.y;
  const f32x4* part = static_cast<const f32x4*>(a.ws) + ((size_t)sp.ws_base + (size_t)j * sp.parts) * (64 * 256) +
                      q * (MBS * 8 * 256) + tid;
  f32x4 sum[MBS * 8];
#pragma unroll
  for (int b = 0; b < MBS * 8; ++b) sum[b] = __builtin_nontemporal_load(part + b * 256);
  for (int p = 1; p < sp.parts; ++p) {
    part += 64 * 256;
#pragma unroll
    for (int b = 0; b < MBS * 8; ++b) {
      const f32x4 v = __builtin_nontemporal_load(part + b * 256);
#pragma unroll
      for (int c = 0; c < 4; ++c) sum[b][c] += v[c];
    }
  }
  const int frow = lane & 15, fq = lane >> 4;
  T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
  for (int mb = 0; mb < MBS; ++mb) {
    const int row = t.row_begin + wm * 128 + (q * MBS + mb) * 16 + frow;
    if (row >= t.row_end) continue;
    const int orow = a.scatter ? a.sorted_scattered[row] : row;
#pragma unroll
    for (int nb = 0; nb < (GLU ? 4 : 8); ++nb) {
      const int col = t.nt * BN + (GLU ? wn * 64 + 32 * (nb / 2) + 8 * fq + 4 * (nb % 2) : wn * 128 + nb * 16 + fq * 4);
      if (col >= a.N) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float up = sum[mb * 8 + nb][i];
        if (GLU) {
          const float gt = sum[mb * 8 + nb + 4][i];
          v[i] = up * silu_rcp_f32(gt);
        } else {
          v[i] = up;
        }
      }
      const u32x2 p2 = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
      *reinterpret_cast<u32x2*>(out + (size_t)orow * a.N + col) = p2;
    }
  }
}

// ---- host side ----------------------------------------------------------------------------------------------------------------
template <typename T, bool GLU, bool WT, bool KEEP>
static int launch_persistent(GemmArgs a, hipStream_t s) {
  constexpr int BM = 256, BN = GLU ? 128 : 256;
  auto kern = grouped_gemm_persistent_kernel<T, GLU, WT, KEEP>;
  static std::atomic<uint64_t> lds_ok{0};
  int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), PG_LDS, lds_ok);
  if (rc != MI_MOE_OK) return rc;
  int grid = 0;
  if ((rc = persistent_prepare(a, BM, BN, &grid)) != MI_MOE_OK) return rc;
  // no contraction length that a split could shorten by PERSIST_SPLIT_MIN_SAVED slices, or one slot per XCD
  if (!mi_gemm_persistent_splits(a.K) || grid < 16 || a.pre != nullptr) a.ws = nullptr;  // (the finishing launch writes the result only)
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), PG_LDS, s, a);
  if ((rc = mi_launch_status()) != MI_MOE_OK || a.ws == nullptr) return rc;
  return mi_gemm_split_finish(a, std::is_same<T, bf16_t>::value ? MI_MOE_BF16 : MI_MOE_F16, GLU ? PG_SWIGLU : PG_PLAIN, grid / 8, false, s);
}

int mi_gemm_split_finish(const GemmArgs& a, int dtype, int form, int nslot, bool by_load, hipStream_t s) {
  auto kern = form == PG_SWIGLU ? (dtype == MI_MOE_BF16 ? grouped_gemm_split_finish_kernel<bf16_t, true> : grouped_gemm_split_finish_kernel<f16_t, true>)
                                : (dtype == MI_MOE_BF16 ? grouped_gemm_split_finish_kernel<bf16_t, false> : grouped_gemm_split_finish_kernel<f16_t, false>);
  // the tiles that were cut: at most half of the slots of a round that was split hold tiles (rounded up: an odd
  // number of slots per XCD)
  hipLaunchKernelGGL(kern, dim3(8u * (unsigned)((nslot + 1) / 2), 4), dim3(256), 0, s, a, nslot, by_load ? form : -1);
  return mi_launch_status();
}

bool mi_gemm_persistent_splits(int K) { return persistent_may_split(K); }

bool mi_gemm_persistent_ok(const GemmArgs& a) {
  return a.K % 8 == 0 && a.N % 8 == 0 && a.E <= PERSIST_MAX_E && mi_aligned(a.out, 16);
}

int mi_gemm_persistent(const GemmArgs& a, int dtype, int form, hipStream_t s) {
  if (!mi_gemm_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
  if (!(a.remap & PERSIST_REMAP_FIXED)) {
    const int tile = mi_gemm_tiles_of_any_load(a, form);
    if (tile == EVEN_BY_LOAD) return mi_gemm_by_load(a, dtype, form, s);
    if (tile != EVEN_NONE) return mi_gemm_even(a, dtype, form, tile, s);
  }
  if (dtype == MI_MOE_BF16) {
    switch (form) {
      case PG_PLAIN: return launch_persistent<bf16_t, false, false, false>(a, s);
      case PG_SWIGLU: return launch_persistent<bf16_t, true, false, false>(a, s);
      case PG_SWIGLU_KEEP: return launch_persistent<bf16_t, true, false, true>(a, s);
      case PG_WEIGHT_KN: return launch_persistent<bf16_t, false, true, false>(a, s);
    }
  } else if (dtype == MI_MOE_F16) {
    switch (form) {
      case PG_PLAIN: return launch_persistent<f16_t, false, false, false>(a, s);
      case PG_SWIGLU: return launch_persistent<f16_t, true, false, false>(a, s);
      case PG_SWIGLU_KEEP: return launch_persistent<f16_t, true, false, true>(a, s);
      case PG_WEIGHT_KN: return launch_persistent<f16_t, false, true, false>(a, s);
    }
  }
  return MI_MOE_EDTYPE;
}
