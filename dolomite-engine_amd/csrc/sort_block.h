// Block-level pieces of the stable counting sort of expert ids (see routing.hip), shared with the small-batch router,
// whose last workgroup sorts the ids it has just written.
#pragma once

#include "common.h"

#define SORT_THREADS 256
#define SORT_WAVES (SORT_THREADS / 64)
#define SORT_CHUNK 2048
#define SORT_SMALL_CHUNK 512
#define SORT_MAX_E 1024

__device__ __forceinline__ int wave_incl_scan_i32(int v, int lane) {
#pragma unroll
  for (int off = 1; off < 64; off <<= 1) {
    int o = __shfl_up(v, off, MI_WAVE);
    if (lane >= off) v += o;
  }
  return v;
}

// sum over the lanes of a wave, in scalar registers
__device__ __forceinline__ int wave_total_i32(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr 1, 2, 4, 8: rows of 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15: into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31: into rows 2 and 3
  return __builtin_amdgcn_readlane(v, 63);
}

// One step of the stable scatter: a wave's 64 slots from `slot - lane` on, lane l holding slot's expert e (ok: a valid one).
// mybase[e]: output position of the wave's next slot of expert e.
__device__ __forceinline__ void sort_scatter_step(int slot, int e, bool ok, int nbits, int* mybase,
                                                  int32_t* __restrict__ sorted_expert,
                                                  int32_t* __restrict__ sorted_scattered) {
  const int lane = threadIdx.x & 63;
  if (!ok) e = 0;
  uint64_t peers = __ballot(ok);
  for (int b = 0; b < nbits; ++b) {
    uint64_t bal = __ballot((e >> b) & 1);
    peers &= ((e >> b) & 1) ? bal : ~bal;
  }
  if (ok) {
    const uint64_t below = peers & ((1ull << lane) - 1ull);
    const int rank = __popcll(below);
    const int pos = mybase[e] + rank;
    sorted_expert[pos] = e;
    sorted_scattered[pos] = slot;
    // every lane of the group has read mybase[e] (one LDS instruction, wave-wide) before the
    // group's first lane bumps it for the next step
    if (below == 0ull) mybase[e] += __popcll(peers);
  }
}

// Stable scatter of one chunk [chunk_begin, chunk_end).  wbase[w * E + e] must hold, on entry, the
// output position of the first slot of expert e seen by wave w.
__device__ __forceinline__ void sort_scatter_chunk(const int32_t* __restrict__ ids, int chunk_begin, int chunk_end,
                                                   int per_wave, int E, int nbits, int* wbase,
                                                   int32_t* __restrict__ sorted_expert,
                                                   int32_t* __restrict__ sorted_scattered) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  int* mybase = wbase + wave * E;
  const int begin = chunk_begin + wave * per_wave;
  int end = begin + per_wave;
  if (end > chunk_end) end = chunk_end;
  for (int s0 = begin; s0 < end; s0 += 64) {
    const int slot = s0 + lane;
    const bool valid = slot < end;
    const int e = valid ? ids[slot] : 0;
    sort_scatter_step(slot, e, valid && (unsigned)e < (unsigned)E, nbits, mybase, sorted_expert, sorted_scattered);
  }
}

// Per-wave histograms of a chunk into wcnt[w * E + e] (LDS, pre-zeroed).
__device__ __forceinline__ void sort_wave_hist(const int32_t* __restrict__ ids, int chunk_begin, int chunk_end,
                                               int per_wave, int E, int* wcnt) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int begin = chunk_begin + wave * per_wave;
  int end = begin + per_wave;
  if (end > chunk_end) end = chunk_end;
  for (int s = begin + lane; s < end; s += 64) {
    int e = ids[s];
    if ((unsigned)e < (unsigned)E) atomicAdd(&wcnt[wave * E + e], 1);
  }
}

// Whole problem in one block of WAVES waves, at most 512 ids a wave: histogram, expert scan and scatter without touching a
// workspace.  `smem`: (WAVES + 1) * E ints of LDS.  It is a chain of latencies, so a wave's ids are loaded at once and
// kept for both passes, and sixteen waves share them from SORT_FEW_IDS ids on (four waves that loaded the ids step by
// step, twice: 12.5 us for 2840 ids of 40 experts, now 5.6).
#define SORT_ID_STEPS 8
template <int WAVES>
__device__ __forceinline__ void sort_single_block(const int32_t* __restrict__ ids, int L, int E, int nbits,
                                                  int32_t* __restrict__ sorted_expert,
                                                  int32_t* __restrict__ sorted_scattered,
                                                  int32_t* __restrict__ expert_offsets, int* smem) {
  constexpr int THREADS = WAVES * 64;
  int* wcnt = smem;
  int* totals = smem + WAVES * E;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int per_wave = mi_ceil_div_dev(mi_ceil_div_dev(L, WAVES), 64) * 64;
  int id[SORT_ID_STEPS];
#pragma unroll
  for (int j = 0; j < SORT_ID_STEPS; ++j) {
    const int slot = wave * per_wave + j * 64 + lane;
    id[j] = j * 64 < per_wave && slot < L ? ids[slot] : -1;
  }
  for (int i = threadIdx.x; i < WAVES * E; i += THREADS) wcnt[i] = 0;
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SORT_ID_STEPS; ++j)
    if ((unsigned)id[j] < (unsigned)E) atomicAdd(&wcnt[wave * E + id[j]], 1);
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += THREADS) {
    int t = 0;
#pragma unroll
    for (int w = 0; w < WAVES; ++w) t += wcnt[w * E + e];
    totals[e] = t;
  }
  __syncthreads();
  if (wave == 0) {
    int carry = 0;
    for (int e0 = 0; e0 < E; e0 += 64) {
      int e = e0 + lane;
      int v = e < E ? totals[e] : 0;
      int inc = wave_incl_scan_i32(v, lane);
      if (e < E) {
        expert_offsets[e] = carry + inc;
        totals[e] = carry + inc - v;  // exclusive base
      }
      carry += __shfl(inc, 63, MI_WAVE);
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < E; e += THREADS) {
    int run = totals[e];
#pragma unroll
    for (int w = 0; w < WAVES; ++w) {
      int c = wcnt[w * E + e];
      wcnt[w * E + e] = run;
      run += c;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < SORT_ID_STEPS; ++j)
    if (j * 64 < per_wave)
      sort_scatter_step(wave * per_wave + j * 64 + lane, id[j], (unsigned)id[j] < (unsigned)E, nbits, wcnt + wave * E,
                        sorted_expert, sorted_scattered);
}

#define SORT_MANY_WAVES 16
#define SORT_FEW_IDS 512            // up to here four waves sort
#define SORT_SINGLE_BLOCK_MAX 8192  // SORT_MANY_WAVES * 64 * SORT_ID_STEPS
