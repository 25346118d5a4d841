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
//   * A tile boundary has no barrier: a wave stages its results through the eight 1 KB pieces of the free ring unit
//     that its own DMA fills next.  The stores stay in flight under the next tile's first slice (they are counted,
//     vmcnt retires in issue order).  The tile list of a workgroup is decoded once, a lane per tile.
// Measured (8192 x 8192 x 8192, one expert): the loop runs at 0.94 of the matrix pipe's cycles without DMA; the form it
// replaces -- eight waves in two groups that alternated between a memory and a matrix phase, 64-byte rows -- reached
// 0.80 with DMA.
#include "gemm_common.h"
#include "mfma_core.h"
#include "persistent_tiles.h"


#define PG_BK 64        // K slice: one 128-byte line of a 16-bit row
#define PG_U 32768      // bytes of a ring unit: 256 rows of one operand (WT weights: 64 rows of 256 columns)
#define PG_LDS (5 * PG_U)

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


// NT: results are stored non-temporal
template <typename T, bool GLU, bool WT, bool KEEP, bool NT>
__device__ __forceinline__ void persistent_body(const GemmArgs& a) {
  static_assert(!KEEP || GLU, "the pre-activation belongs to the SwiGLU form");
  static_assert(!WT || !GLU, "transposed-weight form");
  constexpr int BM = 256;
  constexpr int BN = GLU ? 128 : 256;               // output columns per tile
  constexpr int NSTORE = KEEP ? 48 : (GLU ? 16 : 32);  // stores of a wave in the epilogue
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;
  typedef short tr_s16x4 __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) tr_s16x4* tr_ptr_t;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const uint32_t lds0 = (uint32_t)(size_t)(lds_ptr_t)smem_raw;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;          // 128 activation rows, 128 weight rows (SwiGLU: 64 up, 64 gate)
  const int frow = lane & 15, fq = lane >> 4;       // fragment: row frow, k = 8 fq + [0, 8) of the half slice

  // ---- which tiles -----------------------------------------------------------------------------------------------
  PgTable tb;
  pg_table<BM>(a.expert_offsets, a.L, a.E, tb);
  const int total = tb.total * a.n_tiles;
  const int nfull = a.K / PG_BK;                    // whole slices; a partial one is padded with zeros
  int nk = (a.K + PG_BK - 1) / PG_BK;
  if (nk < 2) nk = 2;                               // (the ring wants two: a second slice of zeros)
  const SplitPlan sp = persist_split_plan(total, blockIdx.x & 7, blockIdx.x >> 3, gridDim.x >> 3, nk, a.ws != nullptr,
                                          (a.remap & PERSIST_REMAP_INTERLEAVE) != 0);
  const int my_part = sp.parts > 1 ? sp.lslot / sp.rem : 0, my_rem_tile = sp.rem > 0 ? sp.lslot % sp.rem : 0;
  const int n_items = sp.full_rounds + (sp.lslot < sp.rem * sp.parts ? 1 : 0);
  if (n_items == 0) return;
  // K slices [k0, k1) of item i
  auto item_k = [&](int i, int& k0, int& k1) {
    const bool part = i == sp.full_rounds && sp.parts > 1;
    k0 = part ? my_part * nk / sp.parts : 0;
    k1 = part ? (my_part + 1) * nk / sp.parts : nk;
  };
  PgTile list;                                      // lane l: item (64-item block) + l
  auto fetch = [&](int i) -> PgTile {               // called with i = 0, 1, 2, ...; past the last item: the last item
    if (i >= n_items) i = n_items - 1;
    else if ((i & 63) == 0) {
      const int it = i + lane;
      const int tile = it < sp.full_rounds ? sp.base + it * sp.stride : sp.rem_base + my_rem_tile;
      list = pg_locate<BM>(tb, a.E, a.n_tiles, it < n_items ? tile : 0);
    }
    const int l = i & 63;
    PgTile t;
    t.expert = __builtin_amdgcn_readlane(list.expert, l);
    t.nt = __builtin_amdgcn_readlane(list.nt, l);
    t.row_begin = __builtin_amdgcn_readlane(list.row_begin, l);
    t.row_end = __builtin_amdgcn_readlane(list.row_end, l);
    return t;
  };

  // ---- DMA sources ---------------------------------------------------------------------------------------------------
  // Unit image: row r of 128 bytes keeps its 16-byte chunks at slots chunk ^ ((r >> 1) & 7), which serves the 16 rows x
  // 4 chunks of a fragment without bank conflicts.  Instruction j of a wave fills rows 8 (4 j + wave) .. + 8 in lane
  // order, so the swizzle is applied on the global side: lane l fetches chunk (l % 8) ^ ((r >> 1) & 7).
  const int drow = wave * 8 + (lane >> 3);          // row of instruction 0 (instruction j: + 32 j)
  const int lchunk = (lane & 7) ^ ((wave & 1) * 4 + (lane >> 4));
  const uint32_t row_bytes = (uint32_t)a.K * 2u;
  const u32x4 xsrd = pg_srd(a.in, (uint64_t)(a.gather ? a.L / a.kdiv : a.L) * row_bytes);
  const uint64_t w_bytes = (uint64_t)a.E * (GLU ? 2 : 1) * a.N * row_bytes;
  auto make_wsrd = [&](const PgTile& t) -> u32x4 {
    const uint64_t o = ((uint64_t)t.expert * (GLU ? 2 : 1) * a.N * a.K + (uint64_t)t.nt * BN * (WT ? 1 : a.K)) * 2u;
    return pg_srd(static_cast<const unsigned char*>(a.w) + o, w_bytes - o);
  };
  // sorted-order row index of the activation rows a lane fetches (clamped into the tile's expert), and the byte offsets
  // they give; rows past the expert's end lie past the buffer: zeros, no traffic, and multipliers at rest
  auto load_rows = [&](const PgTile& t, int (&raw)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = t.row_begin + drow + 32 * j;
      raw[j] = r < t.row_end ? r : t.row_end - 1;
    }
    if (a.gather) {
#pragma unroll
      for (int j = 0; j < 8; ++j) raw[j] = a.sorted_scattered[raw[j]];
    }
  };
  auto make_xoff = [&](const PgTile& t, const int (&raw)[8], uint32_t (&off)[8]) {
    // (top-k is a power of two in most configurations: a shift instead of a division)
    const int sh = !a.gather ? 0 : a.kshift;
    if (sh >= 0) {
#pragma unroll
      for (int j = 0; j < 8; ++j) off[j] = (uint32_t)(raw[j] >> sh) * row_bytes + lchunk * 16u;
    } else {
#pragma unroll
      for (int j = 0; j < 8; ++j) off[j] = (uint32_t)(raw[j] / a.kdiv) * row_bytes + lchunk * 16u;
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = t.row_begin + drow + 32 * j < t.row_end ? off[j] : PG_OOB;
  };
  // Weight rows are at fixed distances (rows past N are another matrix's, or past the buffer: never stored).
  // WT: instruction j fills rows 8 j + 2 wave + lane / 32 of the slice; 16-byte piece l % 32 of row r holds the logical
  // piece whose 32-byte group is (piece / 2) ^ (r % 4 | (r / 8 % 4) << 2): the swizzle the transposing reads expect.
  uint32_t woff[8];
  auto make_woff = [&]() {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      if constexpr (WT) {
        const int r = 8 * j + 2 * wave + (lane >> 5), f = (r & 3) | ((j & 3) << 2);
        woff[j] = ((uint32_t)r * a.N + ((((lane & 31) >> 1) ^ f) << 4) + (lane & 1) * 8) * 2u;
      } else {
        const int r = GLU ? 32 * (j & 3) + (j >= 4 ? a.N : 0) : 32 * j;
        woff[j] = (uint32_t)(r + drow) * row_bytes + lchunk * 16u;
      }
    }
  };
  const uint32_t w_step = WT ? (uint32_t)a.N * (2u * PG_BK) : 2u * PG_BK;  // bytes from slice to slice
  // a slice with fewer than 64 values: the lanes past them fetch zeros
  auto mask_x = [&](uint32_t (&off)[8], int k) {
    const bool gone = lchunk * 8 >= a.K - k * PG_BK;
#pragma unroll
    for (int j = 0; j < 8; ++j) off[j] = gone ? PG_OOB : off[j];
  };
  auto mask_w = [&](int k) {
    if constexpr (WT) {
#pragma unroll
      for (int j = 0; j < 8; ++j) woff[j] = 8 * j + 2 * wave + (lane >> 5) >= a.K - k * PG_BK ? PG_OOB : woff[j];
    } else {
      mask_x(woff, k);
    }
  };

  // ---- fragment reads ------------------------------------------------------------------------------------------------
  const uint32_t fswz = (frow >> 1) & 7;
  const uint32_t fx = (wm * 128 + frow) * 128, fw = (wn * (GLU ? 64 : 128) + frow) * 128;
  const uint32_t fc0 = lds0 + ((fq ^ fswz) * 16), fc1 = lds0 + (((fq + 4) ^ fswz) * 16);
  // WT: ds_read_b64_tr_b16 transposes 4 rows x 16 columns across 16 lanes: lane i of the group supplies the address of
  // (row i / 4, columns 4 (i % 4) ..) and receives column i of the four rows.  Lane group q reads rows 8q .. 8q + 3 and,
  // 2 KiB further, 8q + 4 .. 8q + 7: together the 8 contraction values the matrix instruction wants.
  const uint32_t trb = (8 * fq + (frow >> 2)) * 512 + ((((frow >> 2) | (fq << 2))) << 5) + (frow & 3) * 8;
  u32x4 wf[2][8], xf[2][8];
  auto read_w = [&](uint32_t base, int ks, int nb) -> u32x4 {
    if constexpr (WT) {
      const uint32_t ad = base + (trb ^ ((uint32_t)(wn * 8 + nb) << 5));
      const tr_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(size_t)(ad + ks * 16384));
      const tr_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(size_t)(ad + ks * 16384 + 2048));
      return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      typedef __attribute__((address_space(3))) const u32x4* p;
      return *(p)(size_t)(base + (GLU && nb >= 4 ? 16384 + (nb - 4) * 2048 : nb * 2048));
    }
  };
  auto read_x = [&](uint32_t base, int mb) -> u32x4 {
    typedef __attribute__((address_space(3))) const u32x4* p;
    return *(p)(size_t)(base + mb * 2048);
  };

  // ---- ring and source state ------------------------------------------------------------------------------------------
  // Slots of X_k, W_k, X_k+1, W_k+1 and the free one (W_k+2; then X_k+2 goes to the slot of X_k); X = activations.
  uint32_t p0 = 0, p1 = PG_U, p2 = 2 * PG_U, p3 = 3 * PG_U, p4 = 4 * PG_U;
  uint32_t xoff[8], xoff_n[8];
  u32x4 wsrd, wsrd_n;
  int kx, kx_end, kx_ev, kw, kw_end, kw_ev;         // next slice of the source tile, its end, the next one with an event
  int k0_n, k1_n;                                   // slices of the next item
  auto event_of = [&](int end) { return nfull < end ? nfull : end; };
  auto x_event = [&]() {
    if (kx == kx_end) {
#pragma unroll
      for (int j = 0; j < 8; ++j) xoff[j] = xoff_n[j];
      kx = k0_n;
      kx_end = k1_n;
    }
    if (kx >= nfull) mask_x(xoff, kx);
    kx_ev = event_of(kx_end);
  };
  auto w_event = [&]() {
    if (kw == kw_end) {
      wsrd = wsrd_n;
      if (nfull != nk) make_woff();
      kw = k0_n;
      kw_end = k1_n;
    }
    if (kw >= nfull) mask_w(kw);
    kw_ev = event_of(kw_end);
  };

  // One half slice: 64 matrix instructions.  B = 0: values [0, 32) of slice k out of the registers read before, while
  // values [32, 64) are read and W_k+2 is fetched; B = 1: those, while slice k + 1 is read and X_k+2 is fetched.
  // `hook(m)` runs after matrix instruction m.
  const uint32_t dma0 = lds0 + wave * 1024;
  uint32_t rw, rx;                                  // addresses of the next half's fragments
  auto half = [&](auto btag, auto ftag, uint32_t dst, auto hook) {
    constexpr int B = decltype(btag)::value;
    constexpr bool FIRST = decltype(ftag)::value;
    const uint32_t soff = B ? (uint32_t)kx * (2u * PG_BK) : (uint32_t)kw * w_step;
    pg_own_agprs();
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      const int nb = m & 7, mb = m >> 3;
      if constexpr (FIRST) pg_mfma_first<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
      else pg_mfma<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
      if (m % 2 == 0 && m < 32) {
        const int q = m / 2;
        PG_SCHED();
        if (q < 8) wf[B ^ 1][q] = read_w(rw, B ^ 1, q);
        else xf[B ^ 1][q - 8] = read_x(rx, q - 8);
        PG_SCHED();
      }
      if (m % 8 == 1) {
        PG_SCHED();
        pg_dma_dst(dst, m / 8 * 4096);
        PG_SCHED();
      }
      if (m % 8 == 3) {
        PG_SCHED();
        pg_dma(B ? xoff[m / 8] : woff[m / 8], B ? xsrd : wsrd, soff);
        PG_SCHED();
      }
      hook(m);
    }
  };
  auto read_bases = [&](int ks, uint32_t ps_w, uint32_t ps_x) {
    rw = WT ? lds0 + ps_w : (ks ? fc1 : fc0) + fw + ps_w;
    rx = (ks ? fc1 : fc0) + fx + ps_x;
    asm volatile("" : "+v"(rx));
    if constexpr (!WT) asm volatile("" : "+v"(rw));
  };
  // stores_after_dma: the epilogue of a tile lies between the DMA this slice waits for and now
  auto step = [&](auto ftag, bool stores_after_dma) {
    if (kw >= kw_ev) w_event();
    half(std::integral_constant<int, 0>{}, ftag, dma0 + p4, [&](int m) {
      if (m == 62) {
        PG_SCHED();
        ++kw;
        read_bases(0, p3, p2);
        PG_SCHED();
      }
    });
    // slice k + 1 has landed (W_k+2 stays in flight); slice k is in everybody's registers
    if (decltype(ftag)::value && stores_after_dma) __builtin_amdgcn_s_waitcnt(pg_wait(8 + NSTORE, 0));
    else __builtin_amdgcn_s_waitcnt(pg_wait(8, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    PG_SCHED();
    if (kx >= kx_ev) x_event();
    half(std::integral_constant<int, 1>{}, std::false_type{}, dma0 + p0, [&](int m) {
      if (m == 62) ++kx;
      if (m == 60) {
        PG_SCHED();
        const uint32_t t0 = p0, t1 = p1;
        p0 = p2;
        p1 = p3;
        p2 = t0;
        p3 = p4;
        p4 = t1;
        asm volatile("" : "+s"(p0), "+s"(p1), "+s"(p2), "+s"(p3), "+s"(p4));
        PG_SCHED();
      }
      if (m == 62) {
        PG_SCHED();
        read_bases(1, p1, p0);
        PG_SCHED();
      }
    });
  };

  // ---- epilogue: accumulators -> (SwiGLU) -> the wave's pieces of the free ring unit -> 16-byte stores ------------------
  // Plain: four passes of 32 rows x 128 columns (256-byte rows, 4 to a piece); SwiGLU: two of 64 rows x 64 columns.
  // Chunk c of scratch row r lies at slot c ^ (r % 16) (SwiGLU: c ^ (r / 2 % 8)): writes and reads free of conflicts,
  // and the read-back is linear in the lane.
  T* __restrict__ out = static_cast<T*>(a.out);
  constexpr int SB = GLU ? 128 : 256;               // bytes of a scratch row
  constexpr int RPP = 1024 / SB;                    // scratch rows per piece and per store instruction
  constexpr int PASS_ROWS = 8 * RPP, NPASS = 128 / PASS_ROWS, MBP = PASS_ROWS / 16, NBO = GLU ? 4 : 8;
  const uint32_t scr_swz = GLU ? (frow >> 1) & 7 : frow;
  const uint32_t scr_w = (frow / RPP) * 4096 + (frow % RPP) * SB + (((fq >> 1) ^ scr_swz) * 16) + (fq & 1) * 8;
  const int srow = lane / (SB / 16), sslot = lane % (SB / 16);
  const int scc0 = GLU ? sslot ^ ((srow >> 1) & 7) : sslot ^ (srow & 15);  // chunk of store 0; store it: ^ 4 (it % ..)
  int orow_lo, orow_hi;                             // output rows of the wave's rows lane and 64 + lane
  auto load_out_rows = [&](const PgTile& t, int& lo, int& hi) {
    const int r0 = t.row_begin + wm * 128 + lane;
    lo = r0;
    hi = r0 + 64;
    if (a.scatter) {
      lo = a.sorted_scattered[lo < t.row_end ? lo : t.row_end - 1];
      hi = a.sorted_scattered[hi < t.row_end ? hi : t.row_end - 1];
    }
  };
  // WHAT: 0 the kernel's result (SwiGLU: up * silu(gate)); 1 / 2 (KEEP): the up / the gate half of h, into a.pre.  KEEP
  // forms the result from the ROUNDED halves, as the separate activation kernel forms it from the stored h.
  // Every tile issues the same number of stores on one path; what does not exist is a lane past the buffer.  With a branch for
  // edge tiles the compiler, which counts stores along the shortest way it can construct, waited for all of them wherever it
  // needed the next tile's rows, and again in the next tile's first slice: 40 experts, 512 -> 1536, 32768 tokens 401 -> 390 us,
  // 32 experts, 512 -> 1024, 16384 tokens 142 -> 139, 1536 -> 512 SwiGLU, 32768 tokens 613 -> 608.
  // WHAT 0 writes the rows [row0, row0 + out_window) of the output: all of them, unless it has more than 4 GiB.
  auto epilogue_as = [&](auto what_tag, const PgTile& t, uint32_t row0) __attribute__((always_inline)) {
    constexpr int WHAT = decltype(what_tag)::value;
    typedef __attribute__((address_space(3))) u32x2* wp_t;
    typedef __attribute__((address_space(3))) const u32x4* rp_t;
    const uint32_t ld = (WHAT == 0 ? a.N : 2 * a.N) * 2u;
    // (rows of the pre-activation are the sorted order's: addressed from the tile's first, as the whole can exceed 4 GiB)
    const int r0 = wm * 128 + lane, rows = t.row_end - t.row_begin;
    const uint32_t window = WHAT == 0 ? a.out_window : (uint32_t)rows, left = WHAT == 0 ? a.L - row0 : (uint32_t)rows;
    unsigned char* dst = WHAT == 0 ? reinterpret_cast<unsigned char*>(out) + (uint64_t)row0 * ld
                                   : static_cast<unsigned char*>(a.pre) + (uint64_t)t.row_begin * ld;
    const auto srd = __builtin_amdgcn_make_buffer_rsrc(dst, (short)0, (int)((left < window ? left : window) * ld), 0x00020000);
    const uint32_t s0 = dma0 + p4;
    const int col0 = t.nt * BN + wn * (GLU ? 64 : 128);
    // byte offsets of the wave's rows lane and 64 + lane, and of the lane's columns in store it (% CP); saturating sums keep what
    // does not exist past the buffer
    constexpr int CP = GLU ? 2 : 4;
    const uint32_t lo = WHAT == 0 ? (uint32_t)orow_lo - row0 : r0, hi = WHAT == 0 ? (uint32_t)orow_hi - row0 : r0 + 64;
    const uint32_t rlo = r0 < rows && lo < window ? lo * ld : PG_OOB, rhi = r0 + 64 < rows && hi < window ? hi * ld : PG_OOB;
    uint32_t coff[CP];
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int col = col0 + (scc0 ^ (4 * c)) * 8;
      coff[c] = col < a.N ? (uint32_t)((WHAT == 2 ? a.N : 0) + col) * 2u : PG_OOB;
    }
#pragma unroll
    for (int p = 0; p < NPASS; ++p) {
#pragma unroll
      for (int mbp = 0; mbp < MBP; ++mbp)
#pragma unroll
        for (int nb = 0; nb < NBO; ++nb) {
          const int blk = (p * MBP + mbp) * 8 + nb;
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            if (WHAT == 1) {
              v[i] = pg_acc(blk * 4 + i);
            } else if (WHAT == 2) {
              v[i] = pg_acc((blk + 4) * 4 + i);
            } else if (GLU) {
              float up = pg_acc(blk * 4 + i), gt = pg_acc((blk + 4) * 4 + i);
              if (KEEP) {
                up = Elt<T>::round(up);
                gt = Elt<T>::round(gt);
              }
              v[i] = up * silu_rcp_f32(gt);
            } else {
              v[i] = pg_acc(blk * 4 + i);
            }
          }
          *(wp_t)(size_t)(s0 + (scr_w ^ (nb * 32)) + mbp * (16 / RPP) * 4096) =
              (u32x2){pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        }
      pg_own_agprs();
      // (four at a time: one LDS latency for all of them)
#pragma unroll
      for (int it0 = 0; it0 < 8; it0 += 4) {
        u32x4 val[4];
        uint32_t roff[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = p * PASS_ROWS + (it0 + j) * RPP;  // + srow: row of the wave's 128
          val[j] = *(rp_t)(size_t)(s0 + (it0 + j) * 4096 + lane * 16);
          roff[j] = (uint32_t)__builtin_amdgcn_ds_bpermute(((r & 63) + srow) * 4, (int)(r < 64 ? rlo : rhi));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(val[j], srd, (int)__builtin_elementwise_add_sat(roff[j], coff[(it0 + j) % CP]), 0, NT ? 2 : 0);
      }
      pg_own_agprs();
    }
  };
  auto epilogue = [&](const PgTile& t) __attribute__((always_inline)) {
    uint32_t row0 = 0;
    do {
      epilogue_as(std::integral_constant<int, 0>{}, t, row0);
      row0 += a.out_window;
    } while (row0 < (uint32_t)a.L);
    if constexpr (KEEP) {
      // both halves of the pre-activation next to the activation
      epilogue_as(std::integral_constant<int, 1>{}, t, 0);
      epilogue_as(std::integral_constant<int, 2>{}, t, 0);
    }
  };
  // a part of a split tile: accumulators -> workspace, block b of thread t at [b][t]
  auto store_part = [&]() {
    f32x4* base = static_cast<f32x4*>(a.ws) +
                  ((size_t)sp.ws_base + (size_t)my_rem_tile * sp.parts + my_part) * (64 * 256) + threadIdx.x;
#pragma unroll
    for (int b = 0; b < 64; ++b) {
      if (b % 8 == 0) {
        pg_own_agprs();
        asm volatile("" : "+v"(base));              // (or the 64 addresses are kept in registers from the first tile on)
      }
      const f32x4 v = {pg_acc(4 * b), pg_acc(4 * b + 1), pg_acc(4 * b + 2), pg_acc(4 * b + 3)};
      base[b * 256] = v;
    }
  };

  // ---- prologue -----------------------------------------------------------------------------------------------------------
  PgTile cur = fetch(0), nxt = fetch(1);
  int k0, k1;
  item_k(0, k0, k1);
  {
    int raw[8], raw_n[8];
    load_rows(cur, raw);
    load_rows(nxt, raw_n);
    load_out_rows(cur, orow_lo, orow_hi);
    make_xoff(cur, raw, xoff);
    make_xoff(nxt, raw_n, xoff_n);
  }
  make_woff();
  wsrd = make_wsrd(cur);
  wsrd_n = make_wsrd(nxt);
  item_k(n_items > 1 ? 1 : 0, k0_n, k1_n);
  asm volatile("" : "+v"(orow_lo), "+v"(orow_hi));
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));
  kx = kw = k0;
  kx_end = kw_end = k1;
  kx_ev = kw_ev = event_of(k1);
#pragma unroll
  for (int s = 0; s < 2; ++s) {
    if (kx >= nfull) mask_x(xoff, kx);
    if (kw >= nfull) mask_w(kw);
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      pg_dma_dst(dma0 + (s ? p2 : p0), j * 4096);
      asm volatile("s_nop 0");
      pg_dma(xoff[j], xsrd, (uint32_t)kx * (2u * PG_BK));
    }
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      pg_dma_dst(dma0 + (s ? p3 : p1), j * 4096);
      asm volatile("s_nop 0");
      pg_dma(woff[j], wsrd, (uint32_t)kw * w_step);
    }
    ++kx;
    ++kw;
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(16, 0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_bases(0, p1, p0);
#pragma unroll
  for (int i = 0; i < 8; ++i) wf[0][i] = read_w(rw, 0, i);
#pragma unroll
  for (int i = 0; i < 8; ++i) xf[0][i] = read_x(rx, i);
  read_bases(1, p1, p0);

  // ---- tile loop ------------------------------------------------------------------------------------------------------------
  bool stores_pending = false;
  for (int i = 0;; ++i) {
    step(std::true_type{}, stores_pending);
    for (int k = k0 + 1; k < k1; ++k) step(std::false_type{}, false);
    pg_acc_settle();
    if (k1 - k0 != nk) {
      // a part of a split tile, always a workgroup's last item: the finishing launch adds the parts up
      store_part();
      break;
    }
    // rows of the tile after next, and where the next tile's results go: requested here, taken after the epilogue
    const PgTile after = fetch(i + 2);
    int raw[8], lo_n, hi_n;
    load_rows(after, raw);
    load_out_rows(nxt, lo_n, hi_n);
    epilogue(cur);
    // (the waits for the loads above belong here: they count the epilogue's stores, which stay in flight)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(raw[j]));
    asm volatile("" : "+v"(lo_n), "+v"(hi_n));
    if (i + 1 >= n_items) break;
    stores_pending = true;
    make_xoff(after, raw, xoff_n);
    wsrd_n = make_wsrd(after);
    orow_lo = lo_n;
    orow_hi = hi_n;
    k0 = k0_n;
    k1 = k1_n;
    if (i + 2 < n_items) item_k(i + 2, k0_n, k1_n);  // (else: surplus DMA re-reads the last item's first slices)
    cur = nxt;
    nxt = after;
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(xoff_n[j]));
    asm volatile("" : "+v"(orow_lo), "+v"(orow_hi));
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));  // surplus DMA must not outlive the workgroup's LDS
}

template <typename T, bool GLU, bool WT, bool KEEP>
__global__ __launch_bounds__(256, 1) void grouped_gemm_persistent_kernel(GemmArgs a) {
  if constexpr (!GLU) {
    persistent_body<T, GLU, WT, KEEP, true>(a);
  } else if constexpr (KEEP) {
    persistent_body<T, GLU, WT, KEEP, false>(a);    // (the backward reads both again)
  } else {
    if (a.out_nt) persistent_body<T, GLU, WT, KEEP, true>(a);
    else persistent_body<T, GLU, WT, KEEP, false>(a);
  }
}

// The tiles the persistent kernel cut along K (see PERSIST_SPLIT_MAX): one workgroup per (XCD, tile of its last round)
// and quarter of the accumulator blocks recomputes the same plan, adds the tile's partial accumulators in part order
// and writes them the way the persistent kernel's epilogue does (same arithmetic, same rounding; thread t holds what
// thread t of a part held).  Workgroups whose tile does not exist or was not split return at once.
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void grouped_gemm_split_finish_kernel(GemmArgs a, int nslot) {
  constexpr int BM = 256, BN = GLU ? 128 : 256;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, wm = wave & 1, wn = wave >> 1;
  PgTable tb;
  pg_table<BM>(a.expert_offsets, a.L, a.E, tb);
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
      const int col = t.nt * BN + wn * (GLU ? 64 : 128) + nb * 16 + fq * 4;
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
  a.n_tiles = mi_ceil_div(a.N, BN);
  a.out_window = PG_OOB / ((uint32_t)a.N * 2u);
  a.kshift = -1;
  if (a.kdiv > 0 && (a.kdiv & (a.kdiv - 1)) == 0)
    for (a.kshift = 0; (1 << a.kshift) < a.kdiv;) ++a.kshift;
  if (!(a.remap & PERSIST_REMAP_FIXED) && a.n_tiles >= 8) a.remap |= PERSIST_REMAP_INTERLEAVE;  // (see there)
  int cus = 0;
  if ((rc = mi_cu_count(&cus)) != MI_MOE_OK) return rc;
  const long max_tiles = ((long)a.L / BM + (a.E < a.L ? a.E : a.L)) * a.n_tiles;
  long grid = cus < max_tiles ? cus : max_tiles;
  grid = (grid + 7) / 8 * 8;
  // no contraction length that a split could shorten by PERSIST_SPLIT_MIN_SAVED slices, or one slot per XCD
  if (!mi_gemm_persistent_splits(a.K) || grid < 16 || a.pre != nullptr) a.ws = nullptr;  // (the finishing launch writes the result only)
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), PG_LDS, s, a);
  if ((rc = mi_launch_status()) != MI_MOE_OK || a.ws == nullptr) return rc;
  // the tiles that were cut: at most half of the slots of a round that was split hold tiles (rounded up: an odd
  // number of slots per XCD)
  const int nslot = (int)(grid / 8);
  hipLaunchKernelGGL((grouped_gemm_split_finish_kernel<T, GLU>), dim3(8u * (unsigned)((nslot + 1) / 2), 4), dim3(256), 0, s, a,
                     nslot);
  return mi_launch_status();
}

bool mi_gemm_persistent_splits(int K) { return persistent_may_split(K); }

bool mi_gemm_persistent_ok(const GemmArgs& a) {
  return a.K % 8 == 0 && a.N % 8 == 0 && a.E <= PERSIST_MAX_E && mi_aligned(a.out, 16);
}

int mi_gemm_persistent(const GemmArgs& a, int dtype, int form, hipStream_t s) {
  if (!mi_gemm_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
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
