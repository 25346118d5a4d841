// Persistent grouped GEMM with fp8 (e4m3fn) expert weights, from a few rows per expert to full batches.
//
//   out[orow(i), :] = scale[e_i] * (in[irow(i), :] @ Wq[e_i]^T)    (+ SwiGLU over the [up ; gate] halves)
//
// A workgroup of four waves per CU walks a list of 128 x 256 tiles (SwiGLU: 128 up + 128 gate rows) with the core of
// persistent_gemm.hip: accumulators by number, whole-line DMA spread between the matrix instructions, one barrier per
// 64-wide slice, no drain at a tile boundary.  What is different:
//   * The weights stay fp8 until a wave holds them: half the LDS and half the L2 -> LDS bytes of a widened copy.  A
//     16-byte read brings 16 values of a row, the operands of two matrix instructions; they are widened (exactly, two
//     values an instruction) in the issue slots that the matrix instructions leave free.  The contraction index is
//     permuted within a slice -- matrix instruction j of a pair takes values 16 q + 8 j + [0, 8) -- on both operands.
//   * 128 rows: an expert of a few hundred tokens' batch has about that many, and its weights -- 4 to 11 MB of HBM traffic
//     an expert, what bounds these sizes -- are then read once.  Rows that do not exist are lanes past the buffer: zeros,
//     and no traffic.  The ring holds three 128-wide weight slices and four 64-wide activation slices.
//   * Waves 0 and 1 fetch activations, waves 2 and 3 weights: requests retire in order within a wave, and a wave that
//     fetched both could not let its activations (L2) overtake weights (HBM) that were requested before.
//   * The channel scale meets the fp32 accumulators in the epilogue.
// Measured (64 experts of 2816 x 4096 and 4096 x 1408 weights, both projections, before -> after on one box): 24 rows per
// expert 308 -> 254 us, 96 rows 506 -> 315, 384 rows 1478 -> 844, 768 rows 2040 (widened copy) -> 1536.  What bounds it:
// with few rows the wait for the weights' next slice and the tile boundary, 1.6 - 1.8 times the matrix instructions' own
// time (matrix pipe busy 0.50 of the cycles); at full batches 0.59 of the cycles at 2.0 GHz, the rest of a slice being
// its barrier and the DMA instructions' queue.  Without the conversions, or with the weights fetched non-temporally, it
// takes the same time; reading the fragments one per two matrix instructions instead of one each is no faster either.
#include "mfma_core.h"
#include "persistent_tiles.h"

#define PF_BM 128
#define PF_XU 16384             // an activation slot: 128 rows x 64 values
#define PF_WU 32768             // a weight slot: 256 rows x 128 fp8 values
#define PF_NX 4
#define PF_NW 3
#define PF_LDS (PF_NX * PF_XU + PF_NW * PF_WU)

template <typename T> __device__ __forceinline__ uint32_t pf_widen2(uint32_t v, bool hi);
template <> __device__ __forceinline__ uint32_t pf_widen2<bf16_t>(uint32_t v, bool hi) {
  return hi ? __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, true))
            : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(v, 1.0f, false));
}
template <> __device__ __forceinline__ uint32_t pf_widen2<f16_t>(uint32_t v, bool hi) {
  return hi ? __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, true))
            : __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(v, 1.0f, false));
}

template <typename T, bool GLU>
__global__ __launch_bounds__(256, 1) void grouped_gemm_fp8_persistent_kernel(GemmArgs a) {
  constexpr int BN = GLU ? 128 : 256;               // output columns per tile
  constexpr int NSTORE = GLU ? 8 : 16;              // stores of a wave in the epilogue
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;
  typedef __attribute__((address_space(3))) const u32x4* frag_ptr_t;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const uint32_t lds_w = (uint32_t)(size_t)(lds_ptr_t)smem_raw, lds_x = lds_w + PF_NW * PF_WU;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;          // 64 activation rows, 128 weight rows (SwiGLU: 64 up, 64 gate)
  const int frow = lane & 15, fq = lane >> 4;
  const bool isx = wave < 2;                        // fetches activations (else weights)
  const int dw = wave & 1;                          // pieces 2 j + dw of a slot (1 KB: 8 rows of 128 bytes)

  // ---- which tiles -----------------------------------------------------------------------------------------------
  PgTable tb;
  pg_table<PF_BM>(pg_rows(a.expert_offsets, a.L, a.E), a.E, tb);
  const int nd = (a.K + 127) / 128;                 // weight slices (at least 3); two activation slices each
  const SplitPlan sp = persist_split_plan(tb.total * a.n_tiles, blockIdx.x & 7, blockIdx.x >> 3, gridDim.x >> 3, 2 * nd, false,
                                          (a.remap & PERSIST_REMAP_INTERLEAVE) != 0);
  const int n_items = sp.full_rounds + (sp.lslot < sp.rem ? 1 : 0);
  if (n_items == 0) return;
  PgTile list;                                      // lane l: item (64-item block) + l
  auto fetch = [&](int i) -> PgTile {               // called with i = 0, 1, 2, ...; past the last item: the last item
    if (i >= n_items) i = n_items - 1;
    else if ((i & 63) == 0) {
      const int it = i + lane;
      const int tile = it < sp.full_rounds ? sp.base + it * sp.stride : sp.rem_base + sp.lslot;
      list = pg_locate<PF_BM>(tb, a.E, a.n_tiles, it < n_items ? tile : 0);
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
  // Slot image: row r of 128 bytes keeps its 16-byte chunks at positions ^ ((r >> 1) & 7).  Lane l of piece 2 j + dw fills
  // position l % 8 of row 16 j + drow.  Weights: position p holds chunk p (16 fp8 values); activations: positions
  // 0-3 hold the even chunks (8 values), 4-7 the odd ones, so that position q + 4 j is values 16 q + 8 j + [0, 8).
  const int drow = dw * 8 + (lane >> 3);
  const int lpos = (lane & 7) ^ (dw * 4 + (lane >> 4));
  const int xchunk = 2 * (lpos & 3) + (lpos >> 2);
  const uint32_t row_bytes = (uint32_t)a.K * 2u;
  const u32x4 xsrd = pg_srd(a.in, (uint64_t)(a.gather ? a.L / a.kdiv : a.L) * row_bytes);
  const int wrows = (GLU ? 2 : 1) * a.N;
  // the streamed-tile layout (decode_fp8.hip): units of 32 rows, 4 KB a unit and 128 values
  const uint32_t unit = (uint32_t)(a.K >> 7) * 4096u;
  const int units = (a.N + (GLU ? 15 : 31)) / (GLU ? 16 : 32);
  const uint64_t w_bytes = a.w_tiled ? (uint64_t)a.E * units * unit : (uint64_t)a.E * wrows * a.K;
  auto make_wsrd = [&](const PgTile& t) -> u32x4 {
    const uint64_t o = a.w_tiled ? ((uint64_t)t.expert * units + t.nt * 8) * unit
                                 : ((uint64_t)t.expert * wrows + (uint64_t)t.nt * BN) * a.K;
    return pg_srd(static_cast<const unsigned char*>(a.w) + o, w_bytes - o);
  };
  // sorted-order row index of the activation rows a lane fetches (clamped), and the byte offsets they give (rows past
  // the expert's end: past the buffer)
  auto load_rows = [&](const PgTile& t, int (&raw)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int r = t.row_begin + drow + 16 * j;
      raw[j] = r < t.row_end ? r : t.row_end - 1;
    }
    if (a.gather) {
#pragma unroll
      for (int j = 0; j < 8; ++j) raw[j] = a.sorted_scattered[raw[j]];
    }
  };
  auto make_xoff = [&](const PgTile& t, const int (&raw)[8], uint32_t (&off)[8]) {
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const int s = !a.gather ? raw[j] : (a.kshift >= 0 ? raw[j] >> a.kshift : raw[j] / a.kdiv);
      off[j] = t.row_begin + drow + 16 * j < t.row_end ? (uint32_t)s * row_bytes + xchunk * 16u : PG_OOB;
    }
  };
  // Source offsets of a wave, four per half slice A .. D of a weight slice.  Activations: pieces 0-3 in A and C, 4-7 in
  // B and D; weights: pieces 0-3 in D, then 4-7, 8-11, 12-15 in the next A, B, C.
  uint32_t dof[16], xoff_n[8];
  auto set_x = [&]() {
#pragma unroll
    for (int j = 0; j < 16; ++j) dof[j] = xoff_n[j & 7];
  };
  auto set_w = [&]() {
#pragma unroll
    for (int j = 0; j < 16; ++j) {
      const int R = 16 * ((j + 4) & 15) + drow;     // slot row
      const int t = R & 31;
      if (a.w_tiled) {
        dof[j] = (uint32_t)(R >> 5) * unit + t * 128u + ((lpos ^ (((t >> 1) & 1) | (((t >> 2) & 1) << 2))) * 16u);
      } else {
        const int r = GLU ? (t >> 4) * a.N + (R >> 5) * 16 + (t & 15) : R;
        dof[j] = (uint32_t)r * (uint32_t)a.K + lpos * 16u;
      }
    }
  };
  // position of a wave's source in its tile: slices of 64 values (activations) or 128 (weights)
  u32x4 srd, wsrd_n;
  int pos = 0;
  const int pend = isx ? 2 * nd : nd, pfull = isx ? a.K / 64 : a.K / 128;
  const uint32_t pstep = !isx && a.w_tiled ? 4096u : 128u;
  uint32_t soff = 0;                                // byte offset of the position's values
  uint32_t ring;                                    // LDS address of its slot, this wave's pieces
  auto mask = [&]() {                               // a slice that K does not fill: lanes past K fetch zeros
    const bool gone = isx ? xchunk * 8 >= a.K - pos * 64 : lpos * 16 >= a.K - pos * 128;
#pragma unroll
    for (int j = 0; j < 16; ++j) dof[j] = gone ? PG_OOB : dof[j];
  };
  auto advance_x = [&]() {
    if (pos >= pend) {
      set_x();
      pos = 0;
    }
    if (pos >= pfull) mask();
    soff = (uint32_t)pos * 128u;
    ring = ring + PF_XU >= lds_x + PF_NX * PF_XU ? ring + PF_XU - PF_NX * PF_XU : ring + PF_XU;
    ++pos;
  };
  auto advance_w = [&]() {
    if (pos >= pend) {
      srd = wsrd_n;
      if (pfull != pend) set_w();
      pos = 0;
    }
    if (pos >= pfull) mask();
    soff = (uint32_t)pos * pstep;
    ring = ring + PF_WU >= lds_w + PF_NW * PF_WU ? ring + PF_WU - PF_NW * PF_WU : ring + PF_WU;
    ++pos;
  };

  // ---- fragment reads ------------------------------------------------------------------------------------------------
  const uint32_t fswz = (frow >> 1) & 7;
  const uint32_t fp0 = frow * 128 + ((fq ^ fswz) * 16), fp1 = frow * 128 + (((fq + 4) ^ fswz) * 16);
  const uint32_t fw0 = lds_w + wn * 16384 + fp0, fw1 = lds_w + wn * 16384 + fp1;
  const uint32_t fx0 = lds_x + wm * 8192 + fp0, fx1 = lds_x + wm * 8192 + fp1;
  uint32_t xo = 0, wo = 0;                          // slots of the slice at hand, relative to the rings
  u32x4 raw[8], wf[2][8], xf[2][4];
  auto read_raw = [&](uint32_t base, int nb) -> u32x4 {
    return *(frag_ptr_t)(size_t)(base + (GLU ? (nb & 3) * 4096 + (nb >> 2) * 2048 : nb * 2048));
  };
  auto read_x = [&](uint32_t base, int mb) -> u32x4 { return *(frag_ptr_t)(size_t)(base + mb * 2048); };

  // Half slice G (0-3: A-D) of a weight slice: 32 matrix instructions.  A, C (first values of each pair): read the second
  // half of the activation slice, widen the second half of the weights; B, D: read the next slice, widen its first half.
  auto half = [&](auto gtag, auto ftag, uint32_t rw, uint32_t rx) {
    constexpr int G = decltype(gtag)::value, B = G & 1;
    constexpr bool FIRST = decltype(ftag)::value;
    const uint32_t dst = ring + (isx ? B * 8192 : ((G + 1) & 3) * 8192);
    pg_own_agprs();
#pragma unroll
    for (int m = 0; m < 32; ++m) {
      const int nb = m & 7, mb = m >> 3;
      if constexpr (FIRST) pg_mfma_first<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
      else pg_mfma<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
      PG_SCHED();
      if (B == 0) {
        if (m < 8 && m % 2 == 0) xf[1][m / 2] = read_x(rx, m / 2);
        const int q = m >> 2, e = m & 3;
        wf[1][q][e] = pf_widen2<T>(raw[q][2 + (e >> 1)], e & 1);
        if (e == 3) asm volatile("" : "+v"(wf[1][q]));  // (here, and not where it is used: in the half after)
      } else {
        if (m < 8) raw[m] = read_raw(rw, m);
        else if (m < 12) xf[0][m - 8] = read_x(rx, m - 8);
        else if (m >= 16) {
#pragma unroll
          for (int c = (m - 16) * 2; c < (m - 16) * 2 + 2; ++c) {
            const int q = c >> 2, e = c & 3;
            wf[0][q][e] = pf_widen2<T>(raw[q][e >> 1], e & 1);
            if (e == 3) asm volatile("" : "+v"(wf[0][q]));
          }
        }
      }
      PG_SCHED();
      if (m % 8 == 1) {
        pg_dma_dst(dst, m / 8 * 2048);
        PG_SCHED();
      }
      if (m % 8 == 3) {
        pg_dma(dof[G * 4 + m / 8], srd, soff);
        PG_SCHED();
      }
    }
  };
  typedef std::integral_constant<int, 0> half_a;
  typedef std::integral_constant<int, 1> half_b;
  typedef std::integral_constant<int, 2> half_c;
  typedef std::integral_constant<int, 3> half_d;
  // Between the halves of a slice: the next slice has landed -- behind it may be in flight what this wave requested
  // since: activations two slices less a half, weights one slice -- and this one is in everybody's registers.
  // stores: the epilogue of a tile lies between those requests.
  auto meet = [&](bool odd, bool stores) {
    if (isx) {
      if (stores) __builtin_amdgcn_s_waitcnt(pg_wait(12 + NSTORE, 0));
      else __builtin_amdgcn_s_waitcnt(pg_wait(12, 0));
    } else if (odd) {
      if (stores) __builtin_amdgcn_s_waitcnt(pg_wait(16 + NSTORE, 0));
      else __builtin_amdgcn_s_waitcnt(pg_wait(16, 0));
    } else {
      __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    PG_SCHED();
  };
  // one weight slice (two activation slices)
  auto step = [&](auto ftag, bool stores) {
    if (isx) advance_x();
    half(half_a{}, ftag, 0u, fx1 + xo);
    meet(false, stores);
    xo = (xo + PF_XU) & (PF_NX * PF_XU - 1);
    half(half_b{}, std::false_type{}, fw1 + wo, fx0 + xo);
    if (isx) advance_x();
    half(half_c{}, std::false_type{}, 0u, fx1 + xo);
    meet(true, stores);
    xo = (xo + PF_XU) & (PF_NX * PF_XU - 1);
    wo = wo + PF_WU == PF_NW * PF_WU ? 0 : wo + PF_WU;
    if (!isx) advance_w();
    half(half_d{}, std::false_type{}, fw0 + wo, fx0 + xo);
  };

  // ---- epilogue: accumulators x scale -> (SwiGLU) -> pieces of the ring that this wave's own DMA fills next -> 16-byte
  // stores (persistent_gemm.hip's, for 64 rows: two passes of 32 rows x 128 columns, SwiGLU one of 64 x 64) ---------------
  T* __restrict__ out = static_cast<T*>(a.out);
  constexpr int SB = GLU ? 128 : 256;               // bytes of a scratch row
  constexpr int RPP = 1024 / SB;                    // scratch rows per piece and per store instruction
  constexpr int PASS_ROWS = 8 * RPP, NPASS = 64 / PASS_ROWS, MBP = PASS_ROWS / 16, NBO = GLU ? 4 : 8;
  const uint32_t scr_swz = GLU ? (frow >> 1) & 7 : frow;
  const uint32_t scr_w = (frow / RPP) * 2048 + (frow % RPP) * SB + (((fq >> 1) ^ scr_swz) * 16) + (fq & 1) * 8;
  const int srow = lane / (SB / 16), sslot = lane % (SB / 16);
  const int scc0 = GLU ? sslot ^ ((srow >> 1) & 7) : sslot ^ (srow & 15);
  // output row of the wave's row `lane`; scales of its weight rows lane and 64 + lane (SwiGLU: up, gate)
  auto load_ends = [&](const PgTile& t, int& orow, float& lo, float& hi) {
    const int r = t.row_begin + wm * 64 + lane;
    orow = r;
    if (a.scatter) orow = a.sorted_scattered[r < t.row_end ? r : t.row_end - 1];
    const int c = t.nt * BN + wn * (GLU ? 64 : 128) + lane, c2 = GLU ? c : c + 64;
    const float* s = a.wscale + (size_t)t.expert * wrows;
    lo = s[c < a.N ? c : a.N - 1];
    hi = s[(GLU ? a.N : 0) + (c2 < a.N ? c2 : a.N - 1)];
  };
  int orow_l;
  float sc_lo, sc_hi;
  // Every tile issues the same number of stores on one path, what does not exist as lanes past the buffer, and none is waited for
  // before the next tile's first slice (rows [row0, row0 + out_window): persistent_body.h).  Before, with a branch for edge tiles (all
  // tiles of a middling load), and now: a layer of 64 experts, hidden 4096, 309.0 -> 305.0 us at 1024 tokens, 252.7 -> 250.4 at 180,
  // 580 -> 575 at 2500.  Leaving out the matrix instructions of row blocks that a tile does not have gains 2 % at 180 tokens and loses
  // 4 - 10 % from 600 on: with branches in a half slice the fragments are waited for at each, and four copies of the loop spill.
  auto epilogue_as = [&](auto nt_tag, const PgTile& t, uint32_t row0) __attribute__((always_inline)) {
    constexpr bool NT = decltype(nt_tag)::value;
    typedef __attribute__((address_space(3))) u32x2* wp_t;
    const uint32_t ld = (uint32_t)a.N * 2u;
    const uint32_t window = a.out_window, left = a.L - row0;
    const auto osrd = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char*>(out) + (uint64_t)row0 * ld, (short)0,
                                                        (int)((left < window ? left : window) * ld), 0x00020000);
    // activations: the slot behind the last one requested; weights: the second half of the one being requested
    const uint32_t s0 = !isx ? ring + 16384
                             : (ring + PF_XU >= lds_x + PF_NX * PF_XU ? ring + PF_XU - PF_NX * PF_XU : ring + PF_XU);
    const int col0 = t.nt * BN + wn * (GLU ? 64 : 128);
    // byte offsets of the wave's row `lane`, and of the lane's columns in store it (% CP); the sums saturate
    constexpr int CP = GLU ? 2 : 4;
    const uint32_t orel = (uint32_t)orow_l - row0;
    const uint32_t orow_off = wm * 64 + lane < t.row_end - t.row_begin && orel < window ? orel * ld : PG_OOB;
    uint32_t coff[CP];
#pragma unroll
    for (int c = 0; c < CP; ++c) {
      const int col = col0 + (scc0 ^ (4 * c)) * 8;
      coff[c] = col < a.N ? (uint32_t)col * 2u : PG_OOB;
    }
#pragma unroll
    for (int p = 0; p < NPASS; ++p) {
      asm volatile("" : "+v"(sc_lo), "+v"(sc_hi));  // (or all the scales of both passes would be held at once)
#pragma unroll
      for (int nb = 0; nb < NBO; ++nb) {
        float sc[4], sg[4];                         // scales of this lane's four columns
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int from = ((nb & 3) * 16 + fq * 4 + i) * 4;
          sc[i] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(nb < 4 ? sc_lo : sc_hi)));
          if (GLU) sg[i] = __int_as_float(__builtin_amdgcn_ds_bpermute(from, __float_as_int(sc_hi)));
        }
#pragma unroll
        for (int mbp = 0; mbp < MBP; ++mbp) {
          const int blk = (p * MBP + mbp) * 8 + nb;
          float v[4];
#pragma unroll
          for (int i = 0; i < 4; ++i) {
            v[i] = pg_acc(blk * 4 + i) * sc[i];
            if (GLU) {
              v[i] = v[i] * silu_rcp_f32(pg_acc((blk + 4) * 4 + i) * sg[i]);
            }
          }
          *(wp_t)(size_t)(s0 + (scr_w ^ (nb * 32)) + mbp * (16 / RPP) * 2048) =
              (u32x2){pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        }
      }
      pg_own_agprs();
#pragma unroll
      for (int it0 = 0; it0 < 8; it0 += 4) {
        u32x4 val[4];
        uint32_t roff[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          val[j] = *(frag_ptr_t)(size_t)(s0 + (it0 + j) * 2048 + lane * 16);
          roff[j] = (uint32_t)__builtin_amdgcn_ds_bpermute((p * PASS_ROWS + (it0 + j) * RPP + srow) * 4, (int)orow_off);
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(val[j], osrd, (int)__builtin_elementwise_add_sat(roff[j], coff[(it0 + j) % CP]), 0, NT ? 2 : 0);
      }
      pg_own_agprs();
    }
  };
  auto epilogue = [&](const PgTile& t) __attribute__((always_inline)) {
    uint32_t row0 = 0;
    do {
      if (a.out_nt) epilogue_as(std::true_type{}, t, row0);
      else epilogue_as(std::false_type{}, t, row0);
      row0 += a.out_window;
    } while (row0 < (uint32_t)a.L);
  };

  // ---- prologue: activation slices 0-2; weight slices 0, 1 and the first four pieces of 2 ---------------------------------
  PgTile cur = fetch(0), nxt = fetch(1);
  {
    int rows[8], rows_n[8];
    load_rows(cur, rows);
    load_rows(nxt, rows_n);
    load_ends(cur, orow_l, sc_lo, sc_hi);
    make_xoff(cur, rows, xoff_n);
    if (isx) set_x();
    else set_w();
    make_xoff(nxt, rows_n, xoff_n);
  }
  wsrd_n = make_wsrd(cur);
  srd = isx ? xsrd : wsrd_n;
  wsrd_n = make_wsrd(nxt);
  asm volatile("" : "+v"(orow_l), "+v"(sc_lo), "+v"(sc_hi));
#pragma unroll
  for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(xoff_n[j]));
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));
  auto issue4 = [&](auto gtag, uint32_t dst) {
    constexpr int G = decltype(gtag)::value;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      pg_dma_dst(dst, j * 2048);
      asm volatile("s_nop 0");
      pg_dma(dof[G * 4 + j], srd, soff);
    }
  };
  if (isx) {
    ring = lds_x + (PF_NX - 1) * PF_XU + dw * 1024;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      advance_x();
      issue4(half_a{}, ring);
      issue4(half_b{}, ring + 8192);
    }
    __builtin_amdgcn_s_waitcnt(pg_wait(16, 0));
  } else {
    ring = lds_w + (PF_NW - 1) * PF_WU + dw * 1024;
#pragma unroll
    for (int s = 0; s < 3; ++s) {
      advance_w();
      issue4(half_d{}, ring);
      if (s < 2) {
        issue4(half_a{}, ring + 8192);
        issue4(half_b{}, ring + 16384);
        issue4(half_c{}, ring + 24576);
      }
    }
    __builtin_amdgcn_s_waitcnt(pg_wait(20, 0));
  }
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) raw[i] = read_raw(fw0, i);
#pragma unroll
  for (int i = 0; i < 4; ++i) xf[0][i] = read_x(fx0, i);
#pragma unroll
  for (int c = 0; c < 32; ++c) wf[0][c >> 2][c & 3] = pf_widen2<T>(raw[c >> 2][(c & 3) >> 1], c & 1);
  asm volatile("s_nop 3");

  // ---- tile loop ------------------------------------------------------------------------------------------------------------
  bool stores_pending = false;
  for (int i = 0;; ++i) {
    step(std::true_type{}, stores_pending);
    for (int d = 1; d < nd; ++d) step(std::false_type{}, false);
    pg_acc_settle();
    // rows of the tile after next, and the ends of the next tile: requested here, taken after the epilogue
    const PgTile after = fetch(i + 2);
    int rows[8], orow_n;
    float lo_n, hi_n;
    load_rows(after, rows);
    load_ends(nxt, orow_n, lo_n, hi_n);
    epilogue(cur);
    if (i + 1 >= n_items) break;
    stores_pending = true;
    make_xoff(after, rows, xoff_n);
    wsrd_n = make_wsrd(after);
    orow_l = orow_n;
    sc_lo = lo_n;
    sc_hi = hi_n;
    cur = nxt;
    nxt = after;
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+v"(xoff_n[j]));  // (the waits for the loads above belong here)
    asm volatile("" : "+v"(orow_l), "+v"(sc_lo), "+v"(sc_hi));
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));  // surplus DMA must not outlive the workgroup's LDS
}

// ---- host side ----------------------------------------------------------------------------------------------------------------
template <typename T, bool GLU> static int launch_fp8_persistent(GemmArgs a, hipStream_t s) {
  auto kern = grouped_gemm_fp8_persistent_kernel<T, GLU>;
  static std::atomic<uint64_t> lds_ok{0};
  int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), PF_LDS, lds_ok);
  if (rc != MI_MOE_OK) return rc;
  a.n_tiles = mi_ceil_div(a.N, GLU ? 128 : 256);
  a.out_window = PG_OOB / ((uint32_t)a.N * 2u);
  a.kshift = -1;
  if ((a.kdiv & (a.kdiv - 1)) == 0)
    for (a.kshift = 0; (1 << a.kshift) < a.kdiv;) ++a.kshift;
  int cus = 0;
  if ((rc = mi_cu_count(&cus)) != MI_MOE_OK) return rc;
  const long max_tiles = ((long)a.L / PF_BM + (a.E < a.L ? a.E : a.L)) * a.n_tiles;
  long grid = cus < max_tiles ? cus : max_tiles;
  grid = (grid + 7) / 8 * 8;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), PF_LDS, s, a);
  return mi_launch_status();
}

bool mi_gemm_fp8_persistent_ok(const GemmArgs& a) {
  const double in_rows = a.gather ? (double)a.L / a.kdiv : (double)a.L;
  return a.K % 16 == 0 && a.K > 256 && a.N % 8 == 0 && a.E <= PERSIST_MAX_E && mi_aligned(a.out, 16) &&
         in_rows * a.K * 2.0 < (double)PG_OOB;
}

// Where these tiles are the faster form.  Measured, us, up / down projection, these against the register-staged tiles:
//   hidden 4096, 64 experts, I 1408   24 rows per expert 164 / 90 (200 / 108), 96: 200 / 115 (321 / 185), 384: 548 / 296
//                                     (965 / 513), 768: 986 / 551 (1473 / 870)
//   hidden 4096, 8 experts, I 14336   80 rows 217 / 162 (316 / 233), 1024: 1589 / 864 (2317 / 1297)
//   hidden 1536, 40 experts, I 512    19 rows 26.2 / 15.9 (27.4 / 13.4), 64: 26.4 / 15.7 (33.5 / 19.3), 819: 112 / 71 (181 / 148)
//   hidden 1024, 32 experts, I 512    24 rows 20.3 / 14.2 (20.5 / 13.0), 80: 20.5 / 14.5 (20.2 / 13.5), 256: 38 / 25 (43 / 33)
//   hidden 1024, 8 experts, I 512     24 rows 18.4 / 13.0 (16.6 / 11.5), 256: 18.6 / 13.2 (17.3 / 13.4), 1024: 35 / 22 (49 / 39)
// A tile has a latency of its own that only a long contraction, or a tile for most of the CUs, pays back.
bool mi_gemm_fp8_persistent_pick(int L, int K, int N, int E, bool glu) {
  const long avg = (long)L / E;
  const long tiles = (long)E * ((avg + PF_BM) / PF_BM) * mi_ceil_div(N, glu ? 128 : 256);
  return avg >= 192 || K >= 1280 || tiles >= (avg >= 48 ? 200 : 400);
}

int mi_gemm_fp8_persistent(const GemmArgs& a, int dtype, bool glu, hipStream_t s) {
  if (!mi_gemm_fp8_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
  if (dtype == MI_MOE_BF16) return glu ? launch_fp8_persistent<bf16_t, true>(a, s) : launch_fp8_persistent<bf16_t, false>(a, s);
  if (dtype == MI_MOE_F16) return glu ? launch_fp8_persistent<f16_t, true>(a, s) : launch_fp8_persistent<f16_t, false>(a, s);
  return MI_MOE_EDTYPE;
}
