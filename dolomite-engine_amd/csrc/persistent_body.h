// The body of the persistent grouped GEMMs (persistent_gemm.hip: what it is and why; persistent_even.hip: the forms for middling
// loads; persistent_load.h: the one that the load on hand wants).
#pragma once

#include "gemm_common.h"
#include "mfma_core.h"
#include "persistent_tiles.h"

#define PG_BK 64        // K slice: one 128-byte line of a 16-bit row
#define PG_U 32768      // bytes of a ring unit: 256 rows of one operand (WT weights: 64 rows of 256 columns)
#define PG_LDS (5 * PG_U)

// NT: results are stored non-temporal
// NB: blocks of 16 weight rows of a wave (a tile has 4 NB).  EVEN: an expert's row tiles are equally high, in steps of 32 rows, and
// a low tile costs what it has (pg_locate, half)
// SCANNED: pg_form_by_load has summed up the row tiles
template <typename T, bool GLU, bool WT, bool KEEP, bool NT, int NB = 8, bool EVEN = false, int BM = 256, bool SCANNED = false>
__device__ __forceinline__ void persistent_body(const GemmArgs& a, const PgRows& experts) {
  static_assert(!KEEP || GLU, "the pre-activation belongs to the SwiGLU form");
  static_assert(!WT || !GLU, "transposed-weight form");
  static_assert(NB == 8 || !WT, "the image of transposed weights has 256 columns");
  constexpr int BN = (GLU ? 16 : 32) * NB;          // output columns per tile
  constexpr int NX = BM / 32;                       // DMA instructions of a unit of activations; a wave's row blocks
  static_assert(NX >= 5 && NX <= 8 && (NX == 8 || EVEN), "");
  // a ring of three whole slices where that fits the LDS: activations then are requested three slices ahead
  constexpr uint32_t XU = BM * 128, WU = NB * 4096;
  constexpr bool RING3 = 3 * (XU + WU) <= PG_LDS;
  static_assert(RING3 || BM == 256, "");
  constexpr int PIECES = NB == 8 ? 8 : 4;           // plain form: pieces of a unit of weights that the epilogue uses as scratch
  constexpr int NSTORE = GLU ? (KEEP ? 3 : 1) * NX * ((NB / 2 + 1) / 2) : (16 * NX + 4 * PIECES - 1) / (4 * PIECES) * PIECES;  // stores of a wave in the epilogue
  static_assert(NB + (RING3 ? NX : 0) + NSTORE < 64, "a wait counts them all");
  constexpr int MINK = RING3 ? 3 : 2;               // slices of a tile at least
  constexpr int WN = BN / 2, HB = NB / 2;           // ... per wave; SwiGLU: blocks of up, then as many of gate
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
  pg_table<BM, SCANNED>(experts, a.E, tb);
  const int total = tb.total * a.n_tiles;
  const int nfull = a.K / PG_BK;                    // whole slices; a partial one is padded with zeros
  int nk = (a.K + PG_BK - 1) / PG_BK;
  if (nk < MINK) nk = MINK;                         // (the ring wants as many: slices of zeros)
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
      list = pg_locate<BM, EVEN>(tb, a.E, a.n_tiles, it < n_items ? tile : 0);
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
  // SwiGLU weights: row 8 g + 4 wn + i of the 32 of group nb is what wave column wn multiplies as row 4 g + i of its block nb, and
  // the blocks share out the wave's columns so that the accumulators of blocks 2 p and 2 p + 1 are eight neighbours of a row (w_row):
  // results go from registers to memory in 16-byte stores.  Chunks at chunk ^ ((r >> 1) & 1 | (r >> 3) << 1), which again serves
  // the 16 rows x 4 chunks of a fragment without bank conflicts.
  const int wchunk = GLU ? (lane & 7) ^ ((wave << 1) | ((lane >> 4) & 1)) : lchunk;
  auto w_row = [&](int nb) {                        // of the tile's up or gate half, for group nb's row 8 wave + lane / 8
    const int h = nb % HB, i = (lane >> 3) & 3;
    const bool paired = h + 1 < HB || h % 2 == 1;
    return (lane >> 5) * WN + (paired ? 32 * (h / 2) + 8 * wave + 4 * (h % 2) : 16 * h + 4 * wave) + i;
  };
  const uint32_t row_bytes = (uint32_t)a.K * 2u;
  const u32x4 xsrd = pg_srd(a.in, (uint64_t)(a.gather ? a.L / a.kdiv : a.L) * row_bytes);
  const uint64_t w_bytes = (uint64_t)a.E * (GLU ? 2 : 1) * a.N * row_bytes;
  auto make_wsrd = [&](const PgTile& t) -> u32x4 {
    const uint64_t o = ((uint64_t)t.expert * (GLU ? 2 : 1) * a.N * a.K + (uint64_t)t.nt * BN * (WT ? 1 : a.K)) * 2u;
    return pg_srd(static_cast<const unsigned char*>(a.w) + o, w_bytes - o);
  };
  // sorted-order row index of the activation rows a lane fetches (clamped into the tile's expert), and the byte offsets
  // they give; rows past the expert's end lie past the buffer: zeros, no traffic, and multipliers at rest
  auto load_rows = [&](const PgTile& t, int (&raw)[NX]) {
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      const int r = t.row_begin + drow + 32 * j;
      raw[j] = r < t.row_end ? r : t.row_end - 1;
    }
    if (a.gather) {
#pragma unroll
      for (int j = 0; j < NX; ++j) raw[j] = a.sorted_scattered[raw[j]];
    }
  };
  auto make_xoff = [&](const PgTile& t, const int (&raw)[NX], uint32_t (&off)[NX]) {
    // (top-k is a power of two in most configurations: a shift instead of a division)
    const int sh = !a.gather ? 0 : a.kshift;
    if (sh >= 0) {
#pragma unroll
      for (int j = 0; j < NX; ++j) off[j] = (uint32_t)(raw[j] >> sh) * row_bytes + lchunk * 16u;
    } else {
#pragma unroll
      for (int j = 0; j < NX; ++j) off[j] = (uint32_t)(raw[j] / a.kdiv) * row_bytes + lchunk * 16u;
    }
#pragma unroll
    for (int j = 0; j < NX; ++j) off[j] = t.row_begin + drow + 32 * j < t.row_end ? off[j] : PG_OOB;
  };
  // Weight rows are at fixed distances (rows past N are another matrix's, or past the buffer: never stored).
  // WT: instruction j fills rows 8 j + 2 wave + lane / 32 of the slice; 16-byte piece l % 32 of row r holds the logical
  // piece whose 32-byte group is (piece / 2) ^ (r % 4 | (r / 8 % 4) << 2): the swizzle the transposing reads expect.
  uint32_t woff[NB];
  auto make_woff = [&]() {
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      if constexpr (WT) {
        const int r = 8 * j + 2 * wave + (lane >> 5), f = (r & 3) | ((j & 3) << 2);
        woff[j] = ((uint32_t)r * a.N + ((((lane & 31) >> 1) ^ f) << 4) + (lane & 1) * 8) * 2u;
      } else {
        const int r = GLU ? w_row(j) + (j >= HB ? a.N : 0) : 32 * j + drow;
        woff[j] = (uint32_t)r * row_bytes + wchunk * 16u;
      }
    }
  };
  const uint32_t w_step = WT ? (uint32_t)a.N * (2u * PG_BK) : 2u * PG_BK;  // bytes from slice to slice
  // a slice with fewer than 64 values: the lanes past them fetch zeros
  auto mask = [&](auto& off, int chunk, int k) {
    const bool gone = chunk * 8 >= a.K - k * PG_BK;
    for (uint32_t& o : off) o = gone ? PG_OOB : o;
  };
  auto mask_x = [&](auto& off, int k) { mask(off, lchunk, k); };
  auto mask_w = [&](int k) {
    if constexpr (WT) {
#pragma unroll
      for (int j = 0; j < 8; ++j) woff[j] = 8 * j + 2 * wave + (lane >> 5) >= a.K - k * PG_BK ? PG_OOB : woff[j];
    } else {
      mask(woff, wchunk, k);
    }
  };

  // ---- fragment reads ------------------------------------------------------------------------------------------------
  const uint32_t fswz = (frow >> 1) & 7;
  // (EVEN: the two waves of a column take row blocks in turn, so that they share a low tile)
  const uint32_t fx = (wm * (EVEN ? 16 : 128) + frow) * 128, fw = (GLU ? 8 * (frow >> 2) + 4 * wn + (frow & 3) : wn * WN + frow) * 128;
  const uint32_t fc0 = lds0 + ((fq ^ fswz) * 16), fc1 = lds0 + (((fq + 4) ^ fswz) * 16);
  const uint32_t fwswz = GLU ? ((frow >> 1) & 1) | ((frow >> 2) << 1) : fswz;
  const uint32_t fcw0 = lds0 + ((fq ^ fwswz) * 16), fcw1 = lds0 + (((fq + 4) ^ fwswz) * 16);
  // WT: ds_read_b64_tr_b16 transposes 4 rows x 16 columns across 16 lanes: lane i of the group supplies the address of
  // (row i / 4, columns 4 (i % 4) ..) and receives column i of the four rows.  Lane group q reads rows 8q .. 8q + 3 and,
  // 2 KiB further, 8q + 4 .. 8q + 7: together the 8 contraction values the matrix instruction wants.
  const uint32_t trb = (8 * fq + (frow >> 2)) * 512 + ((((frow >> 2) | (fq << 2))) << 5) + (frow & 3) * 8;
  u32x4 wf[2][NB], xf[2][NX];
  auto read_w = [&](uint32_t base, int ks, int nb) -> u32x4 {
    if constexpr (WT) {
      const uint32_t ad = base + (trb ^ ((uint32_t)(wn * 8 + nb) << 5));
      const tr_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(size_t)(ad + ks * 16384));
      const tr_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr_t)(size_t)(ad + ks * 16384 + 2048));
      return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    } else {
      typedef __attribute__((address_space(3))) const u32x4* p;
      return *(p)(size_t)(base + nb * (GLU ? 4096 : 2048));
    }
  };
  auto read_x = [&](uint32_t base, int mb) -> u32x4 {
    typedef __attribute__((address_space(3))) const u32x4* p;
    return *(p)(size_t)(base + mb * (EVEN ? 4096 : 2048));
  };

  // ---- ring and source state ------------------------------------------------------------------------------------------
  // RING3: slots of X_k, X_k+1, X_k+2 and of W_k, W_k+1 and the free one (W_k+2; then X_k+3 goes to the slot of X_k).  Else
  // slots of X_k, W_k, X_k+1, W_k+1 and the free one (W_k+2; then X_k+2 goes to the slot of X_k); X = activations.
  uint32_t p0 = 0, p1 = RING3 ? 3 * XU : PG_U, p2 = RING3 ? XU : 2 * PG_U, p3 = RING3 ? 3 * XU + WU : 3 * PG_U;
  uint32_t p4 = RING3 ? 3 * XU + 2 * WU : 4 * PG_U, px2 = 2 * XU;
  uint32_t xoff[NX], xoff_n[NX];
  u32x4 wsrd, wsrd_n;
  int kx, kx_end, kx_ev, kw, kw_end, kw_ev;         // next slice of the source tile, its end, the next one with an event
  int k0_n, k1_n;                                   // slices of the next item
  auto event_of = [&](int end) { return nfull < end ? nfull : end; };
  auto x_event = [&]() {
    if (kx == kx_end) {
#pragma unroll
      for (int j = 0; j < NX; ++j) xoff[j] = xoff_n[j];
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

  // One half slice: NB matrix instructions for each of the tile's 8 row blocks of a wave (EVEN: `pairs`).  B = 0: values [0, 32)
  // of slice k out of the registers read before, while values [32, 64) are read and W_k+2 is fetched; B = 1: those, while slice
  // k + 1 is read and X_k+2 (RING3: X_k+3) is fetched.  `hook` has two parts, the ring's rotation and
  // the next half's addresses: near the half's end, apart; EVEN, whose end a low tile leaves out: both behind the last read,
  // which is more than the issue slots that one matrix instruction leaves (with the plain form's there too, a layer of 8 experts,
  // 4096 / 14336, 8192 tokens: 4076 -> 4104 us).
  const uint32_t dma0 = lds0 + wave * 1024;
  uint32_t rw, rx;                                  // addresses of the next half's fragments
  auto half = [&](auto btag, auto ftag, int pairs, uint32_t dst, auto hook) __attribute__((always_inline)) {
    constexpr int B = decltype(btag)::value;
    constexpr bool FIRST = decltype(ftag)::value;
    constexpr int ND = B ? NX : NB, M4 = 4 * NB, NR = NB + NX;  // DMA instructions; matrix instructions of four row blocks; reads
    const uint32_t soff = B ? (uint32_t)kx * (2u * PG_BK) : (uint32_t)kw * w_step;
    auto mfma = [&](int m) {
      const int nb = m % NB, mb = m / NB;
      if constexpr (FIRST) pg_mfma_first<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
      else pg_mfma<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
    };
    auto dma_dst = [&](int j) {
      PG_SCHED();
      pg_dma_dst(dst, j * 4096);
      PG_SCHED();
    };
    auto dma = [&](int j) {
      PG_SCHED();
      if constexpr (B) pg_dma(xoff[j], xsrd, soff);
      else pg_dma(woff[j], wsrd, soff);
      PG_SCHED();
    };
    // DMA instructions [j0, j0 + n) spread over matrix instructions [m0, m0 + nm)
    auto run = [&](auto m0tag, auto nmtag, auto j0tag, auto ntag, bool reads) __attribute__((always_inline)) {
      constexpr int m0 = decltype(m0tag)::value, nm = decltype(nmtag)::value, j0 = decltype(j0tag)::value, n = decltype(ntag)::value;
      constexpr int S = nm / n >= 8 ? 1 : 0, D = nm / n >= 4 ? 2 : 1;
#pragma unroll
      for (int i = 0; i < nm; ++i) {
        mfma(m0 + i);
        if (reads && i * NR % M4 < NR) {
          const int q = i * NR / M4;
          PG_SCHED();
          if (q < NB) wf[B ^ 1][q] = read_w(rw, B ^ 1, q);
          else xf[B ^ 1][q - NB] = read_x(rx, q - NB);
          PG_SCHED();
          if (EVEN && q == NR - 1) {
            hook(0);
            hook(1);
          }
          PG_SCHED();
        }
        if (!EVEN && (m0 + i == NB * NX - 4 || m0 + i == NB * NX - 2)) {
          PG_SCHED();
          hook(m0 + i == NB * NX - 4 ? 0 : 1);
          PG_SCHED();
        }
#pragma unroll
        for (int j = 0; j < n; ++j)
          if (i == j * nm / n + S + D) dma(j0 + j);
#pragma unroll
        for (int j = 0; j < n; ++j)
          if (i == j * nm / n + S) dma_dst(j0 + j);
      }
      if constexpr ((n - 1) * nm / n + S + D >= nm) {
        asm volatile("s_nop 0");
        dma(j0 + n - 1);
      }
    };
#define PG_C(v) std::integral_constant<int, (v)>{}
    pg_own_agprs();
    constexpr int N1 = ND / 2, N2 = ND - N1;
    run(PG_C(0), PG_C(M4), PG_C(0), PG_C(N1), true);
    if constexpr (!EVEN) {
      run(PG_C(M4), PG_C(M4), PG_C(N1), PG_C(N2), false);
    } else if (NX >= 8 && pairs >= 8) {
      run(PG_C(M4), PG_C(M4), PG_C(N1), PG_C(N2), false);
    } else if (NX >= 7 && pairs == 7) {
      run(PG_C(M4), PG_C(3 * NB), PG_C(N1), PG_C(N2), false);
    } else if (NX >= 6 && pairs == 6) {
      run(PG_C(M4), PG_C(2 * NB), PG_C(N1), PG_C(N2), false);
    } else if (pairs == 5) {
      run(PG_C(M4), PG_C(NB), PG_C(N1), PG_C(N2), false);
    } else {
#pragma unroll
      for (int j = N1; j < ND; ++j) {
        dma_dst(j);
        asm volatile("s_nop 0");
        dma(j);
      }
    }
#undef PG_C
  };
  auto read_bases = [&](int ks, uint32_t ps_w, uint32_t ps_x) {
    rw = WT ? lds0 + ps_w : (ks ? fcw1 : fcw0) + fw + ps_w;
    rx = (ks ? fc1 : fc0) + fx + ps_x;
    asm volatile("" : "+v"(rx));
    if constexpr (!WT) asm volatile("" : "+v"(rw));
  };
  // stores_after_dma: the epilogue of a tile lies between the DMA this slice waits for and now
  auto step = [&](auto ftag, int pairs, bool stores_after_dma) __attribute__((always_inline)) {
    if (kw >= kw_ev) w_event();
    half(std::integral_constant<int, 0>{}, ftag, pairs, dma0 + p4, [&](int part) __attribute__((always_inline)) {
      if (part == 0) return;
      ++kw;
      read_bases(0, p3, p2);
    });
    // slice k + 1 has landed (W_k+2, RING3: and X_k+2, stay in flight); slice k is in everybody's registers
    constexpr int FLYING = NB + (RING3 ? NX : 0);
    if (decltype(ftag)::value && stores_after_dma) __builtin_amdgcn_s_waitcnt(pg_wait(FLYING + NSTORE, 0));
    else __builtin_amdgcn_s_waitcnt(pg_wait(FLYING, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    PG_SCHED();
    if (kx >= kx_ev) x_event();
    half(std::integral_constant<int, 1>{}, std::false_type{}, pairs, dma0 + p0, [&](int part) __attribute__((always_inline)) {
      if (part == 0) {
        const uint32_t t0 = p0, t1 = p1;
        p0 = p2;
        p1 = p3;
        p2 = RING3 ? px2 : t0;
        p3 = p4;
        p4 = t1;
        px2 = t0;
        if (RING3) asm volatile("" : "+s"(px2));
        asm volatile("" : "+s"(p0), "+s"(p1), "+s"(p2), "+s"(p3), "+s"(p4));
        return;
      }
      ++kx;
      read_bases(1, p1, p0);
    });
  };

  // ---- epilogue: accumulators -> (SwiGLU) -> 16-byte stores --------------------------------------------------------------
  T* __restrict__ out = static_cast<T*>(a.out);
  // rows lane and 64 + lane of the wave's 128 in the tile
  constexpr int TILE_64 = EVEN ? 128 : 64;
  const int tile_row0 = EVEN ? (lane >> 4) * 32 + wm * 16 + (lane & 15) : wm * 128 + lane;
  int orow_lo, orow_hi;                             // output rows of the wave's rows lane and 64 + lane
  auto load_out_rows = [&](const PgTile& t, int& lo, int& hi) {
    const int r0 = t.row_begin + tile_row0;
    lo = r0;
    hi = r0 + TILE_64;
    if (a.scatter) {
      lo = a.sorted_scattered[lo < t.row_end ? lo : t.row_end - 1];
      hi = a.sorted_scattered[hi < t.row_end ? hi : t.row_end - 1];
    }
  };
  // Every tile issues the same number of stores on one path; what does not exist is a lane past the buffer.  With a branch for
  // edge tiles the compiler, which counts stores along the shortest way it can construct, waited for all of them wherever it
  // needed the next tile's rows, and again in the next tile's first slice: 40 experts, 512 -> 1536, 32768 tokens 389 -> 384 us (389
  // again with the body as it is now), 32 experts, 512 -> 1024, 16384 tokens 139 -> 136, 1536 ->
  // 512 SwiGLU, 32768 tokens 639 -> 622.
  // Writes the rows [row0, row0 + out_window) of the output: all of them, unless it has more than 4 GiB.
  // SwiGLU: a lane holds eight neighbouring columns of row lane % 16 of a row block (see w_row), four lanes 64 bytes of it.  KEEP:
  // the result is formed from the ROUNDED halves of the pre-activation, as the separate activation kernel forms it from the stored
  // h, and both halves are stored in the same pass.
  auto epilogue_direct = [&](const PgTile& t, uint32_t row0) __attribute__((always_inline)) {
    const uint32_t ld = a.N * 2u;
    const int behind = t.row_end - t.row_begin, rows = behind < BM ? behind : BM;
    const uint32_t left = a.L - row0;
    const auto srd = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char*>(out) + (uint64_t)row0 * ld, (short)0,
                                                       (int)((left < a.out_window ? left : a.out_window) * ld), 0x00020000);
    // (rows of the pre-activation are the sorted order's: addressed from the tile's first, as the whole can exceed 4 GiB -- and so
    // can what an expert has behind a tile that is not EVEN, whose end is the expert's)
    const auto pre = __builtin_amdgcn_make_buffer_rsrc(KEEP ? static_cast<unsigned char*>(a.pre) + (uint64_t)t.row_begin * (2 * ld) : nullptr,
                                                       (short)0, KEEP && row0 == 0 ? (int)(rows * (2 * ld)) : 0, 0x00020000);
    const uint32_t lo = (uint32_t)orow_lo - row0, hi = (uint32_t)orow_hi - row0;
    const uint32_t rlo = tile_row0 < rows && lo < a.out_window ? lo * ld : PG_OOB;
    const uint32_t rhi = tile_row0 + TILE_64 < rows && hi < a.out_window ? hi * ld : PG_OOB;
    // Two pairs: lanes 8 .. 15 of a row block give their first eight columns to lanes 0 .. 7 for those lanes' second eight, so that a
    // store instruction writes whole 128-byte lines of eight rows, and the next one those of the other eight.
    // Byte offsets of the lane's columns in pair p (two pairs: in either store), and in the block without a partner; saturating
    // sums keep what does not exist past the buffer
    const int col0 = t.nt * BN + wn * WN;
    constexpr int PAIRS = HB / 2, QUADS = EVEN ? 0 : PAIRS / 2, STORES = PAIRS + HB % 2;
    uint32_t coff[STORES];
#pragma unroll
    for (int p = 0; p < STORES; ++p) {
      const int col = col0 + (p < 2 * QUADS ? 64 * (p / 2) + 32 * (frow >> 3) : 32 * p) + (p < PAIRS ? 8 : 4) * fq;
      coff[p] = col < a.N ? (uint32_t)col * 2u : PG_OOB;
    }
#pragma unroll
    for (int mb = 0; mb < NX; ++mb) {
      if (EVEN && mb * 32 >= rows) break;
      // where the row block's rows go: lane's own row, and rows frow % 8 and 8 + frow % 8
      auto row_of = [&](int r) { return (uint32_t)__builtin_amdgcn_ds_bpermute((((mb * 16) & 63) + r) * 4, (int)(mb < 4 ? rlo : rhi)); };
      auto pre_of = [&](int r) {
        const int prow = EVEN ? 32 * mb + 16 * wm + r : 128 * wm + 16 * mb + r;
        return KEEP && prow < rows ? (uint32_t)prow * (2 * ld) : PG_OOB;
      };
      uint32_t roff[3] = {}, poff[3] = {};
      if (QUADS > 0) {
        roff[0] = row_of(frow & 7);
        roff[1] = row_of(8 + (frow & 7));
        poff[0] = pre_of(frow & 7);
        poff[1] = pre_of(8 + (frow & 7));
      }
      if (STORES > 2 * QUADS) {
        roff[2] = row_of(frow);
        poff[2] = pre_of(frow);
      }
      struct Values { uint32_t r[4], u[4], g[4]; };  // two values each
      auto values = [&](int p) __attribute__((always_inline)) {
        Values v;
#pragma unroll
        for (int i = 0; i < (p < PAIRS ? 4 : 2); ++i) {
          const int acc = (mb * 8 + 2 * p + i / 2) * 4 + 2 * (i % 2);
          float v0 = pg_acc(acc), v1 = pg_acc(acc + 1);
          {
            float g0 = pg_acc(acc + 4 * HB), g1 = pg_acc(acc + 4 * HB + 1);
            if constexpr (KEEP) {
              v.u[i] = pack2<T>(v0, v1);
              v.g[i] = pack2<T>(g0, g1);
              v0 = unpack_lo<T>(v.u[i]);
              v1 = unpack_hi<T>(v.u[i]);
              g0 = unpack_lo<T>(v.g[i]);
              g1 = unpack_hi<T>(v.g[i]);
            }
            v0 *= silu_rcp_f32(g0);
            v1 *= silu_rcp_f32(g1);
          }
          v.r[i] = pack2<T>(v0, v1);
        }
        return v;
      };
      auto store4 = [&](const uint32_t (&v)[4], auto rsrc, uint32_t row, uint32_t col) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b128((u32x4){v[0], v[1], v[2], v[3]}, rsrc, (int)__builtin_elementwise_add_sat(row, col), 0, NT ? 2 : 0);
      };
      auto store2 = [&](const uint32_t (&v)[4], auto rsrc, uint32_t row, uint32_t col) __attribute__((always_inline)) {
        __builtin_amdgcn_raw_buffer_store_b64((u32x2){v[0], v[1]}, rsrc, (int)__builtin_elementwise_add_sat(row, col), 0, NT ? 2 : 0);
      };
      auto store_quad = [&](const uint32_t (&v)[4], const uint32_t (&w)[4], auto rsrc, const uint32_t (&row)[3], uint32_t col) __attribute__((always_inline)) {
        uint32_t x[4], y[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          x[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)v[i], (int)w[i], 0x128, 0xf, 0xc, false);  // (row_ror:8)
          y[i] = (uint32_t)__builtin_amdgcn_update_dpp((int)w[i], (int)v[i], 0x128, 0xf, 0x3, false);
        }
        store4(x, rsrc, row[0], col);
        store4(y, rsrc, row[1], col);
      };
#pragma unroll
      for (int p = 0; p < 2 * QUADS; p += 2) {
        const Values v = values(p), w = values(p + 1);
        store_quad(v.r, w.r, srd, roff, coff[p]);
        if constexpr (KEEP) {
          store_quad(v.u, w.u, pre, poff, coff[p]);
          store_quad(v.g, w.g, pre, poff, (uint32_t)__builtin_elementwise_add_sat(coff[p], ld));
        }
      }
#pragma unroll
      for (int p = 2 * QUADS; p < STORES; ++p) {
        const Values v = values(p);
        auto store = [&](const uint32_t (&x)[4], auto rsrc, uint32_t row, uint32_t col) __attribute__((always_inline)) {
          if (p < PAIRS) store4(x, rsrc, row, col);
          else store2(x, rsrc, row, col);
        };
        store(v.r, srd, roff[2], coff[p]);
        if constexpr (KEEP) {
          store(v.u, pre, poff[2], coff[p]);
          store(v.g, pre, poff[2], (uint32_t)__builtin_elementwise_add_sat(coff[p], ld));
        }
      }
      pg_own_agprs();
    }
  };
  // Plain: staged through the wave's pieces of the free ring unit, four passes of 32 rows x 128 columns (256-byte rows, 4 to a
  // piece), so that a store writes 256 bytes of a row: rows go to scattered places here, and in 128-byte pieces from the registers
  // they take longer than the staging saves (40 experts, 512 -> 1536, 32768 tokens 392 us; 403, and 490 in 64-byte pieces).
  // Chunk c of scratch row r lies at slot c ^ (r % 16): writes and reads free of conflicts, and the read-back is linear in the lane.
  constexpr int PASS_ROWS = 4 * PIECES, MBP = PASS_ROWS / 16, NPASS = (16 * NX + PASS_ROWS - 1) / PASS_ROWS;
  const uint32_t scr_w = (frow / 4) * 4096 + (frow % 4) * 256 + (((fq >> 1) ^ frow) * 16) + (fq & 1) * 8;
  const int srow = lane / 16, scc0 = (lane % 16) ^ srow;  // chunk of store 0; store it: ^ 4 (it % 4)
  auto epilogue_staged = [&](const PgTile& t, uint32_t row0) __attribute__((always_inline)) {
    typedef __attribute__((address_space(3))) u32x2* wp_t;
    typedef __attribute__((address_space(3))) const u32x4* rp_t;
    const uint32_t ld = a.N * 2u;
    const int behind = t.row_end - t.row_begin;
    const int r0 = tile_row0, rows = behind < BM ? behind : BM;
    const uint32_t window = a.out_window, left = a.L - row0;
    const auto srd = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<unsigned char*>(out) + (uint64_t)row0 * ld, (short)0,
                                                       (int)((left < window ? left : window) * ld), 0x00020000);
    const uint32_t s0 = dma0 + p4;
    const int col0 = t.nt * BN + wn * WN;
    uint32_t scr = scr_w;
    asm volatile("" : "+v"(scr));                   // (or the addresses that it gives are kept in registers from the first tile on)
    // byte offsets of the wave's rows lane and 64 + lane, and of the lane's columns in store it (% 4); saturating sums keep
    // what does not exist past the buffer
    const uint32_t lo = (uint32_t)orow_lo - row0, hi = (uint32_t)orow_hi - row0;
    const uint32_t rlo = r0 < rows && lo < window ? lo * ld : PG_OOB, rhi = r0 + TILE_64 < rows && hi < window ? hi * ld : PG_OOB;
    uint32_t coff[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const int col = col0 + (scc0 ^ (4 * c)) * 8;
      coff[c] = col < a.N && (scc0 ^ (4 * c)) * 8 < WN ? (uint32_t)col * 2u : PG_OOB;
    }
#pragma unroll
    for (int p = 0; p < NPASS; ++p) {
      if (EVEN && p * PASS_ROWS * 2 >= rows) break;
#pragma unroll
      for (int mbp = 0; mbp < MBP; ++mbp)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
          const int acc = ((p * MBP + mbp) * 8 + nb) * 4;
          const float v0 = pg_acc(acc), v1 = pg_acc(acc + 1), v2 = pg_acc(acc + 2), v3 = pg_acc(acc + 3);
          *(wp_t)(size_t)(s0 + (scr ^ (nb * 32)) + mbp * 4 * 4096) = (u32x2){pack2<T>(v0, v1), pack2<T>(v2, v3)};
        }
      pg_own_agprs();
      // (four at a time: one LDS latency for all of them)
#pragma unroll
      for (int it0 = 0; it0 < PIECES; it0 += 4) {
        u32x4 val[4];
        uint32_t roff[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int r = p * PASS_ROWS + (it0 + j) * 4;  // + srow: row of the wave's 128
          val[j] = *(rp_t)(size_t)(s0 + (it0 + j) * 4096 + lane * 16);
          roff[j] = (uint32_t)__builtin_amdgcn_ds_bpermute(((r & 63) + srow) * 4, (int)(r < 64 ? rlo : rhi));
        }
#pragma unroll
        for (int j = 0; j < 4; ++j)
          __builtin_amdgcn_raw_buffer_store_b128(val[j], srd, (int)__builtin_elementwise_add_sat(roff[j], coff[(it0 + j) % 4]), 0, NT ? 2 : 0);
      }
      pg_own_agprs();
    }
  };
  auto epilogue = [&](const PgTile& t) __attribute__((always_inline)) {
    uint32_t row0 = 0;
    do {
      if constexpr (GLU) epilogue_direct(t, row0);
      else epilogue_staged(t, row0);
      row0 += a.out_window;
    } while (row0 < (uint32_t)a.L);
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
    int raw[NX], raw_n[NX];
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
  for (int s = 0; s < MINK; ++s) {
    if (kx >= nfull) mask_x(xoff, kx);
#pragma unroll
    for (int j = 0; j < NX; ++j) {
      pg_dma_dst(dma0 + (s == 0 ? p0 : s == 1 ? p2 : px2), j * 4096);
      asm volatile("s_nop 0");
      pg_dma(xoff[j], xsrd, (uint32_t)kx * (2u * PG_BK));
    }
    ++kx;
    if (s == 2) break;
    if (kw >= nfull) mask_w(kw);
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      pg_dma_dst(dma0 + (s ? p3 : p1), j * 4096);
      asm volatile("s_nop 0");
      pg_dma(woff[j], wsrd, (uint32_t)kw * w_step);
    }
    ++kw;
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(RING3 ? 2 * NX + NB : NX + NB, 0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_bases(0, p1, p0);
#pragma unroll
  for (int i = 0; i < NB; ++i) wf[0][i] = read_w(rw, 0, i);
#pragma unroll
  for (int i = 0; i < NX; ++i) xf[0][i] = read_x(rx, i);
  read_bases(1, p1, p0);

  // ---- tile loop ------------------------------------------------------------------------------------------------------------
  bool stores_pending = false;
  for (int i = 0;; ++i) {
    const int pairs = EVEN ? pg_row_pairs(cur) : 8;
    step(std::true_type{}, pairs, stores_pending);
    for (int k = k0 + 1; k < k1; ++k) step(std::false_type{}, pairs, false);
    pg_acc_settle();
    if (k1 - k0 != nk) {
      // a part of a split tile, always a workgroup's last item: the finishing launch adds the parts up
      store_part();
      break;
    }
    // rows of the tile after next, and where the next tile's results go: requested here, taken after the epilogue
    const PgTile after = fetch(i + 2);
    int raw[NX], lo_n, hi_n;
    load_rows(after, raw);
    load_out_rows(nxt, lo_n, hi_n);
    epilogue(cur);
    // (the waits for the loads above belong here: they count the epilogue's stores, which stay in flight)
#pragma unroll
    for (int j = 0; j < NX; ++j) asm volatile("" : "+v"(raw[j]));
    asm volatile("" : "+v"(lo_n), "+v"(hi_n));
    if (i + 1 >= n_items) break;
    stores_pending = !EVEN || pairs == NX;          // (a low tile has fewer stores)
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
    for (int j = 0; j < NX; ++j) asm volatile("" : "+v"(xoff_n[j]));
    asm volatile("" : "+v"(orow_lo), "+v"(orow_hi));
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));  // surplus DMA must not outlive the workgroup's LDS
}

// column tiles of BN columns, and the order that goes with their number (persistent_tiles.h), unless the caller fixed one
__host__ __device__ inline void persistent_columns(GemmArgs& a, int BN) {
  a.n_tiles = (a.N + BN - 1) / BN;
  if (a.remap & PERSIST_REMAP_FIXED) return;
  a.remap = a.n_tiles >= 8 ? a.remap | PERSIST_REMAP_INTERLEAVE : a.remap & ~PERSIST_REMAP_INTERLEAVE;
}

// Host side: what a launch with tiles of BM rows and BN columns needs, and its grid.
static inline int persistent_grid(const GemmArgs& a, int cus, int BM, int BN) {
  const long max_tiles = ((long)a.L / BM + (a.E < a.L ? a.E : a.L)) * ((a.N + BN - 1) / BN);
  return ((int)(cus < max_tiles ? cus : max_tiles) + 7) / 8 * 8;
}
static inline int persistent_prepare(GemmArgs& a, int BM, int BN, int* grid) {
  persistent_columns(a, BN);
  a.out_window = PG_OOB / ((uint32_t)a.N * 2u);
  a.kshift = -1;
  if (a.kdiv > 0 && (a.kdiv & (a.kdiv - 1)) == 0)
    for (a.kshift = 0; (1 << a.kshift) < a.kdiv;) ++a.kshift;
  int cus = 0;
  const int rc = mi_cu_count(&cus);
  if (rc == MI_MOE_OK) *grid = persistent_grid(a, cus, BM, BN);
  return rc;
}
// ... and what one needs that picks among the forms: as many workgroups as the one with the most tiles can use, the first form's
// columns, and the workspace only if a contraction of this length is cut at all
static inline int by_load_prepare(GemmArgs& a, int form, int* grid) {
  const int unit = form == PG_SWIGLU || form == PG_SWIGLU_KEEP ? 16 : 32;
  int cus = 0, rc = persistent_prepare(a, persist_form_rows(0), unit * persist_form_blocks(0), grid);
  if (rc != MI_MOE_OK || (rc = mi_cu_count(&cus)) != MI_MOE_OK) return rc;
  for (int i = 1; i < PERSIST_FORMS; ++i) {
    const int slots = persistent_grid(a, cus, persist_form_rows(i), unit * persist_form_blocks(i));
    if (slots > *grid) *grid = slots;
  }
  if (!mi_gemm_persistent_splits(a.K) || *grid < 16 || form == PG_SWIGLU_KEEP) a.ws = nullptr;
  persist_cost(a, form, *grid);
  return MI_MOE_OK;
}
