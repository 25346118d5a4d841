// Per-expert weight gradients of the scattered-MoE layer on gfx950 matrix cores:
//
//   dW[e][m][n] = sum over the rows r of expert e (expert-sorted order) of  A[ai(r)][m] * B[bi(r)][n]
//
// i.e. one "X^T dY" product per expert, contracted over that expert's rows.  The reference gets it from the
// backward of the external scattered_experts op (lm_engine/hf_models/modeling_utils/mlp_blocks/moe.py:91-101);
// its two uses are d c_fc[e] = d_h[rows_e]^T x[token(rows_e)] and d c_proj[e] = dy[token(rows_e)]^T act[rows_e].
//
// Design
//   * Both operands are stored with the contraction index (the row) as the slow dimension, the opposite of what
//     the matrix instruction wants (8 consecutive contraction values per lane).  The tiles are staged in LDS as
//     they lie in HBM -- [row][256 columns] -- and the fragments are read with ds_read_b64_tr_b16, which transposes
//     4 rows x 16 columns across a group of 16 lanes: lane i of the group supplies the address of (row i / 4,
//     columns 4 * (i % 4) ..) and receives column i of the four rows.  Two such reads make one 16x16x32 operand.
//     The 32-byte column groups of a row are XOR-swizzled with the row number so that the 16 rows x 32 bytes of
//     one read spread over the banks.
//   * An expert's rows are cut into groups of `chunk` rows; a work item is one 256 x 256 output tile of one
//     group.  Items are dealt so that the 32 workgroups of an XCD work on the tiles of the same few groups at
//     the same time: the group's rows are then fetched from HBM once per XCD and shared through its L2.
//     Which XCD takes which groups is planned by a one-workgroup kernel in front: the groups are ranked by size,
//     longest first, and dealt to the eight XCDs back and forth (0..7, 7..0, ...), so that the XCDs get equal
//     work up to a small group and every XCD ends on its shortest items.  (Dealing the sorted rows into eight
//     equal ranges instead leaves the XCDs up to one group apart and costs 10 - 20 % under skewed loads.)
//     An item of an expert with several groups writes an fp32 partial tile and a second kernel sums the partials
//     of the expert in group order and rounds once (deterministic); an expert with one group is written directly,
//     one without rows gets zeros from the second kernel.  With few rows per expert none of that pays: whole experts, dealt
//     round by round (wgrad_whole_experts).
//   * One wave per SIMD with 128 x 128 accumulators in the AGPR half of the register file, 64-row slices, and the
//     five-unit DMA ring of persistent_gemm.hip (see there for why): one barrier per slice, one LDS read or DMA
//     instruction between any two matrix instructions.  A lane loads the indices of its eight rows of a gathered
//     operand two slices ahead and forms one offset per DMA instruction between matrix instructions (as scalar
//     arithmetic -- eleven instructions per DMA instruction, in one gap -- the gather cost 12 % of the loop).
//     Measured against the form it replaces (eight waves in two groups, 32-row slices, two barriers each), 40 experts,
//     262144 rows: 1024 x 1536 with b gathered 724 -> 646 us (1277 TFLOP/s), 1536 x 512 with a gathered 381 -> 349 us;
//     4072 rows in 32 experts, 1024 x 1024: 38.7 -> 34.0 us.
#include "mfma_core.h"

#define WGRAD_MAX_E 256

typedef short s16x4 __attribute__((ext_vector_type(4)));
#define MI_LDS __attribute__((address_space(3)))

struct WgradArgs {
  const void* a;                  // (rows_a, M)
  const void* b;                  // (rows_b, N)
  const int32_t* a_idx;           // (L,) row of `a` for sorted row r, or null: r itself
  const int32_t* b_idx;           // same for `b`
  const int32_t* expert_offsets;  // (E,) inclusive ends of the experts' row ranges (null: one expert owns all rows)
  float* partial;                 // [group][row block][column block][lane]: blocks of 16 x 16, four values a lane
  void* dw;                       // (E, M, N): written directly for an expert with a single group
  int* next_item;                 // plan: [0..8) per-XCD work counters, zero on entry; [8..17) first slot of each XCD
                                  // in the list; [32..) the groups in the order the XCDs work through them
  int L, M, N, E, chunk, m_tiles, n_tiles;
  int a_rows, b_rows;
};

// lane l of register c: expert 64 c + l -- groups of experts 0..e, and the end of its rows
struct WgradTable {
  int groups[4], end[4];
};
__device__ __forceinline__ void wgrad_table(const int32_t* __restrict__ off, int L, int E, int chunk, WgradTable& tb) {
  const int lane = threadIdx.x & 63;
  int carry = 0;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    tb.groups[c] = 0x7fffffff;
    tb.end[c] = 0;
    if (c * 64 >= E) continue;
    const int e = c * 64 + lane;
    const int end = e < E ? (off != nullptr ? off[e] : L) : 0;
    const int prev = (e < E && e > 0) ? off[e - 1] : 0;
    int incl = e < E ? (end - prev + chunk - 1) / chunk : 0;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    incl += carry;
    carry = __builtin_amdgcn_readlane(incl, 63);
    tb.groups[c] = e < E ? incl : 0x7fffffff;
    tb.end[c] = end;
  }
}

// An expert with n rows has ceil(n / chunk) groups of equal size (a multiple of 32 rows, the last one shorter).
__device__ __forceinline__ int wgrad_group_rows(int n, int groups) { return ((n + groups - 1) / groups + 31) & ~31; }

#define WG_BK 64        // rows of a slice
#define WG_U 32768      // bytes of a ring unit: one operand's 64 rows x 256 columns
#define WG_LDS (5 * WG_U)

// GA / GB: operand a / b is gathered through its index array
// PLAN: groups and their order come from wgrad_plan_kernel.  Else (wgrad_whole_experts) an item is a tile of a whole expert, round r of
// the chip the items [r grid, (r + 1) grid), of which XCD x takes the x-th eighth; every tile is written here.
template <typename T, bool GA, bool GB, bool PLAN>
__device__ __forceinline__ void wgrad_body(const WgradArgs& a) {
  constexpr int TILE = 256;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  int* item_slot = reinterpret_cast<int*>(smem_raw);  // (between items, when the ring is drained)
  const uint32_t lds0 = (uint32_t)(size_t)(MI_LDS void*)smem_raw;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave & 1, wn = wave >> 1;          // 128 rows (m) x 128 columns (n) of the tile
  const int fi = lane & 15, fq = lane >> 4;
  const int upper = lane >> 5;

  WgradTable tb;
  if constexpr (PLAN) wgrad_table(a.expert_offsets, a.L, a.E, a.chunk, tb);
  const int tiles = a.m_tiles * a.n_tiles;
  const int xcd = blockIdx.x & 7;
  // this XCD's groups: slots [xfirst, xfirst + xgroups) of the planned list
  const int xfirst = PLAN ? a.next_item[8 + xcd] : 0;
  const int xgroups = PLAN ? a.next_item[8 + xcd + 1] - xfirst : 0;
  const int* __restrict__ xlist = a.next_item + 32 + xfirst;
  const int items_x = PLAN ? xgroups * tiles : a.E * tiles;

  // ---- DMA: wave w fetches rows 16 w .. 16 w + 15 of a slice, instruction j the rows j (lanes 0-31) and 8 + j: a lane
  // then needs the indices of eight consecutive rows of a gathered operand, two loads of 16 bytes per slice.  (The two
  // rows of an instruction are neighbours in LDS; the contraction may take the rows in any order that both operands
  // share.)
  // Position lane % 32 of LDS row r holds the logical 16-byte piece whose 32-byte group is (position / 2) ^ f(r),
  // f(r) = r % 4 | (r / 8 % 4) << 2, the swizzle the transposing reads expect: four lane offsets in all.
  uint32_t piece[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int f = ((2 * (v & 1) + upper) & 3) | (((2 * wave + (v >> 1)) & 3) << 2);
    piece[v] = (uint32_t)((((((lane & 31) >> 1) ^ f) & 15) << 4) + (lane & 1) * 8) * 2u;
  }
  auto piece_of = [&](int j) { return piece[(j & 1) + 2 * (j >> 2)]; };
  const uint32_t a_ld = (uint32_t)a.M * 2u, b_ld = (uint32_t)a.N * 2u;  // bytes of a row
  // (columns past an operand's width read the next row's: their products only reach results that are never stored)
  const uint64_t a_bytes = (uint64_t)a.a_rows * a_ld, b_bytes = (uint64_t)a.b_rows * b_ld;
  const uint32_t dma0 = lds0 + wave * 8192;

  // ---- fragment reads: ds_read_b64_tr_b16, row 8 q + 4 h + i / 4, 32-byte column group F ^ f(row), piece i % 4 --------
  const uint32_t trb = (8 * fq + (fi >> 2)) * (TILE * 2) + ((((fi >> 2) | (fq << 2))) << 5) + (fi & 3) * 8;
  auto read_frag = [&](uint32_t base, int ks, int F) -> u32x4 {
    const uint32_t addr = base + (trb ^ ((uint32_t)F << 5));
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((MI_LDS s16x4*)(size_t)(addr + ks * 16384));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((MI_LDS s16x4*)(size_t)(addr + ks * 16384 + 2048));
    return __builtin_bit_cast(u32x4, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  };

  // Items of an XCD are handed out in order through a counter: the workgroups of the XCD stay on neighbouring
  // items (same group of rows, shared through the L2) and none of them idles while another still has a queue.
  // The next item is drawn when the current one has three slices left: early enough that the draw's trip to memory is
  // over when it ends, late enough that a workgroup does not hold an item another one could start.
  constexpr int DRAW_AHEAD = 3;
  int drawn = 0;
  if (PLAN && threadIdx.x == 0) drawn = atomicAdd(a.next_item + xcd, 1);
  for (int round = 0;; ++round) {
    int item = round * (int)gridDim.x + xcd * (int)(gridDim.x >> 3) + (int)(blockIdx.x >> 3);
    // (bare barriers: a fence would also wait for the last item's stores)
    if constexpr (PLAN) {
      if (threadIdx.x == 0) *item_slot = drawn;
      __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      item = __builtin_amdgcn_readfirstlane(*item_slot);
    }
    if (PLAN || round > 0) {                        // (the last item's results are out of the LDS)
      __builtin_amdgcn_s_waitcnt(pg_wait(63, 0));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
    }
    if (item >= items_x) break;
    const int grp = PLAN ? __builtin_amdgcn_readfirstlane(xlist[item / tiles]) : 0;
    // A group's tiles are numbered in bands of 8 row tiles, column tile slowest inside a band: the 32 workgroups
    // of the XCD, which hold 32 consecutive items, then cover 8 x 4 tiles -- 12 operand slabs for 32 tiles.  (Row
    // tile fastest over all of them would re-read every A slab once per column tile: with 112 x 16 tiles that is
    // 16 passes over the whole A operand.)
    const int tile = item % tiles;
    const int band = tile / (8 * a.n_tiles);
    const int rem = tile - band * 8 * a.n_tiles;
    const int left = a.m_tiles - band * 8;
    const int width = left < 8 ? left : 8;
    const int nt = rem / width;
    const int mt = band * 8 + rem - nt * width;

    // group -> expert and its row range (wave-uniform)
    int r0 = 0, r1 = 1, expert = 0, expert_groups = 1;
    if constexpr (!PLAN) {
      expert = item / tiles;
      r0 = expert > 0 ? a.expert_offsets[expert - 1] : 0;
      r1 = a.expert_offsets != nullptr ? a.expert_offsets[expert] : a.L;
      if (r1 <= r0) {                               // no rows: zeros
        T* __restrict__ out = static_cast<T*>(a.dw) + (size_t)expert * a.M * a.N;
        const int n = nt * TILE + (threadIdx.x & 31) * 8;
        for (int m = mt * TILE + (threadIdx.x >> 5); m < a.M && m < (mt + 1) * TILE; m += 8)
          if (n < a.N) *reinterpret_cast<u32x4*>(out + (size_t)m * a.N + n) = (u32x4){0u, 0u, 0u, 0u};
        continue;
      }
    } else {
      int first = 0, prev = 0;
      bool found = false;
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        if (found || c * 64 >= a.E) continue;
        const uint64_t hit = __ballot(tb.groups[c] > grp);
        const int l = hit ? __ffsll((long long)hit) - 1 : 64;
        if (l > 0) {
          first = __builtin_amdgcn_readlane(tb.groups[c], l - 1);
          prev = __builtin_amdgcn_readlane(tb.end[c], l - 1);
        }
        if (l < 64) {
          expert = c * 64 + l;
          expert_groups = __builtin_amdgcn_readlane(tb.groups[c], l) - first;
          const int end = __builtin_amdgcn_readlane(tb.end[c], l);
          const int rows = wgrad_group_rows(end - prev, expert_groups);
          r0 = prev + (grp - first) * rows;
          r1 = r0 + rows < end ? r0 + rows : end;
          found = true;
        }
      }
    }
    const int nrows = r1 - r0, nk = (nrows + WG_BK - 1) / WG_BK, nfull = nrows / WG_BK;

    const u32x4 asrd = pg_srd(static_cast<const unsigned char*>(a.a) + (size_t)mt * (TILE * 2), a_bytes - (uint64_t)mt * (TILE * 2));
    const u32x4 bsrd = pg_srd(static_cast<const unsigned char*>(a.b) + (size_t)nt * (TILE * 2), b_bytes - (uint64_t)nt * (TILE * 2));
    // lane offsets of the eight instructions: of an operand read in place relative to the slice's first row, of a
    // gathered one recomputed every slice from the row indices; rows past the group's end give zeros
    const int lrow = 16 * wave + 8 * upper;         // + j: row of the slice
    uint32_t aoff[8], boff[8];
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      aoff[j] = (uint32_t)(lrow + j) * a_ld + piece_of(j);
      boff[j] = (uint32_t)(lrow + j) * b_ld + piece_of(j);
    }
    auto mask_rows = [&](uint32_t (&off)[8], int sl) {
#pragma unroll
      for (int j = 0; j < 8; ++j) off[j] = lrow + j >= nrows - sl * WG_BK ? PG_OOB : off[j];
    };
    // Row indices of slice sl for this lane.  Requested in assembly (the compiler would wait for everything in flight
    // before their first use); they are older than the DMA that the slice's barrier leaves in flight, so they have
    // arrived behind it.  Indices past the end of the array read as 0 and are masked with their rows.
    const u32x4 isrd = pg_srd(GA ? a.a_idx : a.b_idx, (uint64_t)a.L * 4u), isrd_b = pg_srd(a.b_idx, (uint64_t)a.L * 4u);
    const uint32_t ioff = (uint32_t)lrow * 4u;
    auto load_idx = [&](u32x4 srd, int sl, u32x4 (&ix)[2]) {
      const uint32_t so = (uint32_t)(r0 + sl * WG_BK) * 4u;
      asm volatile("buffer_load_dwordx4 %0, %2, %3, %4 offen\n\tbuffer_load_dwordx4 %1, %2, %3, %4 offen offset:16"
                   : "=&v"(ix[0]), "=&v"(ix[1]) : "v"(ioff), "s"(srd), "s"(so) : "memory");
    };
    auto gathered_off = [&](const u32x4 (&ix)[2], int j, uint32_t ld) -> uint32_t { return ix[j >> 2][j & 3] * ld + piece_of(j); };

    // ---- ring (see persistent_gemm.hip): slots of A_k, B_k, A_k+1, B_k+1 and the free one ---------------------------------
    uint32_t p0 = 0, p1 = WG_U, p2 = 2 * WG_U, p3 = 3 * WG_U, p4 = 4 * WG_U;
    u32x4 ai[2], bi[2];                             // row indices of A_k+3 / B_k+2 where gathered
    u32x4 wf[2][8], xf[2][8];                       // fragments of b (columns n) and a (rows m)
    uint32_t rw, rx;
    int ks_a, ks_b;                                 // next slice of either operand to fetch
    auto half = [&](auto btag, auto ftag, uint32_t dst, auto hook) {
      constexpr int B = decltype(btag)::value;
      constexpr bool FIRST = decltype(ftag)::value;
      constexpr bool G = B ? GB : GA;
      const uint32_t soff = G ? 0u : (uint32_t)(r0 + (B ? ks_b : ks_a) * WG_BK) * (B ? b_ld : a_ld);
      pg_own_agprs();
#pragma unroll
      for (int m = 0; m < 64; ++m) {
        const int nb = m & 7, mb = m >> 3;
        if constexpr (FIRST) pg_mfma_first<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
        else pg_mfma<T>((mb * 8 + nb) * 4, wf[B][nb], xf[B][mb]);
        if (m % 2 == 0 && m < 32) {
          const int q = m / 2;
          PG_SCHED();
          if (q < 8) wf[B ^ 1][q] = read_frag(rw, B ^ 1, 8 * wn + q);
          else xf[B ^ 1][q - 8] = read_frag(rx, B ^ 1, 8 * wm + q - 8);
          PG_SCHED();
        }
        if (m % 8 == 1) {
          PG_SCHED();
          pg_dma_dst(dst, m / 8 * 1024);
          PG_SCHED();
        }
        if (m % 8 == 3) {
          PG_SCHED();
          pg_dma(B ? boff[m / 8] : aoff[m / 8], B ? bsrd : asrd, soff);
          PG_SCHED();
        }
        hook(m);
      }
    };
    auto read_bases = [&](uint32_t ps_b, uint32_t ps_a) {
      rw = lds0 + ps_b;
      rx = lds0 + ps_a;
    };
    auto step = [&](auto ftag) {
      // the indices of A_k+3 and B_k+2 go out ahead of this half's DMA and have arrived at its end
      if (GA) load_idx(isrd, ks_a + 1, ai);
      if (GB) load_idx(isrd_b, ks_b, bi);
      if (ks_a >= nfull) mask_rows(aoff, ks_a);
      half(std::integral_constant<int, 0>{}, ftag, dma0 + p4, [&](int m) {
        if (m == 62) {
          PG_SCHED();
          ++ks_a;
          read_bases(p3, p2);
          PG_SCHED();
        }
      });
      // slice k + 1 has landed (A_k+2 stays in flight); slice k is in everybody's registers
      __builtin_amdgcn_s_waitcnt(pg_wait(8, 0));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      // (the indices are there from here on: the compiler took them as ready where they were requested)
      if (GA) asm volatile("" : "+v"(ai[0]), "+v"(ai[1]));
      if (GB) asm volatile("" : "+v"(bi[0]), "+v"(bi[1]));
      PG_SCHED();
      const bool b_short = ks_b >= nfull;
      if (!GB && b_short) mask_rows(boff, ks_b);
      if (GB && b_short) {
        // (the last slice or two of a group)
#pragma unroll
        for (int j = 0; j < 8; ++j) boff[j] = gathered_off(bi, j, b_ld);
        mask_rows(boff, ks_b);
      }
      // SHORT: the offsets of this half's gathered rows are already there, masked (the last slice or two of a group)
      auto second = [&](auto short_tag) {
        half(std::integral_constant<int, 1>{}, std::false_type{}, dma0 + p0, [&](int m) {
          if (GB && !decltype(short_tag)::value && m % 8 == 2) {
            PG_SCHED();
            boff[m / 8] = gathered_off(bi, m / 8, b_ld);
            PG_SCHED();
          }
          if (GA && m % 8 == 5) {
            PG_SCHED();
            aoff[m / 8] = gathered_off(ai, m / 8, a_ld);
            PG_SCHED();
          }
          if (m == 60) {
            PG_SCHED();
            ++ks_b;
            const uint32_t t0 = p0, t1 = p1;
            p0 = p2;
            p1 = p3;
            p2 = p4;
            p3 = t0;
            p4 = t1;
            asm volatile("" : "+s"(p0), "+s"(p1), "+s"(p2), "+s"(p3), "+s"(p4));
            read_bases(p1, p0);
            PG_SCHED();
          }
        });
      };
      if (GB && b_short) second(std::true_type{});
      else second(std::false_type{});
    };

    // ---- first two slices -------------------------------------------------------------------------------------------
    u32x4 ix[3][2];
    if (GA || GB) {
      if (GA && GB) load_idx(isrd_b, 0, bi);
#pragma unroll
      for (int sl = 0; sl < 3; ++sl) load_idx(isrd, sl, ix[sl]);
      asm volatile("s_waitcnt vmcnt(0)" : "+v"(ix[0][0]), "+v"(ix[0][1]), "+v"(ix[1][0]), "+v"(ix[1][1]), "+v"(ix[2][0]),
                   "+v"(ix[2][1]), "+v"(bi[0]), "+v"(bi[1]) : : "memory");
    }
#pragma unroll
    for (int sl = 0; sl < 2; ++sl) {
      if (GA && GB && sl == 1) {
        load_idx(isrd_b, 1, bi);
        asm volatile("s_waitcnt vmcnt(0)" : "+v"(bi[0]), "+v"(bi[1]) : : "memory");
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        if (GA) aoff[j] = gathered_off(ix[sl], j, a_ld);
        if (GB) boff[j] = gathered_off(GA ? bi : ix[sl], j, b_ld);
      }
      if (sl >= nfull) {
        mask_rows(aoff, sl);
        mask_rows(boff, sl);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pg_dma_dst(dma0 + (sl ? p2 : p0), j * 1024);
        asm volatile("s_nop 0");
        pg_dma(aoff[j], asrd, GA ? 0u : (uint32_t)(r0 + sl * WG_BK) * a_ld);
      }
#pragma unroll
      for (int j = 0; j < 8; ++j) {
        pg_dma_dst(dma0 + (sl ? p3 : p1), j * 1024);
        asm volatile("s_nop 0");
        pg_dma(boff[j], bsrd, GB ? 0u : (uint32_t)(r0 + sl * WG_BK) * b_ld);
      }
    }
    if (GA) {
#pragma unroll
      for (int j = 0; j < 8; ++j) aoff[j] = gathered_off(ix[2], j, a_ld);
    }
    ks_a = ks_b = 2;
    __builtin_amdgcn_s_waitcnt(pg_wait(16, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    read_bases(p1, p0);
#pragma unroll
    for (int i = 0; i < 8; ++i) wf[0][i] = read_frag(rw, 0, 8 * wn + i);
#pragma unroll
    for (int i = 0; i < 8; ++i) xf[0][i] = read_frag(rx, 0, 8 * wm + i);

    // ---- slices -------------------------------------------------------------------------------------------------------
    step(std::true_type{});
    int k = 1;
    for (; k < nk - DRAW_AHEAD; ++k) step(std::false_type{});
    if (PLAN && threadIdx.x == 0) drawn = atomicAdd(a.next_item + xcd, 1);
    for (; k < nk; ++k) step(std::false_type{});
    pg_acc_settle();
    // surplus DMA (two slices of zeros) has to land before the ring is used again
    __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");

    // ---- output tile: register i of block (mb, nb) is row 16 mb + lane % 16, column 16 nb + 4 (lane / 16) + i -------------
    // An expert with one group is final: rounded, staged through 8 KB of LDS per wave (32 rows x 128 columns at a time,
    // 16-byte chunk c of row r at slot c ^ (r % 16)) and stored as whole 256-byte rows.  Otherwise the fp32
    // accumulators go to the group's partial slab as they are: [row block][column block][lane].
    if (!PLAN || expert_groups == 1) {
      T* __restrict__ out = static_cast<T*>(a.dw) + (size_t)expert * a.M * a.N;
      unsigned char* scratch = smem_raw + 1024 + wave * 8192;  // (past the item slot)
      const bool interior = (mt + 1) * TILE <= a.M && (nt + 1) * TILE <= a.N;
#pragma unroll
      for (int p = 0; p < 4; ++p) {
#pragma unroll
        for (int mbp = 0; mbp < 2; ++mbp)
#pragma unroll
          for (int nb = 0; nb < 8; ++nb) {
            const int blk = ((2 * p + mbp) * 8 + nb) * 4;
            const float v0 = pg_acc(blk), v1 = pg_acc(blk + 1), v2 = pg_acc(blk + 2), v3 = pg_acc(blk + 3);
            *reinterpret_cast<u32x2*>(scratch + (mbp * 16 + fi) * 256 + (((2 * nb + (fq >> 1)) ^ fi) * 16) + (fq & 1) * 8) =
                (u32x2){pack2<T>(v0, v1), pack2<T>(v2, v3)};
          }
        pg_own_agprs();
#pragma unroll
        for (int it = 0; it < 8; ++it) {
          const int r = 4 * it + (lane >> 4);
          const u32x4 v = *reinterpret_cast<const u32x4*>(scratch + r * 256 + (lane & 15) * 16);
          const int m = mt * TILE + wm * 128 + p * 32 + r, n = nt * TILE + wn * 128 + ((lane & 15) ^ (r & 15)) * 8;
          if (interior || (m < a.M && n < a.N)) *reinterpret_cast<u32x4*>(out + (size_t)m * a.N + n) = v;
        }
        pg_own_agprs();
      }
    } else {
      // (blocks wholly past M or N do not exist: a router's gradient, 40 x 1536, is a sixth of its tiles)
      const int mb0 = mt * 16 + wm * 8, nb0 = nt * 16 + wn * 8, m_blocks = (a.M + 15) / 16, n_blocks = (a.N + 15) / 16;
      f32x4* base = reinterpret_cast<f32x4*>(a.partial) + (((size_t)grp * m_blocks + mb0) * n_blocks + nb0) * 64 + lane;
#pragma unroll
      for (int mb = 0; mb < 8; ++mb) {
        pg_own_agprs();
        if (mb0 + mb >= m_blocks) continue;
#pragma unroll
        for (int nb = 0; nb < 8; ++nb) {
          const int acc = 4 * (8 * mb + nb);
          if (nb0 + nb < n_blocks)
            base[((size_t)mb * n_blocks + nb) * 64] = (f32x4){pg_acc(acc), pg_acc(acc + 1), pg_acc(acc + 2), pg_acc(acc + 3)};
        }
      }
    }
  }
}

template <typename T, bool GA, bool GB> __global__ __launch_bounds__(256, 1) void grouped_wgrad_kernel(WgradArgs a) {
  wgrad_body<T, GA, GB, true>(a);
}
template <typename T, bool GA, bool GB> __global__ __launch_bounds__(256, 1) void grouped_wgrad_whole_kernel(WgradArgs a) {
  wgrad_body<T, GA, GB, false>(a);
}

// Plan of one launch (one workgroup, in front of the main kernel): zero the eight work counters, rank the
// groups by their number of rows (longest first, ties in row order) and deal them to the XCDs back and forth.
//   plan[0..8)   work counters
//   plan[8..17)  first slot of XCD x in the list (slot 8 + 8 = one past the end)
//   plan[17]     number of experts the reduction has to write (those with no group or with several)
//   plan[32..)   group numbers (row order numbering, as the partial slabs and the reduction use) by slot
//   plan[red_at..)  (expert, first group, groups) of each of those experts, in expert order
// Up to WGRAD_PLAN_SORT groups are ranked; beyond that the groups are dealt in row order.
#define WGRAD_PLAN_SORT 8192
__global__ __launch_bounds__(1024) void wgrad_plan_kernel(const int32_t* __restrict__ offsets, int L, int E, int chunk,
                                                          int* __restrict__ plan, int red_at) {
  __shared__ int first[WGRAD_MAX_E + 1];  // groups in front of expert e
  __shared__ int ends[WGRAD_MAX_E];       // the offsets (one round trip to memory for all of them)
  __shared__ int cnt[WGRAD_MAX_E];        // groups of expert e
  __shared__ int rows[WGRAD_PLAN_SORT];
  const int tid = threadIdx.x;
  if (tid < 8) plan[tid] = 0;
  for (int e = tid; e < E; e += blockDim.x) ends[e] = offsets != nullptr ? offsets[e] : L;
  __syncthreads();
  // groups of expert e, then every expert adds up the ones in front of it by itself (E <= 256: no scan needed)
  for (int e = tid; e < E; e += blockDim.x) {
    const int n = ends[e] - (e > 0 ? ends[e - 1] : 0);
    cnt[e] = (n + chunk - 1) / chunk;
  }
  __syncthreads();
  for (int e = tid; e <= E; e += blockDim.x) {
    int g = 0, nred = 0;
    for (int i = 0; i < e; ++i) {
      const int c = cnt[i];
      g += c;
      nred += c != 1 ? 1 : 0;
    }
    first[e] = g;
    if (e == E) {
      plan[17] = nred;
    } else if (cnt[e] != 1) {  // not written by the main kernel
      plan[red_at + 3 * nred] = e;
      plan[red_at + 3 * nred + 1] = g;
      plan[red_at + 3 * nred + 2] = cnt[e];
    }
  }
  __syncthreads();
  const int G = first[E];
  const bool sorted = G <= WGRAD_PLAN_SORT;
  if (sorted) {
    // rows of every group: group i of an expert with n rows in `groups` groups of `per` rows each
    for (int e = tid; e < E; e += blockDim.x) {
      const int n = ends[e] - (e > 0 ? ends[e - 1] : 0);
      const int groups = first[e + 1] - first[e];
      if (groups == 0) continue;
      const int per = ((n + groups - 1) / groups + 31) & ~31;
      for (int i = 0; i < groups; ++i) {
        const int r1 = (i + 1) * per < n ? (i + 1) * per : n;
        rows[first[e] + i] = r1 - i * per;
      }
    }
  }
  __syncthreads();
  // XCD x gets the ranks 16 j + x and 16 j + 15 - x: G / 8 full rounds and part of one more
  const int full = G >> 3, rem = G & 7;
  if (tid < 9) {
    int start = 0;
    for (int x = 0; x < tid; ++x) start += full + (((full & 1) == 0 ? x < rem : x >= 8 - rem) ? 1 : 0);
    plan[8 + tid] = start;
  }
  for (int g = tid; g < G; g += blockDim.x) {
    int rank = g;
    if (sorted) {
      const int mine = rows[g];
      rank = 0;
      for (int o = 0; o < G; ++o) {
        const int r = rows[o];
        rank += (r > mine || (r == mine && o < g)) ? 1 : 0;
      }
    }
    const int round = rank >> 3, pos = rank & 7;
    const int x = (round & 1) == 0 ? pos : 7 - pos;
    int start = 0;
    for (int y = 0; y < x; ++y) start += full + (((full & 1) == 0 ? y < rem : y >= 8 - rem) ? 1 : 0);
    plan[32 + start + round] = g;
  }
}

// dW[e] = sum of expert e's partial slabs in group order, rounded once (experts with several groups); zeros for an
// expert without rows.  blockIdx.y walks the plan's list of such experts (without a plan -- a call with no rows at
// all -- every expert gets zeros); the waves of an entry's workgroups stride over the expert's 16 x 16 blocks, four slabs'
// loads in flight per block.  (Partial results of whole 256 x 256 tiles, in place of the blocks that exist: a router's gradient,
// 32768 rows, 40 x 1536, 68 us and 102 MB of workspace, 48 us and 20 MB now; 17 skewed experts, 920 x 520, 67.7 / 60.6 us.)
template <typename T>
__global__ __launch_bounds__(256) void wgrad_reduce_kernel(const float* __restrict__ partial,
                                                           const int* __restrict__ plan, int red_at,
                                                           T* __restrict__ dw, int M, int N, int m_blocks, int n_blocks) {
  int e = blockIdx.y, first = 0, count = 0;
  if (plan != nullptr) {
    if ((int)blockIdx.y >= plan[17]) return;
    const int* entry = plan + red_at + 3 * blockIdx.y;
    e = entry[0];
    first = entry[1];
    count = entry[2];
  }
  const long blocks = (long)m_blocks * n_blocks;
  const size_t slab = (size_t)blocks * 64;  // f32x4 per group
  const f32x4* base = reinterpret_cast<const f32x4*>(partial) + (size_t)first * slab;
  T* out = dw + (size_t)e * M * N;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  // a lane's piece of a block: row lane % 16, columns 4 (lane / 16) + 0 .. 3
  for (long id = (long)blockIdx.x * 4 + wave; id < blocks; id += (long)gridDim.x * 4) {
    const int bm = (int)(id / n_blocks), bn = (int)(id - (long)bm * n_blocks);
    const int m = bm * 16 + (lane & 15), n = bn * 16 + (lane >> 4) * 4;
    f32x4 s = {0.f, 0.f, 0.f, 0.f};
    const f32x4* p = base + id * 64 + lane;
    int g = 0;
    for (; g + 4 <= count; g += 4) {
      f32x4 v[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) v[j] = __builtin_nontemporal_load(p + (size_t)(g + j) * slab);
#pragma unroll
      for (int j = 0; j < 4; ++j) s += v[j];
    }
    for (; g < count; ++g) s += __builtin_nontemporal_load(p + (size_t)g * slab);
    if (m < M && n < N) *reinterpret_cast<u32x2*>(out + (size_t)m * N + n) = (u32x2){pack2<T>(s[0], s[1]), pack2<T>(s[2], s[3])};
  }
}

// Rows per group: between 256 and 16384, a multiple of 32, and few enough groups that the fp32 partial tiles of
// the experts with several groups stay cheap: about 384 items (1.5 per CU) before the cap.  Measured on the
// Granite-3B-A800M shapes (262144 rows, 40 experts): every megabyte of partial tiles costs about as much as
// 0.07 % of the products, so long groups beat groups of 3040 - 6080 rows (about four items per CU) by 4 - 7 %
// under skewed loads and by 12 - 18 % under an even load (where no expert is split any more); the longest-first
// plan keeps the few long items balanced.
static int wgrad_chunk(int L, int E, int M, int N) {
  const long tiles = (long)mi_ceil_div(M, 256) * mi_ceil_div(N, 256);
  long groups = (384 + tiles - 1) / tiles;
  long chunk = L / (groups > 0 ? groups : 1);
  // With at least one item per CU from whole experts alone, an expert is only cut when it is half again as long as
  // the average one: under an even load nobody is (no partial tiles, no second pass over them); the long experts of
  // a skewed load still are.
  if ((long)E * tiles >= 256 && chunk < 3L * (L / E) / 2) chunk = 3L * (L / E) / 2;
  if (chunk > 16384) chunk = 16384;
  if (chunk < 256) chunk = 256;
  return (int)(chunk / 32 * 32);
}

// Few rows per expert: every expert whole, the items dealt without a plan, which saves two launches and, in the main one, the trips to
// the plan and to the counters.  What it costs is the balance: the most loaded expert is one item a tile however many rows it has.
// Planned / whole, us (the load's unevenness in brackets, in ln(rank) of the logits): 40 experts, 1024 x 1536, 1600 tokens of 8 slots
// 74 / 60 (0), 83 / 67 (0.49), 3000 tokens 96 / 86 and 107 / 98, 5000 tokens 138 / 135 (0.3); 1536 x 512, 2048 tokens 61 / 44 (0.3), 5000
// tokens 94 / 98 (0.49); 32 experts, 1024 x 1024, 509 tokens 36 / 25 (0); 8 experts, 28672 x 4096, 1000 tokens of 2 slots 873 / 759
// (0.3).  One expert, which always wants its rows cut: 32 x 1024, 509 rows 17.1 / 15.6, 640 rows 17.5 / 17.8, 40 x 1536, 768 rows 18.1 /
// 19.9.
// `most`: rows that one expert can have at most, one a token.  If every token chooses the same experts, L / most of them, their tiles are
// all the work there is, one item of `most` rows each: the more there are of them, the more rows they may have.  Planned / whole, us, the
// load even, with half and with all of the tokens on the same experts: 1024 x 1024, top-1 of 8 experts (16 tiles), 1536 tokens 23 / 14, 33 / 26
// and 39 / 37, 4096 57 / 21, 53 / 51 and 46 / 82; top-1 of 64, 32768 tokens 93 / 82, 126 / 339 and 139 / 618; top-2 of 32 (32), 2048 37 / 26, 52 /
// 40 and 54 / 53, 8192 54 / 44, 74 / 105 and 87 / 166; 1024 x 512, top-8 of 32 (64), 3072 41 / 31, 51 / 50 and 59 / 69; 1536 x 512, top-8 of 40
// (96), 3840 64 / 57, 87 / 75 and 98 / 96; 512 x 256, top-2 of 8 (4), 1024 21 / 13, 21 / 20 and 21 / 25; 4096 x 4096, top-1 of 8 (256), 6144
// 217 / 216, 410 / 217 and 698 / 186.  At the line half of the tokens cost less than planned, all of them up to a fifth more.  (256 CUs)
static bool wgrad_whole_experts(int L, int E, long most, long tiles) {
  if (E == 1) return L <= 640;
  return (long)L <= 768L * E && L <= 32768 && (L == 0 || most <= 1024 + 32 * (L / most * tiles));
}

// (an operand with fewer rows than there are slots is gathered, and a token chooses an expert once)
static long wgrad_most_rows(int L, int a_rows, int b_rows) {
  const int rows = a_rows < b_rows ? a_rows : b_rows;
  return rows < 1 ? 1 : rows < L ? rows : L;
}

static long wgrad_max_groups(int L, int E, int chunk) { return (long)L / chunk + (E < L ? E : L); }
static size_t wgrad_plan_bytes(long groups, int E) { return ((size_t)(32 + groups + 3 * (long)E) * sizeof(int) + 255) / 256 * 256; }

// partial slabs: whole 16 x 16 blocks
static size_t wgrad_slab_bytes(long groups, int M, int N) {
  return (size_t)groups * (size_t)mi_ceil_div(M, 16) * (size_t)mi_ceil_div(N, 16) * (16 * 16 * sizeof(float));
}

extern "C" size_t mi_moe_grouped_wgrad_workspace_bytes(int L, int E, int M, int N) {
  if (L < 1 || E < 1 || M < 1 || N < 1) return 0;
  // [partial slabs][plan: 32 ints (work counters, first slots) + one int per group + three per expert, padded to
  // 256 bytes]
  const long groups = wgrad_max_groups(L, E, wgrad_chunk(L, E, M, N));
  return wgrad_slab_bytes(groups, M, N) + wgrad_plan_bytes(groups, E);
}

// what a call inside the library needs: whole experts leave no partial results
size_t mi_grouped_wgrad_bytes(int L, int a_rows, int b_rows, int M, int N, int E) {
  const long tiles = (long)mi_ceil_div(M, 256) * mi_ceil_div(N, 256);
  return wgrad_whole_experts(L, E, wgrad_most_rows(L, a_rows, b_rows), tiles) ? 0 : mi_moe_grouped_wgrad_workspace_bytes(L, E, M, N);
}

template <typename T, bool GA, bool GB, bool PLAN> static int launch_wgrad_as(const WgradArgs& g, int grid, hipStream_t s) {
  auto kern = PLAN ? grouped_wgrad_kernel<T, GA, GB> : grouped_wgrad_whole_kernel<T, GA, GB>;
  static std::atomic<uint64_t> lds_ok{0};
  const int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), WG_LDS, lds_ok);
  if (rc != MI_MOE_OK) return rc;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(256), WG_LDS, s, g);
  return mi_launch_status();
}

template <typename T, bool PLAN> static int launch_wgrad_main(const WgradArgs& g, int grid, hipStream_t s) {
  if (g.a_idx != nullptr) return g.b_idx != nullptr ? launch_wgrad_as<T, true, true, PLAN>(g, grid, s) : launch_wgrad_as<T, true, false, PLAN>(g, grid, s);
  return g.b_idx != nullptr ? launch_wgrad_as<T, false, true, PLAN>(g, grid, s) : launch_wgrad_as<T, false, false, PLAN>(g, grid, s);
}

template <typename T> static int launch_wgrad(const WgradArgs& g, int grid, int red_at, hipStream_t s) {
  if (g.L > 0) {
    if (g.next_item == nullptr) return launch_wgrad_main<T, false>(g, grid, s);
    const int rc = launch_wgrad_main<T, true>(g, grid, s);
    if (rc != MI_MOE_OK) return rc;
  }
  const int m_blocks = mi_ceil_div(g.M, 16), n_blocks = mi_ceil_div(g.N, 16);
  const long wgs = ((long)m_blocks * n_blocks + 3) / 4;  // a wave per block
  const int rblocks = wgs < 256 ? (int)wgs : 256;
  hipLaunchKernelGGL((wgrad_reduce_kernel<T>), dim3((unsigned)rblocks, (unsigned)g.E), dim3(256), 0, s, g.partial, g.next_item,
                     red_at, static_cast<T*>(g.dw), g.M, g.N, m_blocks, n_blocks);
  return mi_launch_status();
}

// `entry`: called through the library's interface, where offsets and the whole workspace are asked for.  Else no expert_offsets: one
// expert owns all rows; and mi_grouped_wgrad_bytes of workspace, or none.
int mi_grouped_wgrad(const void* a, const int32_t* a_idx, const void* b, const int32_t* b_idx, const int32_t* expert_offsets, void* dw,
                     void* workspace, size_t workspace_bytes, int L, int a_rows, int b_rows, int M, int N, int E, int dtype,
                     mi_moe_stream_t stream, bool entry) {
  if (L < 0 || M < 1 || N < 1 || E < 1) return MI_MOE_ESHAPE;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  if (M % 8 != 0 || N % 8 != 0 || E > WGRAD_MAX_E) return MI_MOE_EUNSUPPORTED;
  if (a_rows < 0 || b_rows < 0) return MI_MOE_ESHAPE;
  // rows are addressed with 32-bit byte offsets
  if ((uint64_t)a_rows * M * 2 >= (1ull << 32) || (uint64_t)b_rows * N * 2 >= (1ull << 32)) return MI_MOE_EUNSUPPORTED;
  if (!dw || (!expert_offsets && (entry || E != 1))) return MI_MOE_ENULL;
  if (L > 0 && (!a || !b)) return MI_MOE_ENULL;
  if (!mi_aligned(a, 16) || !mi_aligned(b, 16) || !mi_aligned(dw, 16) || !mi_aligned(workspace, 16)) return MI_MOE_EALIGN;
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t need = entry ? mi_moe_grouped_wgrad_workspace_bytes(L, E, M, N) : mi_grouped_wgrad_bytes(L, a_rows, b_rows, M, N, E);
  if (need > 0 && (!workspace || workspace_bytes < need)) return MI_MOE_EWORKSPACE;

  WgradArgs g;
  g.a = a; g.b = b; g.a_idx = a_idx; g.b_idx = b_idx; g.expert_offsets = expert_offsets;
  g.partial = static_cast<float*>(workspace);
  g.dw = dw;
  g.next_item = nullptr;
  g.L = L; g.M = M; g.N = N; g.E = E;
  g.a_rows = a_rows; g.b_rows = b_rows;
  g.chunk = wgrad_chunk(L, E, M, N);
  const long max_groups = wgrad_max_groups(L, E, g.chunk);
  const int red_at = (int)(32 + max_groups);
  g.m_tiles = mi_ceil_div(M, 256);
  g.n_tiles = mi_ceil_div(N, 256);
  const long tiles = (long)g.m_tiles * g.n_tiles;
  const bool whole = wgrad_whole_experts(L, E, wgrad_most_rows(L, a_rows, b_rows), tiles);
  if (L > 0 && !whole) {
    g.next_item = reinterpret_cast<int*>(static_cast<unsigned char*>(workspace) + wgrad_slab_bytes(max_groups, M, N));
    hipLaunchKernelGGL(wgrad_plan_kernel, dim3(1), dim3(1024), 0, s, expert_offsets, L, E, g.chunk, g.next_item, red_at);
  }
  int cus = 0;
  int rc = mi_cu_count(&cus);
  if (rc != MI_MOE_OK) return rc;
  // (an XCD can be dealt an eighth of the groups, rounded up: with as many workgroups as items alone, two groups of a router's
  // gradient, 509 rows, 32 x 1024, were the work of one workgroup each, 33 us)
  const long per_xcd = whole ? ((long)E * tiles + 7) / 8 : (max_groups + 7) / 8 * tiles;
  const long grid = 8 * (per_xcd < cus / 8 ? per_xcd : (cus + 7) / 8);
  return dtype == MI_MOE_BF16 ? launch_wgrad<bf16_t>(g, (int)grid, red_at, s) : launch_wgrad<f16_t>(g, (int)grid, red_at, s);
}

extern "C" int mi_moe_grouped_wgrad_whole(int L, int a_rows, int b_rows, int M, int N, int E) {
  if (L < 0 || a_rows < 0 || b_rows < 0 || M < 1 || N < 1 || E < 1) return MI_MOE_ESHAPE;
  return wgrad_whole_experts(L, E, wgrad_most_rows(L, a_rows, b_rows), (long)mi_ceil_div(M, 256) * mi_ceil_div(N, 256));
}

extern "C" int mi_moe_grouped_wgrad(const void* a, const int32_t* a_idx, const void* b, const int32_t* b_idx,
                                    const int32_t* expert_offsets, void* dw, void* workspace, size_t workspace_bytes,
                                    int L, int a_rows, int b_rows, int M, int N, int E, int dtype, mi_moe_stream_t stream) {
  return mi_grouped_wgrad(a, a_idx, b, b_idx, expert_offsets, dw, workspace, workspace_bytes, L, a_rows, b_rows, M, N, E, dtype, stream, true);
}

// ---- fp32 weight gradient on the matrix cores ----------------------------------------------------------------
// One workgroup per (expert, 128 x 128 tile of dW) walks the expert's rows 16 at a time: both operand slices go
// global -> registers -> LDS exactly as they lie in memory ([row][column], the loads of the next slice in flight
// while this one is multiplied), and the fragments of v_mfma_f32_32x32x2f32 are single floats -- lane l supplies
// a[row 2 j + l / 32][column l % 32] and the same element of b -- so no transposing read is needed: 32 lanes read
// 32 consecutive floats of one slice row.  The row pitch of 160 floats puts the two half waves (rows 2 j and
// 2 j + 1) on different halves of the 64 banks.  The rows are added in ascending order by one workgroup:
// deterministic, no workspace; experts without rows get zeros.  M % 4 == N % 4 == 0.
#define WGRAD_F32_TILE 128
#define WGRAD_F32_ROWS 16
#define WGRAD_F32_PITCH 160
__global__ __launch_bounds__(256) void grouped_wgrad_f32_kernel(const float* __restrict__ a,
                                                                const int32_t* __restrict__ a_idx,
                                                                const float* __restrict__ b,
                                                                const int32_t* __restrict__ b_idx,
                                                                const int32_t* __restrict__ offsets,
                                                                float* __restrict__ dw, int M, int N) {
  constexpr int TILE = WGRAD_F32_TILE, RS = WGRAD_F32_ROWS, PITCH = WGRAD_F32_PITCH;
  __shared__ __attribute__((aligned(16))) float sa[2][RS * PITCH];
  __shared__ __attribute__((aligned(16))) float sb[2][RS * PITCH];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave & 1, wn = wave >> 1;
  const int e = blockIdx.z;
  const int m0 = blockIdx.y * TILE, n0 = blockIdx.x * TILE;
  const int begin = e > 0 ? offsets[e - 1] : 0, end = offsets[e];
  const int nslices = (end - begin + RS - 1) / RS;

  // staging: thread t takes the float4 at column 4 (t % 32) of the slice rows t / 32 and t / 32 + 8, of both operands
  const int lrow = tid >> 5, lcol = (tid & 31) * 4;
  f32x4 ra[2], rb[2];
  auto load_slice = [&](int sl) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int r = begin + sl * RS + lrow + 8 * j;
      ra[j] = rb[j] = (f32x4){0.f, 0.f, 0.f, 0.f};  // rows past the expert's end and columns past the edge add nothing
      if (r < end) {
        const size_t ar = a_idx ? (size_t)a_idx[r] : (size_t)r;
        const size_t br = b_idx ? (size_t)b_idx[r] : (size_t)r;
        if (m0 + lcol < M) ra[j] = *reinterpret_cast<const f32x4*>(a + ar * M + m0 + lcol);
        if (n0 + lcol < N) rb[j] = *reinterpret_cast<const f32x4*>(b + br * N + n0 + lcol);
      }
    }
  };
  auto store_slice = [&](int buf) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      *reinterpret_cast<f32x4*>(&sa[buf][(lrow + 8 * j) * PITCH + lcol]) = ra[j];
      *reinterpret_cast<f32x4*>(&sb[buf][(lrow + 8 * j) * PITCH + lcol]) = rb[j];
    }
  };

  f32x16 acc[2][2];
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[mb][nb][i] = 0.f;

  const int fcol = lane & 31, fk = lane >> 5;
  if (nslices > 0) {
    load_slice(0);
    store_slice(0);
  }
  __syncthreads();
  for (int sl = 0; sl < nslices; ++sl) {
    const int buf = sl & 1;
    if (sl + 1 < nslices) load_slice(sl + 1);
#pragma unroll
    for (int j = 0; j < RS / 2; ++j) {
      const float* pa = &sa[buf][(2 * j + fk) * PITCH + wm * 64 + fcol];
      const float* pb = &sb[buf][(2 * j + fk) * PITCH + wn * 64 + fcol];
      const float af[2] = {pa[0], pa[32]}, bf[2] = {pb[0], pb[32]};
#pragma unroll
      for (int mb = 0; mb < 2; ++mb)
#pragma unroll
        for (int nb = 0; nb < 2; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[mb], bf[nb], acc[mb][nb], 0, 0, 0);
    }
    if (sl + 1 < nslices) store_slice(buf ^ 1);
    __syncthreads();
  }
  // register i of lane l: row 8 (i / 4) + 4 (l / 32) + i % 4 of the block (the a operand's index), column l % 32
  float* __restrict__ out = dw + (size_t)e * M * N;
#pragma unroll
  for (int mb = 0; mb < 2; ++mb)
#pragma unroll
    for (int nb = 0; nb < 2; ++nb) {
      const int n = n0 + wn * 64 + nb * 32 + fcol;
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int m = m0 + wm * 64 + mb * 32 + 8 * (i / 4) + 4 * fk + (i % 4);
        if (m < M && n < N) out[(size_t)m * N + n] = acc[mb][nb][i];
      }
    }
}

extern "C" int mi_moe_grouped_wgrad_f32(const float* a, const int32_t* a_idx, const float* b, const int32_t* b_idx,
                                        const int32_t* expert_offsets, float* dw, int L, int M, int N, int E,
                                        mi_moe_stream_t stream) {
  if (L < 0 || M < 1 || N < 1 || E < 1 || E > 65535) return MI_MOE_ESHAPE;
  if (M % 4 != 0 || N % 4 != 0) return MI_MOE_EUNSUPPORTED;
  if (!dw || !expert_offsets) return MI_MOE_ENULL;
  if (L > 0 && (!a || !b)) return MI_MOE_ENULL;
  if (!mi_aligned(a, 16) || !mi_aligned(b, 16)) return MI_MOE_EALIGN;
  const dim3 grid(mi_ceil_div(N, WGRAD_F32_TILE), mi_ceil_div(M, WGRAD_F32_TILE), E);
  if (grid.y > 65535u) return MI_MOE_ESHAPE;
  hipLaunchKernelGGL(grouped_wgrad_f32_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), a, a_idx, b, b_idx,
                     expert_offsets, dw, M, N);
  return mi_launch_status();
}

// ---- any-shape / any-dtype weight gradient (one thread per element of dW) ------------------------------------
// For fp32 and for shapes the matrix-core kernel above does not take.  Every element sums its expert's rows in
// ascending order in fp32 (deterministic) and is rounded once.  Correct, not fast; no workspace, no host round trip.
template <typename T>
__global__ __launch_bounds__(256) void grouped_wgrad_naive_kernel(const T* __restrict__ a, const int32_t* __restrict__ a_idx,
                                                                  const T* __restrict__ b, const int32_t* __restrict__ b_idx,
                                                                  const int32_t* __restrict__ offsets, T* __restrict__ dw,
                                                                  int M, int N) {
  const int e = blockIdx.z;
  const int n = blockIdx.x * 64 + (threadIdx.x & 63);
  const int m = blockIdx.y * 4 + (threadIdx.x >> 6);
  if (m >= M || n >= N) return;
  const int begin = e > 0 ? offsets[e - 1] : 0, end = offsets[e];
  float acc = 0.f;
  for (int r = begin; r < end; ++r) {
    const size_t ar = a_idx ? (size_t)a_idx[r] : (size_t)r;
    const size_t br = b_idx ? (size_t)b_idx[r] : (size_t)r;
    acc = fmaf(Elt<T>::load(a + ar * M + m), Elt<T>::load(b + br * N + n), acc);
  }
  Elt<T>::store(dw + ((size_t)e * M + m) * N + n, acc);
}

extern "C" int mi_moe_grouped_wgrad_naive(const void* a, const int32_t* a_idx, const void* b, const int32_t* b_idx,
                                          const int32_t* expert_offsets, void* dw, int L, int M, int N, int E, int dtype,
                                          mi_moe_stream_t stream) {
  if (L < 0 || M < 1 || N < 1 || E < 1 || E > 65535) return MI_MOE_ESHAPE;
  if (dtype != MI_MOE_F32 && dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  if (!dw || !expert_offsets) return MI_MOE_ENULL;
  if (L > 0 && (!a || !b)) return MI_MOE_ENULL;
  const dim3 grid(mi_ceil_div(N, 64), mi_ceil_div(M, 4), E);
  if (grid.y > 65535u) return MI_MOE_ESHAPE;
  hipStream_t s = static_cast<hipStream_t>(stream);
  switch (dtype) {
    case MI_MOE_F32:
      hipLaunchKernelGGL((grouped_wgrad_naive_kernel<float>), grid, dim3(256), 0, s, static_cast<const float*>(a), a_idx,
                         static_cast<const float*>(b), b_idx, expert_offsets, static_cast<float*>(dw), M, N);
      break;
    case MI_MOE_F16:
      hipLaunchKernelGGL((grouped_wgrad_naive_kernel<f16_t>), grid, dim3(256), 0, s, static_cast<const f16_t*>(a), a_idx,
                         static_cast<const f16_t*>(b), b_idx, expert_offsets, static_cast<f16_t*>(dw), M, N);
      break;
    default:
      hipLaunchKernelGGL((grouped_wgrad_naive_kernel<bf16_t>), grid, dim3(256), 0, s, static_cast<const bf16_t*>(a), a_idx,
                         static_cast<const bf16_t*>(b), b_idx, expert_offsets, static_cast<bf16_t*>(dw), M, N);
  }
  return mi_launch_status();
}
