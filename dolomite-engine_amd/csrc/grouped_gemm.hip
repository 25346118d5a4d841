// Grouped ("scatter2scatter") GEMM of the scattered-MoE forward on gfx950 matrix cores.
//
//   out[orow(i), :] = in[irow(i), :] @ W[e_i]^T        for every row i of the expert-sorted order
//
// with an optional SwiGLU epilogue (W rows [0,N) are "up", [N,2N) "gate"; out = up * silu(gate)).
// Stands in for the external scattered_experts op called at
// lm_engine/hf_models/modeling_utils/mlp_blocks/moe.py:91-101 (call sites moe.py:273-290) and for
// GLUActivation (activations/glu.py:42-43) when fused.
//
// Kernels in this file, in order:
//   grouped_gemm_kernel             register-staged tiles (any K that is a multiple of one 16-byte chunk; bf16, fp16
//                                   and fp32): the design notes below
//   grouped_gemm_dma_kernel         the same tile with the operands brought to LDS by DMA, one tile per workgroup
//   grouped_gemm_naive_kernel       one thread per output element, only on request (cfg 3)
// Large expert loads run on the persistent kernel of persistent_gemm.hip.
//
// Design
//   * One workgroup computes a BM x BN output tile of ONE expert.  The tile list is not built on the
//     host (that would need the per-expert counts, i.e. a device->host sync): every workgroup derives
//     "its" (expert, row-tile, column-tile) from the E inclusive offsets with a short scalar scan.  The
//     grid is the host-side upper bound floor(L/BM)+min(E,L) row tiles; surplus workgroups exit.
//   * Workgroup ids are re-mapped so that each of the 8 XCDs (ids are dealt round-robin to XCDs)
//     works on a contiguous range of tiles: neighbouring tiles share the gathered activation rows
//     (column tiles of one row tile) and the expert's weight matrix, which then stay in that XCD's L2.
//   * Both operands are K-contiguous in HBM (activations (rows, K), weights (E, N, K)), so both are
//     fetched as 16-byte chunks, staged in LDS with an XOR swizzle (conflict-free ds_write_b128 /
//     ds_read_b128) and fed to v_mfma_f32_32x32x16 as the A (weights) and B (activations) operands.
//     With the weights as operand A each lane ends up with 4 consecutive output columns of one row,
//     so the epilogue packs 4 results into one 8-byte store.
//   * Two LDS stages: the global loads of K-tile i+1 are issued before the MFMAs of tile i and
//     written to the other stage afterwards; one barrier per K-tile.
#include "gemm_common.h"

#include <type_traits>

template <typename T> struct Mfma32;
template <> struct Mfma32<bf16_t> {
  typedef bf16x8 vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
  }
};
template <> struct Mfma32<f16_t> {
  typedef f16x8 vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0);
  }
};

// fp32 operands: a 16-byte chunk holds four k values; the lane halves (lane / 32) hold different chunks, so four
// 32x32x2 instructions -- element i of both operands -- consume the eight k values of a chunk pair.  Which k a
// lane contributes in which step does not matter as long as both operands use the same assignment.
template <> struct Mfma32<float> {
  typedef f32x4 vec;
  static __device__ __forceinline__ f32x16 run(vec a, vec b, f32x16 c) {
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[i], c, 0, 0, 0);
    return c;
  }
};

// 8 fp8 e4m3fn values (two dwords) -> 8 values of a 16-bit type (exact: e4m3 fits in either)
template <typename T> struct Widen8;
template <> struct Widen8<bf16_t> {
  static __device__ __forceinline__ u32x4 run(uint32_t lo, uint32_t hi) {
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 p0 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false);
    const bf16x2 p1 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true);
    const bf16x2 p2 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false);
    const bf16x2 p3 = __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true);
    return (u32x4){__builtin_bit_cast(uint32_t, p0), __builtin_bit_cast(uint32_t, p1), __builtin_bit_cast(uint32_t, p2),
                   __builtin_bit_cast(uint32_t, p3)};
  }
};
template <> struct Widen8<f16_t> {
  static __device__ __forceinline__ u32x4 run(uint32_t lo, uint32_t hi) {
    typedef float f32x2 __attribute__((ext_vector_type(2)));
    const f32x2 p0 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, false), p1 = __builtin_amdgcn_cvt_pk_f32_fp8(lo, true);
    const f32x2 p2 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, false), p3 = __builtin_amdgcn_cvt_pk_f32_fp8(hi, true);
    return (u32x4){pack2<f16_t>(p0[0], p0[1]), pack2<f16_t>(p1[0], p1[1]), pack2<f16_t>(p2[0], p2[1]),
                   pack2<f16_t>(p3[0], p3[1])};
  }
};
template <> struct Widen8<float> {  // (not used: fp32 activations have no fp8 form)
  static __device__ __forceinline__ u32x4 run(uint32_t, uint32_t) { return (u32x4){0u, 0u, 0u, 0u}; }
};


// Tile -> (expert, row range, column tile).  Row tiles are numbered expert by expert (expert e has
// ceil(n_e / BM) of them), column tiles innermost.  The walk over the E inclusive offsets is done by
// one wavefront 64 experts at a time (one coalesced load + a shuffle scan) instead of E dependent
// scalar loads; every wave of the workgroup does it redundantly, so no LDS or barrier is involved.
// With `remap` the workgroup ids (dealt round-robin to the 8 XCDs) are permuted so that each XCD
// owns a contiguous range of tiles.  Returns false for surplus workgroups.
struct TileCoord {
  int expert, row_begin, row_end, nt;
};

template <int BM>
__device__ __forceinline__ bool decode_tile(const int32_t* __restrict__ off, int L, int E, int n_tiles, int remap,
                                            TileCoord& tc) {
  const int lane = threadIdx.x & 63;
  // pass 1: total number of row tiles
  int total_m = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int end = e < E ? mi_expert_end(off, L, e) : 0;
    const int prev = (e < E && e > 0) ? off[e - 1] : 0;
    int t = e < E ? (end - prev + BM - 1) / BM : 0;
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) t += __shfl_xor(t, o, 64);
    total_m += t;
  }
  const int total = total_m * n_tiles;
  int tile;
  if (remap & 1) {
    const int per = (total + 7) >> 3;
    const int local = blockIdx.x >> 3;
    if (local >= per) return false;
    tile = (blockIdx.x & 7) * per + local;
  } else {
    tile = blockIdx.x;
  }
  if (tile >= total) return false;
  const int mt = tile / n_tiles;
  tc.nt = tile - mt * n_tiles;
  // pass 2: the expert whose row tiles contain mt
  int carry = 0;
  for (int e0 = 0; e0 < E; e0 += 64) {
    const int e = e0 + lane;
    const int end = e < E ? mi_expert_end(off, L, e) : 0;
    const int prev = (e < E && e > 0) ? off[e - 1] : 0;
    const int t = e < E ? (end - prev + BM - 1) / BM : 0;
    int incl = t;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      int v = __shfl_up(incl, o, 64);
      if (lane >= o) incl += v;
    }
    incl += carry;
    const uint64_t hit = __ballot(incl > mt);
    if (hit) {
      const int src = __ffsll((long long)hit) - 1;
      const int first_tile = __shfl(incl - t, src, 64);
      const int p = __shfl(prev, src, 64);
      tc.expert = e0 + src;
      tc.row_begin = p + (mt - first_tile) * BM;
      tc.row_end = __shfl(end, src, 64);
      return true;
    }
    carry = __shfl(incl, 63, 64);
  }
  return false;
}

// scheduling-group masks of __builtin_amdgcn_sched_group_barrier
#define SG_MFMA 0x008
#define SG_VMEM_RD 0x020
#define SG_DS_RD 0x100
#define SG_DS_WR 0x200

// W8: the weights are fp8 e4m3fn bytes with one fp32 scale per weight row (a.wscale); a thread fetches the 8 bytes
// of its chunk and widens them on their way into LDS, the scale meets the accumulators in the epilogue.  For batches
// between decode (decode_fp8.hip streams an expert's weights once per 16 rows) and the sizes where widening all
// weights first pays (mi_moe_fp8_dequant).
template <typename T, int BM, int BNW, int WM, int WN, bool GLU, bool KTAIL, bool W8 = false>
__global__ __launch_bounds__(WM* WN * 64) void grouped_gemm_kernel(GemmArgs a) {
  static_assert(!W8 || sizeof(T) == 2, "fp8 weights go with 16-bit activations");
  constexpr int CE = 16 / sizeof(T);        // elements per 16-byte chunk (8 for the 16-bit types, 4 for fp32)
  constexpr int BK = 8 * CE;                // K tile: 128 bytes per row
  constexpr int NT = WM * WN * 64;
  constexpr int CPR = BK / CE;              // 16-byte chunks per tile row
  constexpr int RS = NT / CPR;              // tile rows covered by one pass of the workgroup
  constexpr int XCH = BM * CPR / NT;        // chunks per thread, activation tile
  constexpr int WCH = BNW * CPR / NT;       // chunks per thread, weight tile
  constexpr int BN = GLU ? BNW / 2 : BNW;   // output columns per tile
  constexpr int WTM = BM / WM;              // wave tile, rows
  constexpr int WTN = BNW / WN;             // wave tile, weight rows
  constexpr int MB = WTM / 32, NB = WTN / 32;
  constexpr int STAGE_ELEMS = (BM + BNW) * BK;
  constexpr int NMFMA = MB * NB;            // MFMAs per 16-wide k step
  constexpr int NRD = MB + NB;              // fragment reads per k step
  constexpr int NWR = XCH + WCH;            // LDS chunk writes per K tile
  constexpr int RD_PER = (NRD + NMFMA - 1) / NMFMA;
  constexpr int WR_PER = (NWR + 2 * NMFMA - 1) / (2 * NMFMA);
  constexpr int LD_PER = (NWR + NMFMA - 1) / NMFMA;
  static_assert(RS % 16 == 0 && BM % RS == 0 && BNW % RS == 0, "tile/thread shape");
  static_assert(!GLU || NB % 2 == 0, "SwiGLU needs an even number of column blocks per wave");
  typedef typename Mfma32<T>::vec frag_t;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  T* smem = reinterpret_cast<T*>(smem_raw);

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave % WM, wn = wave / WM;

  TileCoord tc;
  if (!decode_tile<BM>(a.expert_offsets, a.L, a.E, a.n_tiles, a.remap, tc)) return;
  const int expert = tc.expert, row_begin = tc.row_begin, row_end = tc.row_end, nt = tc.nt;

  // ---- per-thread global sources ---------------------------------------------------------------
  const int c = tid % CPR;   // chunk within a tile row
  const int r0 = tid / CPR;  // first tile row of this thread
  constexpr int WROWS_MUL = GLU ? 2 : 1;
  const T* __restrict__ xbase = static_cast<const T*>(a.in);
  const T* __restrict__ wbase = static_cast<const T*>(a.w) + (W8 ? 0 : (size_t)expert * WROWS_MUL * a.N * a.K);
  // W8: byte address of the expert's weights; woff[j] is a byte offset (row-major: of the row's chunk c; tiled: of
  // the row inside stage 0 of its unit) and wfx[j] the row's slot swizzle in the tiled layout
  const uint8_t* __restrict__ wbase8 = nullptr;
  if constexpr (W8) {
    const size_t expert_bytes =
        a.w_tiled ? (size_t)mi_ceil_div_dev(a.N, GLU ? 16 : 32) * (size_t)(a.K >> 7) * 4096 : (size_t)WROWS_MUL * a.N * a.K;
    wbase8 = static_cast<const uint8_t*>(a.w) + (size_t)expert * expert_bytes;
  }
  int wfx[WCH];

  uint32_t xoff[XCH], woff[WCH];
#pragma unroll
  for (int j = 0; j < XCH; ++j) {
    int srow = row_begin + r0 + j * RS;
    if (srow > row_end - 1) srow = row_end - 1;  // tail rows re-read the last valid row; never stored
    int src = a.gather ? a.sorted_scattered[srow] / a.kdiv : srow;
    xoff[j] = (uint32_t)src * (uint32_t)a.K + c * CE;
  }
#pragma unroll
  for (int j = 0; j < WCH; ++j) {
    int r = r0 + j * RS;
    int col, half = 0;
    if (GLU) {
      half = r >= BN;
      col = nt * BN + (half ? r - BN : r);
    } else {
      col = nt * BN + r;
    }
    if (col > a.N - 1) col = a.N - 1;  // column tail re-reads the last weight row; never stored
    woff[j] = (uint32_t)(half * a.N + col) * (uint32_t)a.K + c * CE;
    wfx[j] = 0;
    if constexpr (W8) {
      if (a.w_tiled) {
        // unit u = 16 up + 16 gate channels (GLU) or 32 channels; row t of the unit's 32-row stage image
        const int u = GLU ? col >> 4 : col >> 5;
        const int t = GLU ? (col & 15) + 16 * half : (col & 31);
        woff[j] = (uint32_t)u * (uint32_t)(a.K >> 7) * 4096u + (uint32_t)t * 128u;
        wfx[j] = ((t >> 1) & 1) | (((t >> 2) & 1) << 2);
      }
    }
  }

  // LDS tile layout: row r holds its eight 16-byte chunks at slots  chunk ^ swz(r),
  // swz(r) = (r & 7) ^ ((r >> 3) & 1): any 8 consecutive rows AND any 16 consecutive rows of one
  // logical chunk fall into distinct bank groups (row parity selects the upper / lower 32 banks).
  // RS % 16 == 0, so all chunks of a thread share one swizzle.
  const int sw_c = c ^ ((r0 & 7) ^ ((r0 >> 3) & 1));
  const int st_x = (r0 * CPR + sw_c) * CE;              // element offset inside the X tile
  const int st_w = BM * BK + (r0 * CPR + sw_c) * CE;    // ... inside the W tile (after the X tile)

  u32x4 xreg[XCH], wreg[WCH];
  u32x2 wraw[W8 ? WCH : 1];  // W8: the chunk's 8 bytes as loaded (widened when they go to LDS)
  const int nk = (a.K + BK - 1) / BK;
  // W8: byte offset of this thread's 8-byte chunk of the K tile that starts at k0 (tiled: K % 128 == 0, so every
  // chunk exists and kc = k0 + 8 c < K)
  auto w8_at = [&](int j, int k0) -> uint32_t {
    if (!a.w_tiled) return woff[j] + (uint32_t)k0;
    const int kc = k0 + c * CE;
    return woff[j] + (uint32_t)(kc >> 7) * 4096u + (uint32_t)((((kc & 127) >> 4) ^ wfx[j]) << 4) + (uint32_t)(kc & 8);
  };

  auto load_global = [&](int kt) {
    int k0 = kt * BK;
    if (KTAIL) {
      // the last K tile may be partial: out-of-range chunks re-read chunk 0 of the row and are zeroed
      const bool kvalid = (k0 + c * CE) < a.K;
      const int koff = kvalid ? k0 : -(c * CE);
#pragma unroll
      for (int j = 0; j < XCH; ++j) {
        u32x4 v = *reinterpret_cast<const u32x4*>(xbase + xoff[j] + koff);
        xreg[j] = kvalid ? v : (u32x4){0u, 0u, 0u, 0u};
      }
#pragma unroll
      for (int j = 0; j < WCH; ++j) {
        if constexpr (W8) {
          // (a partial K tile only exists with row-major weights: the tiled layout has whole 128-wide stages)
          const u32x2 v = *reinterpret_cast<const u32x2*>(wbase8 + woff[j] + koff);
          wraw[j] = kvalid ? v : (u32x2){0u, 0u};
        } else {
          u32x4 v = *reinterpret_cast<const u32x4*>(wbase + woff[j] + koff);
          wreg[j] = kvalid ? v : (u32x4){0u, 0u, 0u, 0u};
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < XCH; ++j) xreg[j] = *reinterpret_cast<const u32x4*>(xbase + xoff[j] + k0);
#pragma unroll
      for (int j = 0; j < WCH; ++j) {
        if constexpr (W8) wraw[j] = *reinterpret_cast<const u32x2*>(wbase8 + w8_at(j, k0));
        else wreg[j] = *reinterpret_cast<const u32x4*>(wbase + woff[j] + k0);
      }
    }
  };
  // chunk writes [first, first + count) of this thread's NWR chunks (X chunks first, then W chunks)
  auto store_lds = [&](int stage, int first, int count) {
    T* s = smem + stage * STAGE_ELEMS;
#pragma unroll
    for (int j = 0; j < NWR; ++j) {
      if (j < first || j >= first + count) continue;
      if (j < XCH)
        *reinterpret_cast<u32x4*>(s + st_x + j * RS * BK) = xreg[j];
      else if constexpr (W8)
        *reinterpret_cast<u32x4*>(s + st_w + (j - XCH) * RS * BK) = Widen8<T>::run(wraw[j - XCH][0], wraw[j - XCH][1]);
      else
        *reinterpret_cast<u32x4*>(s + st_w + (j - XCH) * RS * BK) = wreg[j - XCH];
    }
  };

  // ---- fragment reads ---------------------------------------------------------------------------
  // lane l reads tile row (block_row0 + l%32), logical chunk 2*kk + l/32
  const int frow = lane & 31, fhalf = lane >> 5;
  const int fswz = (frow & 7) ^ ((frow >> 3) & 1);  // block_row0 is a multiple of 32
  int frag_x_off[MB], frag_w_off[NB];                // element offsets of the row inside a stage
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) frag_x_off[mb] = (wm * WTM + mb * 32 + frow) * BK;
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    int r;
    if (GLU) {
      constexpr int HB = NB / 2;  // blocks per half
      int h = nb >= HB;
      r = h * BN + wn * (WTN / 2) + (h ? nb - HB : nb) * 32 + frow;
    } else {
      r = wn * WTN + nb * 32 + frow;
    }
    frag_w_off[nb] = BM * BK + r * BK;
  }
  int chunk_off[4];
#pragma unroll
  for (int kk = 0; kk < 4; ++kk) chunk_off[kk] = ((kk * 2 + fhalf) ^ fswz) * CE;

  frag_t xf[2][MB], wf[2][NB];
  auto read_frags = [&](int stage, int kk, int buf) {
    const T* s = smem + stage * STAGE_ELEMS + chunk_off[kk];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      wf[buf][nb] = __builtin_bit_cast(frag_t, *reinterpret_cast<const u32x4*>(s + frag_w_off[nb]));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      xf[buf][mb] = __builtin_bit_cast(frag_t, *reinterpret_cast<const u32x4*>(s + frag_x_off[mb]));
  };

  f32x16 acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nb][mb][i] = 0.f;

  auto mfma_step = [&](int buf) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = Mfma32<T>::run(wf[buf][nb], xf[buf][mb], acc[nb][mb]);
  };

  // ---- software pipeline ------------------------------------------------------------------------
  // Per K tile (4 k-steps of two chunks each), with LDS stages cur / nxt and fragment buffers 0 / 1:
  //   step 0: MFMA(buf0) | read frags(step1, cur) -> buf1
  //   step 1: MFMA(buf1) | read frags(step2, cur) -> buf0 | write first half of tile kt+1 -> nxt
  //   step 2: MFMA(buf0) | read frags(step3, cur) -> buf1 | write second half            -> nxt
  //   barrier            (nxt complete; everybody has fetched its last fragments of cur)
  //   step 3: MFMA(buf1) | read frags(step0, nxt) -> buf0 | global loads of tile kt+2 -> registers
  // The sched_group_barrier sequences ask the backend to issue the LDS / global instructions in the
  // shadow of the MFMAs (one wave per SIMD: nothing else hides their issue slots).
  load_global(0);
  store_lds(0, 0, NWR);
  __syncthreads();
  load_global(nk > 1 ? 1 : 0);
  read_frags(0, 0, 0);

  // The last round stages a surplus tile (a re-read of the last one) that nobody consumes; keeping the
  // loop body uniform keeps the accumulators in place (no peeled copy of the 256 accumulator registers).
  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & 1, nxt = cur ^ 1;
    read_frags(cur, 1, 1);
    mfma_step(0);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);

    read_frags(cur, 2, 0);
    store_lds(nxt, 0, NWR / 2);
    mfma_step(1);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_WR, WR_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);

    read_frags(cur, 3, 1);
    store_lds(nxt, NWR / 2, NWR - NWR / 2);
    mfma_step(0);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_WR, WR_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    __syncthreads();

    read_frags(nxt, 0, 0);
    load_global(kt + 2 < nk ? kt + 2 : nk - 1);  // the surplus load of the last round is never used
    mfma_step(1);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
      __builtin_amdgcn_sched_group_barrier(SG_VMEM_RD, LD_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  // ---- epilogue ---------------------------------------------------------------------------------
  // acc[nb][mb][i]: weight row (output column) = 8*(i/4) + 4*(lane/32) + i%4 of block nb,
  //                 activation row             = lane%32 of block mb
  T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = row_begin + wm * WTM + mb * 32 + frow;
    if (row >= row_end) continue;
    const int orow = a.scatter ? a.sorted_scattered[row] : row;
    T* orow_ptr = out + (size_t)orow * a.N;
    constexpr int OB = GLU ? NB / 2 : NB;
#pragma unroll
    for (int nb = 0; nb < OB; ++nb) {
      const int col0 = nt * BN + (GLU ? wn * (WTN / 2) : wn * WTN) + nb * 32 + fhalf * 4;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = col0 + g * 8;
        if (col >= a.N) continue;
        float v[4];
        f32x4 su = {1.f, 1.f, 1.f, 1.f}, sg = {1.f, 1.f, 1.f, 1.f};
        if constexpr (W8) {  // (N % 4 == 0 and col % 4 == 0: the four columns exist together)
          const float* sc = a.wscale + (size_t)expert * WROWS_MUL * a.N + col;
          su = *reinterpret_cast<const f32x4*>(sc);
          if (GLU) sg = *reinterpret_cast<const f32x4*>(sc + a.N);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (GLU) {
            float up = acc[nb][mb][g * 4 + i];
            float gt = acc[nb + NB / 2][mb][g * 4 + i];
            if constexpr (W8) {
              up *= su[i];
              gt *= sg[i];
            }
            v[i] = up * silu_f32(gt);
          } else {
            v[i] = acc[nb][mb][g * 4 + i];
            if constexpr (W8) v[i] *= su[i];
          }
        }
        if constexpr (sizeof(T) == 4) {
          *reinterpret_cast<f32x4*>(orow_ptr + col) = (f32x4){v[0], v[1], v[2], v[3]};
        } else {
          u32x2 p = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
          *reinterpret_cast<u32x2*>(orow_ptr + col) = p;
        }
      }
    }
  }
}

// ------------------------------------------------------------------------------------------------
// Main kernel: global -> LDS by DMA (global_load_lds_dwordx4), 4 LDS stages of 32 k each.
//
// The register-staged kernel above keeps only one K tile in flight; under load the L2 -> CU latency
// exceeds one tile's worth of MFMA time and the matrix cores idle.  Here the tiles never pass through
// VGPRs: every wave issues 16-byte-per-lane DMA loads whose destination is a contiguous 1 KiB run of
// LDS (lane i -> base + 16*i).  Three tiles are in flight while a fourth is consumed.
//
//   stage layout   (BM + BNW) rows x 32 k, 64 bytes per row = 4 slots of 16 bytes;
//                  slot of logical chunk c in row r:  c ^ ((r >> 2) & 3)   (ds_read_b128 conflict-free)
//   DMA mapping    one wave instruction fills 16 rows: lane l -> row l/4, slot l%4, so the lane fetches
//                  logical chunk (l%4) ^ ((row >> 2) & 3) of its row: the swizzle is applied on the
//                  global side, 4 lanes still cover one contiguous 64-byte piece of a row
//   iteration kt   (stage cur = kt % 4, fragment buffers 0/1, two k-steps of 16)
//       A: MFMA(step 0, buf0)      | ds_read step 1 of cur -> buf1
//       s_waitcnt vmcnt(2 tiles)   : my share of tile kt+1 has landed;  lgkmcnt(0): my reads of cur are done
//       s_barrier                  : tile kt+1 complete, stage cur free
//       B: MFMA(step 1, buf1)      | ds_read step 0 of tile kt+1 -> buf0 | DMA tile kt+4 -> stage cur
// The waits are explicit (s_waitcnt immediates); a fence-carrying __syncthreads would drain all DMA.
// (Eight stages where a CU has one workgroup: one expert of 509 rows, 1024 -> 512 SwiGLU, 12.5 -> 12.9 us.)
// KTAIL: the last slice has fewer than 32 values of k.  Lanes past them fetch the row's last chunk, and their fragments are zeros.
// ------------------------------------------------------------------------------------------------

__device__ __forceinline__ constexpr int waitcnt_imm(int vm, int lgkm) {
  // gfx9 encoding: vmcnt = {imm[15:14], imm[3:0]}, expcnt = imm[6:4] (7 = no wait), lgkmcnt = imm[11:8]
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 15) << 8);
}

// One DMA instruction: every lane moves 16 bytes from (scalar base + its 32-bit byte offset) to LDS; the
// 64 destinations are the contiguous run starting at the LDS byte address in M0.  Written as inline
// assembly on purpose: for the builtin the compiler assumes that any later LDS read may alias the DMA write
// and puts "s_waitcnt vmcnt(0)" in front of it, which drains the prefetch ring every K slice.  Here the
// ordering is done by hand (s_waitcnt immediates before the barrier that publishes a stage).
// The offset register is read when the instruction issues, but the compiler treats a register named by an
// assembly statement as busy until vmcnt reaches 0 and waits before overwriting it: callers pass offsets
// that live in registers of their own for a whole tile, never a per-slice temporary.  TAG keeps otherwise
// identical statements in the two arms of a branch from being merged back into one with a selected
// (temporary) operand.
template <int TAG>
__device__ __forceinline__ void dma16_to_lds(const void* base, uint32_t byte_off, uint32_t lds_addr) {
  if (TAG == 0)
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2" : : "s"(lds_addr), "v"(byte_off), "s"(base)
                 : "memory", "m0");
  else
    asm volatile("s_mov_b32 m0, %0\n\tglobal_load_lds_dwordx4 %1, %2 ; next tile" : : "s"(lds_addr), "v"(byte_off), "s"(base)
                 : "memory", "m0");
}

template <typename T, int BM, int BNW, int WM, int WN, bool GLU, bool KTAIL>
__global__ __launch_bounds__(WM* WN * 64) void grouped_gemm_dma_kernel(GemmArgs a) {
  constexpr int BK = 32;
  constexpr int NSTAGE = 4;
  constexpr int NW = WM * WN;
  constexpr int NT = NW * 64;
  constexpr int ROWS = BM + BNW;
  constexpr int STAGE_BYTES = ROWS * BK * 2;
  constexpr int NLD = ROWS / 16 / NW;       // DMA instructions per wave per tile
  constexpr int BN = GLU ? BNW / 2 : BNW;
  constexpr int WTM = BM / WM, WTN = BNW / WN;
  constexpr int MB = WTM / 32, NB = WTN / 32;
  constexpr int NMFMA = MB * NB;
  constexpr int NRD = MB + NB;
  constexpr int RD_PER = (NRD + NMFMA - 1) / NMFMA;
  constexpr int LD_PER = (NLD + NMFMA - 1) / NMFMA;
  static_assert(ROWS % (16 * NW) == 0 && BM % 16 == 0, "tile/wave shape");
  static_assert(!GLU || NB % 2 == 0, "SwiGLU needs an even number of column blocks per wave");
  static_assert((NSTAGE - 1) * NLD <= 63 && (NSTAGE & (NSTAGE - 1)) == 0, "vmcnt range");
  typedef typename Mfma32<T>::vec frag_t;
  typedef __attribute__((address_space(3))) void* lds_ptr_t;
  typedef const __attribute__((address_space(1))) void* glb_ptr_t;

  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;

  TileCoord tc;
  if (!decode_tile<BM>(a.expert_offsets, a.L, a.E, a.n_tiles, a.remap, tc)) return;
  const int expert = tc.expert, row_begin = tc.row_begin, row_end = tc.row_end, nt = tc.nt;

  // ---- DMA sources: instruction j of this wave fills stage rows [(j*NW + wave)*16, +16) -----------
  constexpr int WROWS_MUL = GLU ? 2 : 1;
  const T* __restrict__ xbase = static_cast<const T*>(a.in);
  const T* __restrict__ wbase = static_cast<const T*>(a.w) + (size_t)expert * WROWS_MUL * a.N * a.K;
  const int lchunk = (lane & 3) ^ ((lane >> 4) & 3);  // (row >> 2) & 3 == (lane >> 4) & 3: groups are 16-row aligned
  const T* src[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {
    const int r = (j * NW + wave) * 16 + (lane >> 2);  // stage row
    if (r < BM) {
      int srow = row_begin + r;
      if (srow > row_end - 1) srow = row_end - 1;  // tail rows re-read the last valid row; never stored
      const int s = a.gather ? a.sorted_scattered[srow] / a.kdiv : srow;
      src[j] = xbase + (size_t)s * a.K + lchunk * 8;
    } else {
      const int wr = r - BM;
      int col, half = 0;
      if (GLU) {
        half = wr >= BN;
        col = nt * BN + (half ? wr - BN : wr);
      } else {
        col = nt * BN + wr;
      }
      if (col > a.N - 1) col = a.N - 1;  // column tail re-reads the last weight row; never stored
      src[j] = wbase + ((size_t)half * a.N + col) * a.K + lchunk * 8;
    }
  }
  const int nk = KTAIL ? (a.K + BK - 1) / BK : a.K / BK;
  const int k_last = KTAIL ? a.K - 8 - lchunk * 8 : 0;  // where the lane's last chunk of a row begins, less its place in a slice
  auto dma_tile = [&](int kt, int stage) {
    int k0 = (kt < nk ? kt : nk - 1) * BK;  // surplus rounds re-fetch the last tile; never consumed
    if (KTAIL && k0 > k_last) k0 = k_last;
#pragma unroll
    for (int j = 0; j < NLD; ++j) {
      unsigned char* dst = smem_raw + stage * STAGE_BYTES + (j * NW + wave) * 1024;
      __builtin_amdgcn_global_load_lds((glb_ptr_t)(src[j] + k0), (lds_ptr_t)dst, 16, 0, 0);
    }
  };

  // ---- fragment reads --------------------------------------------------------------------------------
  const int frow = lane & 31, fhalf = lane >> 5;
  const int fswz = (frow >> 2) & 3;  // block rows start at multiples of 32
  int frag_x_off[MB], frag_w_off[NB];  // byte offset of the fragment row inside a stage
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) frag_x_off[mb] = (wm * WTM + mb * 32 + frow) * (BK * 2);
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    int r;
    if (GLU) {
      constexpr int HB = NB / 2;
      int h = nb >= HB;
      r = h * BN + wn * (WTN / 2) + (h ? nb - HB : nb) * 32 + frow;
    } else {
      r = wn * WTN + nb * 32 + frow;
    }
    frag_w_off[nb] = (BM + r) * (BK * 2);
  }
  const int chunk_byte[2] = {((0 + fhalf) ^ fswz) * 16, ((2 + fhalf) ^ fswz) * 16};

  frag_t xf[2][MB], wf[2][NB];
  auto read_frags = [&](int stage, int kk, int buf) {
    const unsigned char* s = smem_raw + stage * STAGE_BYTES + chunk_byte[kk];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
      wf[buf][nb] = __builtin_bit_cast(frag_t, *reinterpret_cast<const u32x4*>(s + frag_w_off[nb]));
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
      xf[buf][mb] = __builtin_bit_cast(frag_t, *reinterpret_cast<const u32x4*>(s + frag_x_off[mb]));
  };

  f32x16 acc[NB][MB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb)
#pragma unroll
    for (int mb = 0; mb < MB; ++mb)
#pragma unroll
      for (int i = 0; i < 16; ++i) acc[nb][mb][i] = 0.f;

  auto mfma_step = [&](int buf) {
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = Mfma32<T>::run(wf[buf][nb], xf[buf][mb], acc[nb][mb]);
  };
  auto trim = [&](int kt, int kk) {                 // values past K: zeros in both operands
    const bool in = kt * BK + kk * 16 + fhalf * 8 < a.K;
    const frag_t none = {};
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) wf[kk][nb] = in ? wf[kk][nb] : none;
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) xf[kk][mb] = in ? xf[kk][mb] : none;
  };

  // ---- pipeline ----------------------------------------------------------------------------------------
#pragma unroll
  for (int kt = 0; kt < NSTAGE; ++kt) dma_tile(kt, kt);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm((NSTAGE - 1) * NLD, 0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  read_frags(0, 0, 0);

  for (int kt = 0; kt < nk; ++kt) {
    const int cur = kt & (NSTAGE - 1), nxt = (kt + 1) & (NSTAGE - 1);
    if (KTAIL && kt == nk - 1) trim(kt, 0);
    read_frags(cur, 1, 1);
    mfma_step(0);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_imm((NSTAGE - 2) * NLD, 0));
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);

    if (KTAIL && kt == nk - 1) trim(kt, 1);
    read_frags(nxt, 0, 0);
    dma_tile(kt + NSTAGE, cur);
    mfma_step(1);
#pragma unroll
    for (int i = 0; i < NMFMA; ++i) {
      __builtin_amdgcn_sched_group_barrier(SG_MFMA, 1, 0);
      __builtin_amdgcn_sched_group_barrier(SG_DS_RD, RD_PER, 0);
      __builtin_amdgcn_sched_group_barrier(SG_VMEM_RD, LD_PER, 0);
    }
    __builtin_amdgcn_sched_barrier(0);
  }
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // surplus DMA must not outlive the workgroup's LDS

  // ---- epilogue ---------------------------------------------------------------------------------
  T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    const int row = row_begin + wm * WTM + mb * 32 + frow;
    if (row >= row_end) continue;
    const int orow = a.scatter ? a.sorted_scattered[row] : row;
    T* orow_ptr = out + (size_t)orow * a.N;
    constexpr int OB = GLU ? NB / 2 : NB;
#pragma unroll
    for (int nb = 0; nb < OB; ++nb) {
      const int col0 = nt * BN + (GLU ? wn * (WTN / 2) : wn * WTN) + nb * 32 + fhalf * 4;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int col = col0 + g * 8;
        if (col >= a.N) continue;
        float v[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          if (GLU) {
            float up = acc[nb][mb][g * 4 + i];
            float gt = acc[nb + NB / 2][mb][g * 4 + i];
            v[i] = up * silu_f32(gt);
          } else {
            v[i] = acc[nb][mb][g * 4 + i];
          }
        }
        u32x2 p = {pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
        *reinterpret_cast<u32x2*>(orow_ptr + col) = p;
      }
    }
  }
}

// ---- any-shape / any-dtype fallback (one thread per output element) ------------------------------
// Used for fp32 and for shapes the tiled kernel does not take (K % 8 != 0, N % 4 != 0, unaligned
// pointers).  Correct, not fast.
template <typename T, bool GLU>
__global__ __launch_bounds__(256) void grouped_gemm_naive_kernel(GemmArgs a) {
  const int col = blockIdx.y * 64 + (threadIdx.x & 63);
  const int row = blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= a.L || col >= a.N) return;
  int expert = 0;
  while (expert < a.E - 1 && a.expert_offsets[expert] <= row) ++expert;  // (one expert: no offsets)
  const int src = a.gather ? a.sorted_scattered[row] / a.kdiv : row;
  const int orow = a.scatter ? a.sorted_scattered[row] : row;
  const T* x = static_cast<const T*>(a.in) + (size_t)src * a.K;
  const T* w = static_cast<const T*>(a.w) + ((size_t)expert * (GLU ? 2 : 1) * a.N + col) * a.K;
  float up = 0.f, gt = 0.f;
  for (int k = 0; k < a.K; ++k) {
    float xv = Elt<T>::load(x + k);
    up = fmaf(xv, Elt<T>::load(w + k), up);
    if (GLU) gt = fmaf(xv, Elt<T>::load(w + (size_t)a.N * a.K + k), gt);
  }
  float r = GLU ? up * silu_f32(gt) : up;
  Elt<T>::store(static_cast<T*>(a.out) + (size_t)orow * a.N + col, r);
}

// ---- host side ------------------------------------------------------------------------------------

template <typename T, int BM, int BNW, int WM, int WN, bool GLU, bool KTAIL, bool W8 = false>
static int launch_tiled_k(GemmArgs a, hipStream_t s) {
  constexpr int BN = GLU ? BNW / 2 : BNW;
  constexpr size_t lds = 2ull * (BM + BNW) * 128;  // two stages of 128-byte rows
  auto kern = grouped_gemm_kernel<T, BM, BNW, WM, WN, GLU, KTAIL, W8>;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> lds_ok{0};
    const int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), (int)lds, lds_ok);
    if (rc != MI_MOE_OK) return rc;
  }
  a.n_tiles = mi_ceil_div(a.N, BN);
  long max_m = (long)a.L / BM + (a.E < a.L ? a.E : a.L);
  long grid = max_m * a.n_tiles;
  grid = (grid + 7) / 8 * 8;
  if (grid > 0x7fffffffL) return MI_MOE_ESHAPE;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(WM * WN * 64), lds, s, a);
  return mi_launch_status();
}

template <typename T, int BM, int BNW, int WM, int WN, bool GLU>
static int launch_tiled(GemmArgs a, hipStream_t s) {
  if (a.K % (128 / (int)sizeof(T)) == 0) return launch_tiled_k<T, BM, BNW, WM, WN, GLU, false>(a, s);
  return launch_tiled_k<T, BM, BNW, WM, WN, GLU, true>(a, s);
}

// fp8 weights (K tiles of 64 values: 64 bytes of a weight row)
template <typename T, int BM, int BNW, int WM, int WN, bool GLU>
static int launch_tiled_w8(GemmArgs a, hipStream_t s) {
  if (a.K % 64 == 0) return launch_tiled_k<T, BM, BNW, WM, WN, GLU, false, true>(a, s);
  return launch_tiled_k<T, BM, BNW, WM, WN, GLU, true, true>(a, s);
}

template <typename T, int BM, int BNW, int WM, int WN, bool GLU, bool KTAIL>
static int launch_dma(GemmArgs a, hipStream_t s) {
  constexpr int BN = GLU ? BNW / 2 : BNW;
  constexpr size_t lds = 4ull * (BM + BNW) * 32 * sizeof(T);
  auto kern = grouped_gemm_dma_kernel<T, BM, BNW, WM, WN, GLU, KTAIL>;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> lds_ok{0};
    const int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), (int)lds, lds_ok);
    if (rc != MI_MOE_OK) return rc;
  }
  a.n_tiles = mi_ceil_div(a.N, BN);
  long max_m = (long)a.L / BM + (a.E < a.L ? a.E : a.L);
  long grid = max_m * a.n_tiles;
  grid = (grid + 7) / 8 * 8;
  if (grid > 0x7fffffffL) return MI_MOE_ESHAPE;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(WM * WN * 64), lds, s, a);
  return mi_launch_status();
}

// 128 x 128 tiles of an experts' average load
static double small_tiles(const GemmArgs& a, bool glu) {
  return (double)a.E * mi_ceil_div(mi_ceil_div(a.L, a.E), 128) * mi_ceil_div(a.N, glu ? 64 : 128);
}

// The 128 x 128 tiles of a contraction that is no multiple of 32 come by DMA as well while there is at most one to a CU.  Staged through
// registers / by DMA, us: one expert of 3001 rows, 920 -> 344 SwiGLU fp16 17.4 / 15.6 (144 tiles); 8 experts of 375, 1000 -> 392 18.3 / 16.2
// (168); 7 of 171, 472 -> 200 11.1 / 10.1 (56); but 8 of 750, 1000 -> 392 29.3 / 31.6 (336) and 17 of 188, 920 -> 520 27.5 / 28.6 (306).
// (256: the CUs these were measured on, here and below.  A choice is a function of the sizes, and is asked for without a device.)
template <typename T, bool GLU>
static int launch_128x128(const GemmArgs& a, hipStream_t s) {
  if (a.K % 32 != 0 && small_tiles(a, GLU) <= 256) return launch_dma<T, 128, 128, 2, 2, GLU, true>(a, s);
  return launch_tiled<T, 128, 128, 2, 2, GLU>(a, s);
}

// Cache policy of the persistent kernel's output stores.  The plain form's output -- the (slots, hidden) rows the
// combine streams once -- is stored non-temporal, so that it does not push the operands out of the caches.  Cached /
// non-temporal, us, down-projection alone and up + down + combine: 32 experts, 512 -> 1024, 16384 tokens 156 / 151 and 431 / 423;
// 40 experts, 512 -> 1536, 24576 tokens 314 / 308 and 889 / 881, 32768 tokens 404 / 395 and 1165 / 1148; 8 experts, 14336 -> 4096 the
// same within 1 %.  The SwiGLU form's output is the next GEMM's operand: up to about the size the memory-side cache can hold
// next to the weights it stays cached; beyond that it would not survive until it is read and only evicts the operands
// on its way.  It matters little: up + down + combine 134 MB (32 experts, 16384 tokens) 426 / 431, 134 MB (40 experts) 603 / 605,
// 235 MB (8 experts, I 14336) 2118 / 2135; 268 MB (16 experts, I 1024) 1358 / 1338, 268 MB (40 experts, 32768 tokens) 1154 / 1151,
// 470 MB 4086 / 4073.  Read by the 256 x 256 tiles' SwiGLU form and the fp8 tiles; the other forms have theirs compiled in.
static int persistent_out_nt(const GemmArgs& a, bool glu, int elt) {
  if (!glu) return 1;
  return (double)a.L * a.N * elt > 192.0 * 1024 * 1024;
}

// fp8 expert weights on tiles: out[orow(i)] = scale[e_i] * (in[irow(i)] @ Wq[e_i]^T), with SwiGLU over the [up ; gate]
// halves when glu -- the persistent kernel of persistent_fp8.hip, or the register-staged tiles for what it does not take
// and for small problems.  Called by decode_fp8.hip for batches beyond a few rows per expert (the
// streaming kernels there read an expert's weights once per 16 of its rows).  Shapes: K % 16 == 0, N % 4 == 0,
// w_tiled only with K % 128 == 0; MI_MOE_EUNSUPPORTED otherwise.
template <typename T, bool GLU>
static int dispatch_w8(const GemmArgs& a, hipStream_t s) {
  const long avg = a.E > 0 ? (long)a.L / a.E : a.L;
  if (avg >= 512) return launch_tiled_w8<T, 256, 256, 2, 2, GLU>(a, s);
  if (avg >= 48) return launch_tiled_w8<T, 128, 128, 2, 2, GLU>(a, s);
  return launch_tiled_w8<T, 32, 128, 1, 2, GLU>(a, s);
}

int mi_gemm_fp8_tiled(const void* in, const void* wq, const float* scale, void* out, const int32_t* sorted_scattered,
                      const int32_t* expert_offsets, int L, int K, int N, int E, int kdiv, int gather, int scatter,
                      int glu, int w_tiled, int dtype, int form, hipStream_t s) {
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  if (L == 0) return MI_MOE_OK;
  if (K % 16 != 0 || N % 4 != 0 || (w_tiled && K % 128 != 0)) return MI_MOE_EUNSUPPORTED;
  // 32-bit element offsets into the activations, 32-bit byte offsets inside one expert's weights
  const double in_rows = gather ? (double)L / (kdiv > 0 ? kdiv : 1) : (double)L;
  if (in_rows * K >= 2147483648.0) return MI_MOE_EUNSUPPORTED;
  const double wrows = w_tiled ? (double)mi_ceil_div(N, glu ? 16 : 32) * 32 : (double)(glu ? 2 : 1) * N;
  if (wrows * K >= 2147483648.0) return MI_MOE_EUNSUPPORTED;
  if (!mi_aligned(in, 16) || !mi_aligned(wq, 16) || !mi_aligned(scale, 16) || !mi_aligned(out, 8)) return MI_MOE_EALIGN;
  GemmArgs a;
  a.in = in; a.w = wq; a.out = out;
  a.sorted_scattered = sorted_scattered; a.expert_offsets = expert_offsets;
  a.L = L; a.K = K; a.N = N; a.E = E; a.kdiv = kdiv > 0 ? kdiv : 1; a.kshift = -1; a.n_tiles = 0;
  a.gather = gather; a.scatter = scatter; a.remap = 1; a.ws = nullptr; a.pre = nullptr; a.out_nt = 0;
  a.wscale = scale; a.w_tiled = w_tiled;
  a.out_nt = persistent_out_nt(a, glu != 0, 2);
  if (form == FP8_PERSISTENT || (form == FP8_BY_SHAPE && mi_gemm_fp8_persistent_ok(a) && mi_gemm_fp8_persistent_pick(L, K, N, E, glu != 0)))
    return mi_gemm_fp8_persistent(a, dtype, glu != 0, s);
  if (dtype == MI_MOE_BF16) return glu ? dispatch_w8<bf16_t, true>(a, s) : dispatch_w8<bf16_t, false>(a, s);
  return glu ? dispatch_w8<f16_t, true>(a, s) : dispatch_w8<f16_t, false>(a, s);
}

// workspace of the persistent kernel: one fp32 partial tile per workgroup of the largest grid
extern "C" size_t mi_moe_grouped_gemm_workspace_bytes(void) {
  int cus = 0;
  if (mi_cu_count(&cus) != MI_MOE_OK) return 0;
  return (size_t)((cus + 7) / 8 * 8) * PERSIST_WS_TILE_BYTES;
}

extern "C" int mi_moe_grouped_gemm_splits(int K, int dtype) {
  return (dtype == MI_MOE_BF16 || dtype == MI_MOE_F16) && K > 0 && K % 8 == 0 && mi_gemm_persistent_splits(K);
}

static int check_ws(const void* ws, size_t ws_bytes) {
  if (ws == nullptr) return MI_MOE_OK;
  const size_t need = mi_moe_grouped_gemm_workspace_bytes();
  if (need == 0 || ws_bytes < need) return MI_MOE_EWORKSPACE;
  return mi_aligned(ws, 16) ? MI_MOE_OK : MI_MOE_EALIGN;
}

template <typename T, bool GLU>
static int launch_naive(GemmArgs a, hipStream_t s) {
  dim3 grid(mi_ceil_div(a.L, 4), mi_ceil_div(a.N, 64));
  if (grid.y > 65535u) return MI_MOE_ESHAPE;
  hipLaunchKernelGGL((grouped_gemm_naive_kernel<T, GLU>), grid, dim3(256), 0, s, a);
  return mi_launch_status();
}

// tile configurations
//   0 / 1 / 2 / 5  register-staged 256x256 / 128x128 / 32x256 / 32x128 (any K % 8 == 0; 1 comes by DMA where K % 32 != 0 and the tiles
//              are few, see launch_128x128)
//   3          one thread per output element (any shape, any dtype)
//   4          DMA-staged 128x128, one tile per workgroup (K % 32 == 0)
//   100 + 10 rb + nw  weight stream (stream_gemm.hip): row blocks of 16 per unit, waves that split the contraction
//   7          the persistent kernel (persistent_gemm.hip; K % 8 == 0, N % 8 == 0), tiles by its rule
//   8 / 9      its 256x256 tiles with their order fixed
//   14 / 15 / 16 / 18  its even tiles (persistent_even.hip)
//   19         whichever of these the load on hand wants (persistent_load.h)
static int run_persistent(GemmArgs a, int dtype, int form, int cfg, hipStream_t s) {
  switch (cfg) {
    case 7: return mi_gemm_persistent(a, dtype, form, s);
    case 8:  // 256 x 256 tiles with their order fixed: XCDs own contiguous ranges ...
    case 9:  // ... or take consecutive blocks of one chip-wide round
      a.remap |= PERSIST_REMAP_FIXED | (cfg == 9 ? PERSIST_REMAP_INTERLEAVE : 0);
      return mi_gemm_persistent(a, dtype, form, s);
    case EVEN_256x128:
    case EVEN_160x256:
    case EVEN_224x192:
    case EVEN_256x256: return mi_gemm_even(a, dtype, form, cfg, s);
    case EVEN_BY_LOAD: return mi_gemm_persistent_ok(a) ? mi_gemm_by_load(a, dtype, form, s) : MI_MOE_EUNSUPPORTED;
    default: return MI_MOE_EUNSUPPORTED;
  }
}

template <typename T, bool GLU>
static int dispatch_cfg(GemmArgs a, int cfg, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_tiled<T, 256, 256, 2, 2, GLU>(a, s);
    case 1: return launch_128x128<T, GLU>(a, s);
    case 2: return launch_tiled<T, 32, 256, 1, 4, GLU>(a, s);
    case 5: return launch_tiled<T, 32, 128, 1, 2, GLU>(a, s);
    case 4: return a.K % 32 == 0 ? launch_dma<T, 128, 128, 2, 2, GLU, false>(a, s) : MI_MOE_EUNSUPPORTED;
    default: return run_persistent(a, std::is_same<T, bf16_t>::value ? MI_MOE_BF16 : MI_MOE_F16, GLU ? PG_SWIGLU : PG_PLAIN, cfg, s);
  }
}

// fp32 runs on the register-staged kernels only (32x32x2 matrix instructions)
template <bool GLU>
static int dispatch_cfg_f32(GemmArgs a, int cfg, hipStream_t s) {
  switch (cfg) {
    case 0: return launch_tiled<float, 256, 256, 2, 2, GLU>(a, s);
    case 1: return launch_tiled<float, 128, 128, 2, 2, GLU>(a, s);
    case 2: return launch_tiled<float, 32, 256, 1, 4, GLU>(a, s);
    case 5: return launch_tiled<float, 32, 128, 1, 2, GLU>(a, s);
    default: return MI_MOE_EUNSUPPORTED;
  }
}

// Shapes the matrix-core kernels take: 16-byte chunks along K (8 elements of a 16-bit type, 4 of fp32), four
// results per output piece, 32-bit element offsets inside one operand.
static bool tiled_shape_ok(const GemmArgs& a, int in_rows_bound, bool glu, int elt_bytes) {
  if (a.K % (16 / elt_bytes) != 0 || a.N % 4 != 0) return false;
  if ((double)in_rows_bound * a.K >= 2147483648.0) return false;
  if ((double)(glu ? 2 : 1) * a.N * a.K >= 2147483648.0) return false;
  return true;
}
static bool tiled_aligned(const GemmArgs& a, int elt_bytes) {
  return mi_aligned(a.in, 16) && mi_aligned(a.w, 16) && mi_aligned(a.out, 4 * elt_bytes);
}

// So few 256 x 256 tiles that most CUs would have none: smaller tiles give four times as many workgroups.  Measured, us,
// 256 x 256 tiles against 128 x 128: one expert (shared experts, the router's gradient) of 2048 rows, 1024 -> 1024 (SwiGLU,
// 64 tiles) 24.5 / 15.7, of 1429 rows (24 tiles) 23.3 / 12.9, of 3001 rows, 920 -> 344 fp16 (36 tiles) 23.3 / 17.0; 4096
// rows 1536 -> 512 (64 tiles) 31.6 / 20.8; but 512 -> 1536 (96 tiles) 15.6 / 16.7.
// Beyond that the 128 x 128 tiles win while they are at most one to a CU (experts chosen by random logits, cold weights, up
// projection: 24 experts of 120 rows, 1024 -> 512 (240 of them) 28.9 / 20.9; 12 experts, 2048 -> 1024 (240) 47.2 / 36.4; 6 experts,
// 4096 -> 1792 (210) 81.8 / 63.6; but 32 experts, 1024 -> 512 (320) 29.3 / 32.8 and 24 of 150 rows (384) 29.2 / 27.0, with their
// down-projections 48.2 / 46.3).  Where K is ragged, which costs the persistent tiles' DMA half lines, up to 256 of them (17.3 / 16.2,
// 16.8 / 14.7; but 17 of 188 rows, 920 -> 520 (306) 20.9 / 27.5 and back (272) 14.6 / 17.9, 8 of 750, 1000 -> 392 (336) 20.2 / 29.3 and
// back (384) 14.8 / 16.7), and for contractions below 256 while they are all resident, two to a CU.
static bool few_large_tiles(const GemmArgs& a, bool glu) {
  const int avg = (a.L + a.E - 1) / a.E;
  if (a.K % 32 != 0 && a.K >= 256) return small_tiles(a, glu) <= 256;
  if ((double)a.E * mi_ceil_div(avg, 256) * mi_ceil_div(a.N, glu ? 128 : 256) <= 72) return true;
  // (a quarter of the experts has a row tile more than the average one)
  const double small = small_tiles(a, glu);
  return a.K % 32 == 0 ? 1.25 * small <= 256 : small <= 512;
}

#define PERSIST_MIN_ROWS 120  // rows per expert on average

// The configuration for cfg -1: one of the numbers of mi_moe_scattered_gemm_cfg (100 + row blocks and waves: the weight stream).
static int pick_cfg(const GemmArgs& a, bool glu, int elt) {
  if (mi_gemm_stream_pick(a, glu, elt)) return 100 + mi_gemm_stream_form(a, glu, elt);
  const long avg = a.E > 0 ? (long)a.L / a.E : a.L;  // rows per expert if the load were uniform
  if (elt == 4) {
    // fp32 matrix instructions are slow enough that what matters is how many CUs have a tile.  Measured (up /
    // down projection, us): 128 x 128 tiles beat 256 x 256 at every size tried (262144 rows, 40 experts, hidden
    // 1536: 3240 / 1678 against 3359 / 1690; 65536 rows, 32 experts: 1136 / 585 against 1338 / 686), and below
    // about two 128 x 128 tiles per CU the 32 x 256 tiles win (the reference's correctness configuration, 1024
    // rows in 8 experts: 15 / 24 against 23 / 37; 4096 rows: 38 / 25 against 43 / 38 and, for 256 x 256, 73 / 127).
    const long tiles128 = ((long)a.L / 128 + a.E / 2 + 1) * mi_ceil_div((glu ? 2 : 1) * a.N, 128);
    return avg < 48 ? 5 : ((avg >= 512 && tiles128 >= 512) ? 1 : 2);
  }
  // (128 x 128 tiles need a second row tile, and a second pass over the weights, for the experts with more than 128 rows.
  // Persistent / 128 x 128 tiles, us, up and down projection: hidden 1536, 40 experts, 80 rows per expert 35.8 / 31.6 and
  // 23.7 / 17.8, 120 rows 38.2 / 38.8 and 22.0 / 29.7, 160 rows 37.2 / 46.1 and 20.6 / 32.0; hidden 4096, 8 experts, I 14336,
  // 100 rows 450 / 407 and 284 / 212, 130 rows 435 / 694 and 308 / 372; hidden 1024, 32 experts, 150 rows 27.0 / 26.8 and
  // 18.0 / 19.1)
  if (avg >= PERSIST_MIN_ROWS && mi_gemm_persistent_ok(a) && !few_large_tiles(a, glu)) return 7;
  if (avg >= 512 && !few_large_tiles(a, glu)) return 0;
  // A few rows per expert, just beyond the weight stream's range: many small tiles, except where the contraction is so
  // short or so long that the deeper ring of the DMA tiles wins (31 rows per expert, hidden 1536, 40 experts: layer 74 us
  // with the 32 x 128 tiles, 82 with the DMA tiles).
  if (avg < 48 && !(a.K % 32 == 0 && (a.K <= 1024 || a.K >= 8192))) return 5;
  return a.K % 32 == 0 ? 4 : 1;
}

// cfg < 0 picks a matrix-core kernel from the shape.  Nothing drops to the one-thread-per-output kernel on its own:
// a problem the matrix-core kernels cannot take is refused (MI_MOE_EALIGN for a misaligned pointer,
// MI_MOE_EUNSUPPORTED for the shape) and the caller asks for cfg 3 explicitly if it wants the slow kernel.
static int run_gemm(GemmArgs a, int dtype, bool glu, int cfg, int in_rows_bound, hipStream_t s) {
  a.out_nt = persistent_out_nt(a, glu, dtype == MI_MOE_F32 ? 4 : 2);
  if (a.L == 0) return MI_MOE_OK;
  if (dtype != MI_MOE_F32 && dtype != MI_MOE_F16 && dtype != MI_MOE_BF16) return MI_MOE_EDTYPE;
  if (cfg == 3) {
    switch (dtype) {
      case MI_MOE_F32: return glu ? launch_naive<float, true>(a, s) : launch_naive<float, false>(a, s);
      case MI_MOE_F16: return glu ? launch_naive<f16_t, true>(a, s) : launch_naive<f16_t, false>(a, s);
      default: return glu ? launch_naive<bf16_t, true>(a, s) : launch_naive<bf16_t, false>(a, s);
    }
  }
  const int elt = dtype == MI_MOE_F32 ? 4 : 2;
  if (!tiled_shape_ok(a, in_rows_bound, glu, elt)) return MI_MOE_EUNSUPPORTED;
  if (!tiled_aligned(a, elt)) return MI_MOE_EALIGN;
  if (cfg < 0) cfg = pick_cfg(a, glu, elt);
  if (cfg >= 100) return mi_gemm_stream(a, dtype, glu, cfg - 100, s);
  if (dtype == MI_MOE_F32) return glu ? dispatch_cfg_f32<true>(a, cfg, s) : dispatch_cfg_f32<false>(a, cfg, s);
  if (dtype == MI_MOE_BF16) return glu ? dispatch_cfg<bf16_t, true>(a, cfg, s) : dispatch_cfg<bf16_t, false>(a, cfg, s);
  return glu ? dispatch_cfg<f16_t, true>(a, cfg, s) : dispatch_cfg<f16_t, false>(a, cfg, s);
}

static int check_common(const void* in, const void* w, void* out, const int32_t* ss, const int32_t* off, int L, int K,
                        int N, int E, int k, int dtype, bool need_ss) {
  if (L < 0 || K < 1 || N < 1 || E < 1 || E > 65536 || k < 1) return MI_MOE_ESHAPE;
  if (dtype != MI_MOE_F32 && dtype != MI_MOE_F16 && dtype != MI_MOE_BF16) return MI_MOE_EDTYPE;
  if (L == 0) return MI_MOE_OK;
  if (!in || !w || !out || !off) return MI_MOE_ENULL;
  if (need_ss && !ss) return MI_MOE_ENULL;
  return MI_MOE_OK;
}

extern "C" int mi_moe_grouped_gemm_choice(int L, int K, int N, int E, int glu, int dtype) {
  if (L < 1 || K < 1 || N < 1 || E < 1 || E > 65536) return MI_MOE_ESHAPE;
  if (dtype != MI_MOE_F32 && dtype != MI_MOE_F16 && dtype != MI_MOE_BF16) return MI_MOE_EDTYPE;
  const int elt = dtype == MI_MOE_F32 ? 4 : 2;
  GemmArgs a = {};  // (null pointers count as aligned)
  a.L = L; a.K = K; a.N = N; a.E = E; a.kdiv = 1;
  return tiled_shape_ok(a, L, glu != 0, elt) ? pick_cfg(a, glu != 0, elt) : MI_MOE_EUNSUPPORTED;
}

int mi_gemm_one_expert(const void* in, const void* w, void* out, int L, int K, int N, bool glu, int dtype, mi_moe_stream_t stream) {
  GemmArgs a;
  a.in = in; a.w = w; a.out = out;
  a.sorted_scattered = nullptr; a.expert_offsets = nullptr;
  a.L = L; a.K = K; a.N = N; a.E = 1; a.kdiv = 1; a.n_tiles = 0;
  a.gather = 0; a.scatter = 0; a.remap = 1; a.ws = nullptr; a.pre = nullptr;
  return run_gemm(a, dtype, glu, -1, L, static_cast<hipStream_t>(stream));
}

extern "C" int mi_moe_scattered_gemm_ws(const void* in, const void* w, void* out, const int32_t* sorted_scattered,
                                        const int32_t* expert_offsets, int L, int K, int N, int E, int k,
                                        int grouped_in, int grouped_out, int dtype, int cfg, void* ws,
                                        size_t ws_bytes, mi_moe_stream_t stream) {
  int rc = check_common(in, w, out, sorted_scattered, expert_offsets, L, K, N, E, k, dtype,
                        !grouped_in || !grouped_out);
  if (rc != MI_MOE_OK) return rc;
  if ((rc = check_ws(ws, ws_bytes)) != MI_MOE_OK) return rc;
  GemmArgs a;
  a.in = in; a.w = w; a.out = out;
  a.sorted_scattered = sorted_scattered; a.expert_offsets = expert_offsets;
  a.L = L; a.K = K; a.N = N; a.E = E; a.kdiv = k; a.n_tiles = 0;
  a.gather = !grouped_in; a.scatter = !grouped_out; a.remap = 1; a.ws = ws; a.pre = nullptr;
  return run_gemm(a, dtype, false, cfg, L, static_cast<hipStream_t>(stream));
}

extern "C" int mi_moe_scattered_gemm_cfg(const void* in, const void* w, void* out, const int32_t* sorted_scattered,
                                         const int32_t* expert_offsets, int L, int K, int N, int E, int k,
                                         int grouped_in, int grouped_out, int dtype, int cfg,
                                         mi_moe_stream_t stream) {
  return mi_moe_scattered_gemm_ws(in, w, out, sorted_scattered, expert_offsets, L, K, N, E, k, grouped_in,
                                  grouped_out, dtype, cfg, nullptr, 0, stream);
}

extern "C" int mi_moe_scattered_gemm_wt_cfg(const void* in, const void* w_kn, void* out,
                                            const int32_t* sorted_scattered, const int32_t* expert_offsets, int L,
                                            int K, int N, int E, int k, int grouped_in, int grouped_out, int dtype, int cfg,
                                            void* ws, size_t ws_bytes, mi_moe_stream_t stream) {
  int rc = check_common(in, w_kn, out, sorted_scattered, expert_offsets, L, K, N, E, k, dtype,
                        !grouped_in || !grouped_out);
  if (rc != MI_MOE_OK) return rc;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  if ((rc = check_ws(ws, ws_bytes)) != MI_MOE_OK) return rc;
  if (L == 0) return MI_MOE_OK;
  GemmArgs a;
  a.in = in; a.w = w_kn; a.out = out;
  a.sorted_scattered = sorted_scattered; a.expert_offsets = expert_offsets;
  a.L = L; a.K = K; a.N = N; a.E = E; a.kdiv = k; a.n_tiles = 0;
  a.gather = !grouped_in; a.scatter = !grouped_out; a.remap = 1; a.ws = ws; a.pre = nullptr;
  if (!tiled_shape_ok(a, L, false, 2) || !mi_gemm_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
  if (!tiled_aligned(a, 2)) return MI_MOE_EALIGN;
  return run_persistent(a, dtype, PG_WEIGHT_KN, cfg < 0 ? 7 : cfg, static_cast<hipStream_t>(stream));
}

// one expert that owns every row, in place; w_kn is (K, N)
int mi_gemm_one_expert_wt(const void* in, const void* w_kn, void* out, int L, int K, int N, int dtype, mi_moe_stream_t stream) {
  GemmArgs a;
  a.in = in; a.w = w_kn; a.out = out;
  a.sorted_scattered = nullptr; a.expert_offsets = nullptr;
  a.L = L; a.K = K; a.N = N; a.E = 1; a.kdiv = 1; a.n_tiles = 0;
  a.gather = 0; a.scatter = 0; a.remap = 1; a.ws = nullptr; a.pre = nullptr;
  if (!tiled_shape_ok(a, L, false, 2) || !mi_gemm_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
  if (!tiled_aligned(a, 2)) return MI_MOE_EALIGN;
  return run_persistent(a, dtype, PG_WEIGHT_KN, 7, static_cast<hipStream_t>(stream));
}

extern "C" int mi_moe_scattered_gemm_wt_ws(const void* in, const void* w_kn, void* out,
                                           const int32_t* sorted_scattered, const int32_t* expert_offsets, int L,
                                           int K, int N, int E, int k, int grouped_in, int grouped_out, int dtype,
                                           void* ws, size_t ws_bytes, mi_moe_stream_t stream) {
  return mi_moe_scattered_gemm_wt_cfg(in, w_kn, out, sorted_scattered, expert_offsets, L, K, N, E, k, grouped_in, grouped_out,
                                      dtype, -1, ws, ws_bytes, stream);
}

extern "C" int mi_moe_scattered_gemm_wt(const void* in, const void* w_kn, void* out, const int32_t* sorted_scattered,
                                        const int32_t* expert_offsets, int L, int K, int N, int E, int k,
                                        int grouped_in, int grouped_out, int dtype, mi_moe_stream_t stream) {
  return mi_moe_scattered_gemm_wt_ws(in, w_kn, out, sorted_scattered, expert_offsets, L, K, N, E, k, grouped_in,
                                     grouped_out, dtype, nullptr, 0, stream);
}

extern "C" int mi_moe_scattered_gemm(const void* in, const void* w, void* out, const int32_t* sorted_scattered,
                                     const int32_t* expert_offsets, int L, int K, int N, int E, int k,
                                     int grouped_in, int grouped_out, int dtype, mi_moe_stream_t stream) {
  return mi_moe_scattered_gemm_cfg(in, w, out, sorted_scattered, expert_offsets, L, K, N, E, k, grouped_in,
                                   grouped_out, dtype, -1, stream);
}

extern "C" int mi_moe_up_swiglu_ws(const void* x, const void* w_fc, void* act_out, const int32_t* sorted_scattered,
                                   const int32_t* expert_offsets, int L, int H, int I, int E, int k, int dtype,
                                   int cfg, void* ws, size_t ws_bytes, mi_moe_stream_t stream) {
  int rc = check_common(x, w_fc, act_out, sorted_scattered, expert_offsets, L, H, I, E, k, dtype, true);
  if (rc != MI_MOE_OK) return rc;
  if ((rc = check_ws(ws, ws_bytes)) != MI_MOE_OK) return rc;
  GemmArgs a;
  a.in = x; a.w = w_fc; a.out = act_out;
  a.sorted_scattered = sorted_scattered; a.expert_offsets = expert_offsets;
  a.L = L; a.K = H; a.N = I; a.E = E; a.kdiv = k; a.n_tiles = 0;
  a.gather = 1; a.scatter = 0; a.remap = 1; a.ws = ws; a.pre = nullptr;
  return run_gemm(a, dtype, true, cfg, L, static_cast<hipStream_t>(stream));
}

extern "C" int mi_moe_up_swiglu_keep_cfg(const void* x, const void* w_fc, void* act_out, void* pre_out,
                                         const int32_t* sorted_scattered, const int32_t* expert_offsets, int L, int H, int I,
                                         int E, int k, int dtype, int cfg, mi_moe_stream_t stream) {
  int rc = check_common(x, w_fc, act_out, sorted_scattered, expert_offsets, L, H, I, E, k, dtype, true);
  if (rc != MI_MOE_OK) return rc;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  if (L == 0) return MI_MOE_OK;
  if (!pre_out) return MI_MOE_ENULL;
  if (!mi_aligned(pre_out, 16)) return MI_MOE_EALIGN;
  GemmArgs a;
  a.in = x; a.w = w_fc; a.out = act_out;
  a.sorted_scattered = sorted_scattered; a.expert_offsets = expert_offsets;
  a.L = L; a.K = H; a.N = I; a.E = E; a.kdiv = k; a.n_tiles = 0;
  a.gather = 1; a.scatter = 0; a.remap = 1; a.ws = nullptr; a.pre = pre_out;
  // only the persistent kernel writes the pre-activation from its accumulators: shapes it does not take, and loads of a few
  // rows per expert, are the caller's two-call path
  if (!mi_gemm_persistent_ok(a) || (cfg < 0 && (long)L / E < PERSIST_MIN_ROWS)) return MI_MOE_EUNSUPPORTED;
  if (!tiled_shape_ok(a, L, true, 2)) return MI_MOE_EUNSUPPORTED;
  if (!tiled_aligned(a, 2)) return MI_MOE_EALIGN;
  if (cfg >= 0 && I >= PERSIST_PRE_MAX_I) return MI_MOE_EUNSUPPORTED;
  if (cfg < 0 && (few_large_tiles(a, true) || I >= PERSIST_PRE_MAX_I)) {
    // too few tiles for one launch to pay: the product on its own rule, then the element-wise pass (one expert of 509 rows,
    // 1024 -> 512, 28.2 -> 16.9 us; of 4096 rows, 1536 -> 512, 37.2 -> 26.9; 17 experts of 150 rows, 920 -> 520, 37.3 -> 31.2).
    // Or rows so wide that a tile's part of the pre-activation exceeds 32-bit byte offsets
    a.out = pre_out;
    a.pre = nullptr;
    a.N = 2 * I;
    if ((rc = run_gemm(a, dtype, false, -1, L, static_cast<hipStream_t>(stream))) != MI_MOE_OK) return rc;
    return mi_moe_swiglu_forward(pre_out, act_out, L, I, dtype, stream);
  }
  return run_persistent(a, dtype, PG_SWIGLU_KEEP, cfg < 0 ? 7 : cfg, static_cast<hipStream_t>(stream));
}

extern "C" int mi_moe_up_swiglu_keep(const void* x, const void* w_fc, void* act_out, void* pre_out,
                                     const int32_t* sorted_scattered, const int32_t* expert_offsets, int L, int H, int I,
                                     int E, int k, int dtype, mi_moe_stream_t stream) {
  return mi_moe_up_swiglu_keep_cfg(x, w_fc, act_out, pre_out, sorted_scattered, expert_offsets, L, H, I, E, k, dtype, -1, stream);
}

extern "C" int mi_moe_up_swiglu_cfg(const void* x, const void* w_fc, void* act_out, const int32_t* sorted_scattered,
                                    const int32_t* expert_offsets, int L, int H, int I, int E, int k, int dtype,
                                    int cfg, mi_moe_stream_t stream) {
  return mi_moe_up_swiglu_ws(x, w_fc, act_out, sorted_scattered, expert_offsets, L, H, I, E, k, dtype, cfg, nullptr, 0,
                             stream);
}

extern "C" int mi_moe_up_swiglu(const void* x, const void* w_fc, void* act_out, const int32_t* sorted_scattered,
                                const int32_t* expert_offsets, int L, int H, int I, int E, int k, int dtype,
                                mi_moe_stream_t stream) {
  return mi_moe_up_swiglu_cfg(x, w_fc, act_out, sorted_scattered, expert_offsets, L, H, I, E, k, dtype, -1, stream);
}
