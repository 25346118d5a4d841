// Grouped GEMM for a few rows per expert (generation, small batches): a stream of the touched experts' weights.
//
//   out[orow(i), :] = in[irow(i), :] @ W[e_i]^T     (+ SwiGLU), as in persistent_gemm.hip
//
// Weights are read once per row chunk, so what counts is how many bytes a CU has in flight, and at the smallest
// sizes (one token: 8 of 40 experts, 38 MB of weights) how many CUs have any.
//   * A unit is 32 weight rows (SwiGLU: 16 up, 16 gate) of one expert for a chunk of up to 16 RB of its rows.  The NW
//     waves of a workgroup split the contraction: each streams its range of K through a ring of its own -- no barrier
//     until the partial sums meet in LDS, where they are added in wave order.  Slices are whole 128-byte lines.
//   * Operands come by DMA; rows past the expert's end and values past K are lanes past the buffer: zeros, and no
//     traffic.  (The 128-row tile kernels fetch 112 copies of an expert's last row for 16 real ones.)
//   * An expert with one chunk has its weights fetched non-temporally (see decode_fp8.hip).  With several, the chunks of a
//     unit run side by side on one XCD and share the fetch through its L2: loads are uneven even when the router is not
//     (16 rows per expert on average are 10 to 22), and an expert of 200 MB read once per chunk, all its units at a time, came
//     from HBM each time.  8 experts, 4096 -> 14336, both projections, us, units innermost -> now: 64 tokens 630 -> 463 (tile
//     kernels 516), 48 tokens that all want the same two experts 332 -> 203 (240).
#include "gemm_common.h"
#include "mfma_core.h"

template <typename T> struct StreamMfma {
  static __device__ __forceinline__ f32x4 run(u32x4 w, u32x4 x, f32x4 c) {
    if constexpr (std::is_same<T, bf16_t>::value)
      return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, x), c, 0, 0, 0);
    else
      return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, w), __builtin_bit_cast(f16x8, x), c, 0, 0, 0);
  }
};
// fp32: a chunk holds four k values; lane group q = lane / 16 holds chunk q, so element i of both operands is one
// 16x16x4 product and four of them take the 16 values of four chunks
template <> struct StreamMfma<float> {
  static __device__ __forceinline__ f32x4 run(u32x4 w, u32x4 x, f32x4 c) {
    const f32x4 wv = __builtin_bit_cast(f32x4, w), xv = __builtin_bit_cast(f32x4, x);
#pragma unroll
    for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(wv[i], xv[i], c, 0, 0, 0);
    return c;
  }
};

template <bool NT> __device__ __forceinline__ void stream_dma(uint32_t lds, uint32_t off, u32x4 srd, uint32_t soff) {
  if constexpr (NT)
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen nt lds"
                 : : "s"(lds), "v"(off), "s"(srd), "s"(soff) : "memory");
  else
    asm volatile("s_mov_b32 m0, %0\n\ts_nop 0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                 : : "s"(lds), "v"(off), "s"(srd), "s"(soff) : "memory");
}

#define STREAM_STAGES 4

// ONE: some experts may have one chunk (their weights are fetched non-temporally, a branch in every slice)
template <typename T, bool GLU, int RB, int NW, bool ONE>
__global__ __launch_bounds__(NW * 64) void grouped_gemm_stream_kernel(GemmArgs a) {
  constexpr int CE = 16 / sizeof(T);                // elements of a 16-byte chunk
  constexpr int BK = 8 * CE;                        // K slice: 128 bytes of a row
  constexpr int BM = 16 * RB;
  constexpr int NX = 2 * RB, NLD = 4 + NX;          // DMA instructions of a slice (8 rows of 128 bytes each)
  constexpr int STAGE = NLD * 1024;
  constexpr int NST = STREAM_STAGES;
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int lane = threadIdx.x & 63;
  const int wave = NW > 1 ? __builtin_amdgcn_readfirstlane(threadIdx.x >> 6) : 0;
  const int frow = lane & 15, fq = lane >> 4;

  // ---- unit -> (expert, row chunk, weight rows) -----------------------------------------------------------------------
  int expert = 0, row_begin = 0, row_end = 0, nt = 0;
  bool once = true;                                 // one chunk: nobody else reads this unit's weights
  {
    // (one pass over the offsets: a lane per expert, its blocks side by side)
    const int mt = blockIdx.x / a.n_tiles;
    nt = blockIdx.x - mt * a.n_tiles;
    int carry = 0;
    bool found = false;
    for (int e0 = 0; e0 < a.E && !found; e0 += 64) {
      const int e = e0 + lane;
      const int end = e < a.E ? mi_expert_end(a.expert_offsets, a.L, e) : 0;
      const int prev = (e < a.E && e > 0) ? a.expert_offsets[e - 1] : 0;
      int incl = e < a.E ? (end - prev + BM - 1) / BM : 0;
      const int mine = incl;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(incl, o, 64);
        if (lane >= o) incl += v;
      }
      incl += carry;
      const uint64_t hit = __ballot(incl > mt);
      if (hit) {
        const int l = __ffsll((long long)hit) - 1;
        expert = e0 + l;
        row_end = __builtin_amdgcn_readlane(end, l);
        row_begin = __builtin_amdgcn_readlane(prev, l);
        const int chunks = __builtin_amdgcn_readlane(mine, l);
        if (chunks > 1) {
          once = false;
          // eight units, all their chunks, the next eight: blocks eight apart are on one XCD
          const int local = blockIdx.x - __builtin_amdgcn_readlane(incl - mine, l) * a.n_tiles;
          const int g = (local >> 3) / chunks, rem = local - g * 8 * chunks;
          const int width = a.n_tiles - 8 * g < 8 ? a.n_tiles - 8 * g : 8;
          const int chunk = width == 8 ? rem >> 3 : rem / width;
          nt = 8 * g + rem - chunk * width;
          row_begin += chunk * BM;
        }
        found = true;
      }
      carry = __builtin_amdgcn_readlane(incl, 63);
    }
    if (!found) return;                             // (the grid is the host's upper bound)
  }

  // ---- DMA sources: instruction j of a slice fills stage rows 8 j .. 8 j + 7, lane l fetches chunk
  // (l % 8) ^ ((row >> 1) & 7) of its row, the slot swizzle of persistent_gemm.hip; weights are rows 0-31 ----------------
  const int drow = lane >> 3;
  const uint32_t row_bytes = (uint32_t)a.K * (uint32_t)sizeof(T);
  const uint64_t w_total = (uint64_t)a.E * (GLU ? 2 : 1) * a.N * row_bytes;
  const uint64_t w_at = (uint64_t)expert * (GLU ? 2 : 1) * a.N * row_bytes;
  const u32x4 wsrd = pg_srd(static_cast<const unsigned char*>(a.w) + w_at, w_total - w_at);
  const u32x4 xsrd = pg_srd(a.in, (uint64_t)(a.gather ? a.L / a.kdiv : a.L) * row_bytes);
  const int odd = lane >> 4;                        // (row >> 1) & 7 of row 8 j + drow: 4 (j % 2) + drow / 2
  uint32_t xoff[NX], woff[4];
#pragma unroll
  for (int j = 0; j < NX; ++j) {
    const int r = row_begin + 8 * j + drow;
    const int s = r < row_end ? (a.gather ? a.sorted_scattered[r] / a.kdiv : r) : -1;
    xoff[j] = s < 0 ? PG_OOB : (uint32_t)s * row_bytes + (((lane & 7) ^ (4 * (j & 1) + odd)) * 16);
  }
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int r = GLU ? nt * 16 + 8 * (j & 1) + drow + (j >= 2 ? a.N : 0) : nt * 32 + 8 * j + drow;
    woff[j] = (uint32_t)r * row_bytes + (((lane & 7) ^ (4 * (j & 1) + odd)) * 16);
  }
  const int nk = (a.K + BK - 1) / BK, nfull = a.K / BK;
  const int k0 = wave * nk / NW, k1 = (wave + 1) * nk / NW, n = k1 - k0;
  const uint32_t ring = (uint32_t)(size_t)(lds_ptr_t)smem_raw + wave * (NST * STAGE);
  auto issue = [&](int i) {                         // slice k0 + i, i < n
    const int k = k0 + i;
    const uint32_t st = ring + (i % NST) * STAGE, soff = (uint32_t)k * 128u;
    if (k >= nfull) {                               // the partial last slice of the contraction: chunks past K are zeros
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const bool gone = ((lane & 7) ^ (4 * (j & 1) + odd)) * CE >= a.K - k * BK;
        stream_dma<false>(st + j * 1024, gone ? PG_OOB : woff[j], wsrd, soff);
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) {
        const bool gone = ((lane & 7) ^ (4 * (j & 1) + odd)) * CE >= a.K - k * BK;
        stream_dma<false>(st + (4 + j) * 1024, gone ? PG_OOB : xoff[j], xsrd, soff);
      }
    } else {
      if (ONE && once) {
#pragma unroll
        for (int j = 0; j < 4; ++j) stream_dma<true>(st + j * 1024, woff[j], wsrd, soff);
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) stream_dma<false>(st + j * 1024, woff[j], wsrd, soff);
      }
#pragma unroll
      for (int j = 0; j < NX; ++j) stream_dma<false>(st + (4 + j) * 1024, xoff[j], xsrd, soff);
    }
  };

  f32x4 acc[2][RB];
#pragma unroll
  for (int b = 0; b < 2; ++b)
#pragma unroll
    for (int mb = 0; mb < RB; ++mb) acc[b][mb] = (f32x4){0.f, 0.f, 0.f, 0.f};
  const uint32_t fc[2] = {(uint32_t)((fq ^ ((frow >> 1) & 7)) * 16), (uint32_t)(((fq + 4) ^ ((frow >> 1) & 7)) * 16)};
  typedef __attribute__((address_space(3))) const u32x4* frag_ptr_t;

  // what the compiler loaded (offsets, row indices) retires here, so that it waits for nothing inside the loop
#pragma unroll
  for (int j = 0; j < NX; ++j) asm volatile("" : "+v"(xoff[j]));
#pragma unroll
  for (int i = 0; i < NST - 1; ++i)
    if (i < n) issue(i);
  for (int i = 0; i < n; ++i) {
    // slices behind slice i that may stay in flight
    const int behind = n - 1 - i < NST - 2 ? n - 1 - i : NST - 2;
    if (behind == 2) __builtin_amdgcn_s_waitcnt(pg_wait(2 * NLD, 15));
    else if (behind == 1) __builtin_amdgcn_s_waitcnt(pg_wait(NLD, 15));
    else __builtin_amdgcn_s_waitcnt(pg_wait(0, 15));
    asm volatile("" ::: "memory");
    const uint32_t st = ring + (i % NST) * STAGE;
    u32x4 wf[2][2], xf[2][RB];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
#pragma unroll
      for (int b = 0; b < 2; ++b) wf[ks][b] = *(frag_ptr_t)(size_t)(st + (b * 16 + frow) * 128 + fc[ks]);
#pragma unroll
      for (int mb = 0; mb < RB; ++mb) xf[ks][mb] = *(frag_ptr_t)(size_t)(st + (32 + mb * 16 + frow) * 128 + fc[ks]);
    }
    // (slot (i - 1) % NST: read in the last round, whose products have taken its values)
    if (i + NST - 1 < n) issue(i + NST - 1);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mb = 0; mb < RB; ++mb)
#pragma unroll
        for (int b = 0; b < 2; ++b) acc[b][mb] = StreamMfma<T>::run(wf[ks][b], xf[ks][mb], acc[b][mb]);
  }

  // ---- partial sums of the waves, added in wave order; wave w finishes the row blocks w, w + NW, ... --------------------
  if constexpr (NW > 1) {
    f32x4* part = reinterpret_cast<f32x4*>(smem_raw + wave * (NST * STAGE));
    asm volatile("" ::: "memory");
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int mb = 0; mb < RB; ++mb) part[(b * RB + mb) * 64 + lane] = acc[b][mb];
    __syncthreads();
  }
  T* __restrict__ out = static_cast<T*>(a.out);
#pragma unroll
  for (int mb = 0; mb < RB; ++mb) {
    if (NW > 1 && mb % NW != wave) continue;
    f32x4 s[2];
    if constexpr (NW > 1) {
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        s[b] = reinterpret_cast<const f32x4*>(smem_raw)[(b * RB + mb) * 64 + lane];
#pragma unroll
        for (int w = 1; w < NW; ++w) {
          const f32x4 v = reinterpret_cast<const f32x4*>(smem_raw + w * (NST * STAGE))[(b * RB + mb) * 64 + lane];
#pragma unroll
          for (int i = 0; i < 4; ++i) s[b][i] += v[i];
        }
      }
    } else {
      s[0] = acc[0][mb];
      s[1] = acc[1][mb];
    }
    // register i of a lane: output column 4 (lane / 16) + i of the block, row lane % 16
    const int row = row_begin + mb * 16 + frow;
    if (row >= row_end) continue;
    T* dst = out + (size_t)(a.scatter ? a.sorted_scattered[row] : row) * a.N;
#pragma unroll
    for (int b = 0; b < (GLU ? 1 : 2); ++b) {
      const int col = GLU ? nt * 16 + fq * 4 : nt * 32 + b * 16 + fq * 4;
      if (col >= a.N) continue;
      float v[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) v[i] = GLU ? s[0][i] * silu_f32(s[1][i]) : s[b][i];
      if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4*>(dst + col) = (f32x4){v[0], v[1], v[2], v[3]};
      else *reinterpret_cast<u32x2*>(dst + col) = (u32x2){pack2<T>(v[0], v[1]), pack2<T>(v[2], v[3])};
    }
  }
}

// ---- host side ------------------------------------------------------------------------------------------------------------
template <typename T, bool GLU, int RB, int NW, bool ONE> static int launch_stream_as(GemmArgs a, hipStream_t s) {
  constexpr int lds = NW * STREAM_STAGES * (4 + 2 * RB) * 1024;
  auto kern = grouped_gemm_stream_kernel<T, GLU, RB, NW, ONE>;
  if (lds > 64 * 1024) {
    static std::atomic<uint64_t> lds_ok{0};
    const int rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), lds, lds_ok);
    if (rc != MI_MOE_OK) return rc;
  }
  a.n_tiles = mi_ceil_div(a.N, GLU ? 16 : 32);
  const long chunks = (long)a.L / (16 * RB) + (a.E < a.L ? a.E : a.L);
  const long grid = chunks * a.n_tiles;
  if (grid > 0x7fffffffL) return MI_MOE_ESHAPE;
  hipLaunchKernelGGL(kern, dim3((unsigned)grid), dim3(NW * 64), lds, s, a);
  return mi_launch_status();
}

// fp32 runs here beyond one chunk per expert on average as well, 16 bits never do: no branch for experts with one chunk (hidden 256,
// 8 experts, I 512, 512 tokens, with the division above 15.7 -> 15.0 us; 768 -> 768, 4 experts, 500 tokens 42.1 -> 40.4.  Where most have
// one the branch pays: 4096 -> 4096, 20 tokens, cold weights 222 without it, 204 with).
template <typename T, bool GLU, int RB, int NW> static int launch_stream(const GemmArgs& a, hipStream_t s) {
  if constexpr (sizeof(T) == 4)
    if ((long)a.L > 16L * RB * a.E) return launch_stream_as<T, GLU, RB, NW, false>(a, s);
  return launch_stream_as<T, GLU, RB, NW, true>(a, s);
}

template <typename T, bool GLU, int RB> static int launch_stream_nw(const GemmArgs& a, int nw, hipStream_t s) {
  switch (nw) {
    case 1: return launch_stream<T, GLU, RB, 1>(a, s);
    case 2: return launch_stream<T, GLU, RB, 2>(a, s);
    case 4:
      if constexpr (RB <= 2) return launch_stream<T, GLU, RB, 4>(a, s);
      break;  // (RB 4: four rings of 48 KB do not fit)
  }
  return MI_MOE_EUNSUPPORTED;
}

template <typename T> static int launch_stream_t(const GemmArgs& a, bool glu, int rb, int nw, hipStream_t s) {
  switch (rb) {
    case 1: return glu ? launch_stream_nw<T, true, 1>(a, nw, s) : launch_stream_nw<T, false, 1>(a, nw, s);
    case 2: return glu ? launch_stream_nw<T, true, 2>(a, nw, s) : launch_stream_nw<T, false, 2>(a, nw, s);
    case 4: return glu ? launch_stream_nw<T, true, 4>(a, nw, s) : launch_stream_nw<T, false, 4>(a, nw, s);
    default: return MI_MOE_EUNSUPPORTED;
  }
}

// Where the stream is the faster form.  Measured with cold weights, us, up / down projection, experts chosen by random logits,
// stream against the tile kernels (bf16 unless stated):
//   hidden 1536, 40 experts, I 512     1 token 7.7 / 5.8 (25.6 / 8.3), 16: 23.7 / 14.4 (33.7 / 17.4), 64: 24.4 / 15.9 (33.3 /
//                                      18.2), 96 (19 rows per expert): 28.4 (33.6), 128: 31.2 (33.6), and with Zipf(1.1) loads
//                                      34.5 (33.4)
//   hidden 1024, 32 experts, I 512     64 tokens (16 rows) 16.2 / 9.3 (17.6 / 11.2)
//   hidden 2048, 16 experts, I 1024    64 tokens (16 rows) 26.0 / 15.4 (40.0 / 17.3), 80: 27.5 (39.9)
//   hidden 4096, 8 experts, I 14336    1 token 79 / 36 (85 / 97), 64 (16 rows) 313 / 150 (333 / 184), 128: 399 / 188 (491 / 190);
//                                      192 (48 rows) 439 / 211 (375 / 194)
//   hidden 920, 17 experts, I 520 fp16 64 tokens 12.9 / 8.6 (22.1 / 14.3), 128 (30 rows) 16.5 / 9.4 (22.3 / 14.4), 200 (47 rows) 19.1 /
//                                      10.4 (24.3 / 14.8), all of them on four experts 17.7 / 11.1 (16.4 / 10.8)
//   fp32, hidden 256, 8 experts, I 512 128 tokens (32 rows) 9.3 / 6.9 (13.4 / 21.2), 512: 15.5 / 8.6 (15.3 / 23.9), 2048: 36.0 /
//                                      23.4 (37.0 / 24.5)
//   fp32, hidden 1000, 17 experts      128 tokens 43.7 / 26.3 (51.2 / 29.5), 512: 86 / 48 on the tiles, 84 / 48 on the stream
// So: up to 16 rows per expert always; up to 24 with a contraction long enough to keep the rings full, below 48 where it
// is very long, up to 56 where the tile kernels would pad a ragged one; fp32 as long as there are too few results to give
// every CU a tile.  (Weights that the memory-side cache still holds from the last call -- one layer in a loop -- favour the
// tiles: 40 experts, 80 tokens, 26.6 / 14.1 against 23.6 / 14.5.)
// Never where an operand passes the 32-bit byte offsets of the DMA (fp32 only: the general rule counts elements).
static bool stream_offsets_ok(const GemmArgs& a, bool glu, int elt) {
  const double row = (double)a.K * elt;
  return (a.gather ? a.L / a.kdiv : a.L) * row <= (double)PG_OOB && (glu ? 2.0 : 1.0) * a.N * row <= (double)PG_OOB;
}

bool mi_gemm_stream_pick(const GemmArgs& a, bool glu, int elt) {
  if (!stream_offsets_ok(a, glu, elt)) return false;
  const long rows = a.L, e = a.E;
  if (elt == 4) return rows <= 64 * e || rows * a.N <= (1L << 20);
  if (rows <= 16 * e) return true;
  if (a.K >= 4096) return rows < 48 * e;
  return a.K % 32 != 0 ? rows <= 56 * e : a.K >= 1280 && rows <= 24 * e;
}

int mi_gemm_stream_form(const GemmArgs& a, bool glu, int elt) {
  const double avg = (double)a.L / a.E;
  // row blocks: most experts in one chunk, and nearly all where a second one means long reads (13 of 16 rows on average);
  // fp32 beyond that: small chunks, whatever the load (17 experts, hidden 1000, 256 tokens, up-projection, us, 16 / 64 rows a
  // chunk: even load 54 / 45, Zipf(1.1) 53 / 67, tiles 65)
  const int rb = avg <= (elt == 2 && a.K >= 1280 ? 13 : 16) ? 1 : (avg <= (elt == 4 ? 48 : 28) ? 2 : (elt == 4 ? 1 : 4));
  // waves per unit: enough of them for the chip when there are few units (1 token: 256 units, 7.0 us with four waves
  // each, 9 with one), always four on a long contraction, two with chunks of 32 rows on a fairly long one (hidden 1536, 96
  // tokens: 33.8 -> 28.4 us)
  const int bm = 16 * rb, nk = mi_ceil_div(a.K, 128 / elt);
  const long touched = a.E < a.L ? a.E : a.L;
  const long units = touched * (long)(avg <= bm ? 1 : (avg + bm - 1) / bm) * mi_ceil_div(a.N, glu ? 16 : 32);
  int nw = (units <= 320 || (nk >= 64 && units <= 2048)) && nk >= 4 ? 4 : (units <= 640 && nk >= 4 ? 2 : 1);
  if (nw == 1 && rb == 2 && elt == 2 && nk >= 24) nw = 2;
  // (chunks of 64 rows: two rings of 48 KB cost more than they bring, 17 experts, hidden 920, 128 tokens 21.8 / 12.1 us with two
  // waves, 16.5 / 9.4 with one -- except on the very long contractions: K 14336, 128 tokens 188 / 252)
  if (rb == 4) nw = nw > 1 && nk >= 64 ? 2 : 1;
  return 10 * rb + nw;
}

int mi_gemm_stream(const GemmArgs& a, int dtype, bool glu, int form, hipStream_t s) {
  const int elt = dtype == MI_MOE_F32 ? 4 : 2;
  if (!stream_offsets_ok(a, glu, elt)) return MI_MOE_EUNSUPPORTED;
  if (form < 10) form = mi_gemm_stream_form(a, glu, elt);
  const int rb = form / 10, nw = form % 10;
  switch (dtype) {
    case MI_MOE_F32: return launch_stream_t<float>(a, glu, rb, nw, s);
    case MI_MOE_F16: return launch_stream_t<f16_t>(a, glu, rb, nw, s);
    default: return launch_stream_t<bf16_t>(a, glu, rb, nw, s);
  }
}
