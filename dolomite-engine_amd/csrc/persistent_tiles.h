// Which tiles a workgroup of a persistent kernel runs (persistent_gemm.hip, persistent_fp8.hip).
#pragma once

#include "gemm_common.h"

#define PERSIST_SPLIT_MAX 4
#define PERSIST_SPLIT_MIN_SAVED 60
#define PERSIST_SPLIT_MIN_SLICES 16

// Which tiles a workgroup runs.  Workgroup b sits on XCD b % 8 (the hardware deals workgroup ids round-robin to the
// XCDs) in slot b / 8.  Two ways of dealing the band-ordered tile list to them:
//   * contiguous (the default): XCD x owns the x-th eighth of the list and deals it to its slots in turn, so the
//     CUs of an XCD work on neighbouring tiles out of one L2 and an XCD stays with its experts;
//   * interleaved (PERSIST_REMAP_INTERLEAVE): round r of the whole chip is the tiles [r * grid, (r + 1) * grid), XCD
//     x taking the x-th run of grid / 8 of them.  All XCDs then work on neighbouring tiles at the same time.  When
//     an expert has more column tiles than a band is wide (intermediate size 14336: 112 column tiles, bands of 8),
//     consecutive bands read the same activation rows, and the XCDs share them through the memory-side cache
//     instead of each fetching them from HBM in its own time.
// The host asks for the second from 8 column tiles on.  Contiguous / interleaved, us: 8192 tokens, 8 experts, 14336 -> 4096 (16
// column tiles) 1524 / 1429, 4096 -> 14336 (112) 2727 / 2691; 8192 tokens, 64 experts, 4096 -> 1408 (11) 928 / 911 and back (16)
// 500 / 510; 16384 tokens, 16 experts, 2048 -> 1024 (8) 418 / 417 and back (8) 253 / 244; but below 8, where a band is the whole
// row, 512 -> 1536 (6), 40 experts, 32768 tokens 395 / 420, 16384 tokens 213 / 224, 1024 -> 512 (4), 32 experts, 4096 tokens 80 / 84,
// 1536 -> 512 (4) 335 / 340 (with an uneven load 604 / 597).
// Either way the tiles that do not fill the last round can be cut along K (see PERSIST_SPLIT_MAX).

struct SplitPlan {
  int base, stride;  // tile of this workgroup in round i < full_rounds: base + i * stride
  int full_rounds;   // rounds in which every slot has a tile
  int rem;           // tiles of the last round, the first of them being rem_base
  int rem_base;
  int parts;         // K ranges each of them is cut into (1: not split)
  int lslot;         // this workgroup's slot in the last round: part lslot / rem of tile rem_base + lslot % rem
  int ws_base;       // first partial-tile slot of the last round's tiles in the workspace
};

// K ranges that each of the `rem` tiles of a last round is cut into, on `cap` slots
__host__ __device__ inline int persist_parts(int cap, int rem, int nk) {
  int p = cap / rem;
  if (p > PERSIST_SPLIT_MAX) p = PERSIST_SPLIT_MAX;
  return p >= 2 && nk / p >= PERSIST_SPLIT_MIN_SLICES && nk - nk / p >= PERSIST_SPLIT_MIN_SAVED ? p : 1;
}

// xcd / slot of the workgroup (slot < nslot); for the finishing kernel, slot is the tile of the last round it adds up
__device__ __forceinline__ SplitPlan persist_split_plan(int total, int xcd, int slot, int nslot, int nk, bool have_ws,
                                                        bool interleave) {
  SplitPlan sp;
  int cap;  // slots that share one last round
  if (interleave) {
    cap = nslot * 8;
    sp.lslot = xcd * nslot + slot;
    sp.base = sp.lslot;
    sp.stride = cap;
    sp.full_rounds = total / cap;
    sp.rem = total - sp.full_rounds * cap;
    sp.rem_base = sp.full_rounds * cap;
    sp.ws_base = 0;
  } else {
    cap = nslot;
    const int per = (total + 7) >> 3;
    int n_x = total - xcd * per;
    n_x = n_x < 0 ? 0 : (n_x < per ? n_x : per);
    sp.lslot = slot;
    sp.base = xcd * per + slot;
    sp.stride = nslot;
    sp.full_rounds = n_x / nslot;
    sp.rem = n_x - sp.full_rounds * nslot;
    sp.rem_base = xcd * per + sp.full_rounds * nslot;
    sp.ws_base = xcd * nslot;
  }
  sp.parts = have_ws && sp.rem > 0 ? persist_parts(cap, sp.rem, nk) : 1;
  return sp;
}


// The forms of tiles of the persistent kernel (persistent_even.hip), in the order in which equally fast ones are preferred; all but
// the first are EVEN.  (Shifts of a constant: lane i of a wave asks for form i.)
#define PERSIST_FORMS 5
__host__ __device__ constexpr int persist_form_blocks(int i) { return (0x46888 >> (4 * i)) & 15; }        // nb
__host__ __device__ constexpr int persist_form_rows(int i) { return ((0x87858 >> (4 * i)) & 15) * 32; }  // bm
__host__ __device__ constexpr int persist_form_tile(int i) {
  return i == 0 ? EVEN_NONE : i == 1 ? EVEN_160x256 : i == 2 ? EVEN_256x256 : i == 3 ? EVEN_224x192 : EVEN_256x128;
}
// Time of a launch of form i with `row_tiles` row tiles of a.L rows together, ns.  A round is a tile on every slot; a slice takes
// 0.35 us and 0.013 us for each 16 x 16 block of a wave, a tile's ends 1.5 us and 0.035 us for each; the last round is as long as the
// plan's cut along K leaves it.  The model orders the forms as they were measured, and is within a fifth of most times.  Every
// workgroup of a launch, and the one that finishes its cut tiles, has to come to the same result: one rounding for each operation.
inline void persist_cost(GemmArgs& a, int form, int slots) {
#pragma clang fp contract(off)
  const float nk = a.K <= 2 * 64 ? 2.0f : (float)((a.K + 63) / 64);
  const uint32_t n = (uint32_t)a.N * (form == PG_SWIGLU || form == PG_SWIGLU_KEEP ? 2 : 1);
  a.n_tiles = (int)((n + 255) / 256);
  a.cost.ends = nk * 350.0f + 1500.0f;
  a.cost.pair = nk * 13.0f + (form == PG_SWIGLU_KEEP ? 70.0f : 35.0f);
  a.cost.per_slot = 0.9999995f / (float)slots;  // (a quotient that is whole but for its rounding is whole)
  a.cost.cols6 = (n + 191) / 192;
}
__host__ __device__ inline float persist_time(const GemmArgs& a, int form, int i, uint32_t row_tiles, int slots) {
#pragma clang fp contract(off)
  const int nb = persist_form_blocks(i);
  const uint32_t n = (uint32_t)a.N * (form == PG_SWIGLU || form == PG_SWIGLU_KEEP ? 2 : 1), L = (uint32_t)a.L;
  const uint32_t cols8 = (uint32_t)a.n_tiles, cols6 = a.cost.cols6, cols4 = (n + 127) / 128;
  const uint32_t cols = nb == 8 ? cols8 : (nb == 6 ? cols6 : cols4);
  const float ends = a.cost.ends, pair = a.cost.pair, per_slot = a.cost.per_slot;
  float rounds = ceilf((float)row_tiles * (float)cols * per_slot);
  if (__builtin_expect(a.ws != nullptr, 0)) {
    if (i == 0 && form != PG_SWIGLU_KEEP) {
      const uint32_t rem = row_tiles * cols % (uint32_t)slots;
      const int p = rem > 0 ? persist_parts(slots, (int)rem, (a.K + 63) / 64) : 1;
      if (p > 1) rounds = rounds - 1.0f + 1.0f / (float)p;
    }
  }
  // pairs of row blocks of an even tile of average height, four at least
  const uint32_t most = (uint32_t)persist_form_rows(i) / 32, m = 32 * row_tiles;
  uint32_t pairs = 4 + (L > 4 * m) + (L > 5 * m) + (L > 6 * m) + (L > 7 * m);
  pairs = i == 0 || pairs > most ? most : pairs;
  const float loop = i == 0 ? 0.97f : 1.0f;  // (the first form's loop has no branches)
  // (low tiles gained the most when SwiGLU results stopped going through LDS, 1.2 - 1.75 us a tile, the others 0.2 - 0.8: 40 experts,
  // 1536 -> 512, 3544 tokens, 160 x 256 tiles 101.7 -> 94.7 us, 256 x 256 102.7 -> 102.0; with this line the choice is 1.0 % behind the
  // fastest form over 165 loads of K 920 to 4096, 1.5 % without)
  const float low = i == 1 && form == PG_SWIGLU && a.K >= 512 ? 1500.0f : 0.0f;
  return rounds * ((ends - low + pair * (float)(pairs * (uint32_t)nb)) * loop);
}

struct PgTile {
  int expert, nt, row_begin, row_end;
};

// The tile list of one workgroup, a lane per tile (64 tiles at a time).  A lane of the four table registers holds an
// expert: row tiles of experts 0..e and the end of its rows.  An expert's tiles are numbered band by band: a band is
// up to 8 column tiles wide and runs over all of the expert's row tiles, row tile slowest.  The 32 workgroups of an
// XCD, which take 32 consecutive tiles at a time, then cover about 4 row tiles x 8 column tiles: 12 operand slabs for
// 32 tiles, and each weight slab is fetched once per band instead of once per row tile.  Up to 8 column tiles the
// band is the whole row, so that complete output rows are written at about the same time.
struct PgTable {
  int incl[4], end[4];
  int total;  // row tiles of all experts
};
// inclusive sum over the lanes of a wave
__device__ __forceinline__ int pg_wave_scan(int v) {
  v += __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true);   // row_shr 1, 2, 4, 8: rows of 16
  v += __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true);
  v += __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false);  // row_bcast 15: into rows 1 and 3
  v += __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false);  // row_bcast 31: into rows 2 and 3
  return v;
}
// A launch's arguments requested at once.  Otherwise the compiler asks for each line of them where it first needs it, one trip after
// the other: 40 experts, 1536 -> 512 SwiGLU, 2048 tokens, 160 x 256 tiles 59.5 -> 59.0 us.
__device__ __forceinline__ void pg_fetch_arguments(const GemmArgs& a) {
  asm volatile("" : : "s"(a.in), "s"(a.n_tiles), "s"(a.kdiv), "s"(a.scatter), "s"(a.out_window));
}

// Where an expert's rows begin and end, an expert to a lane of four registers
struct PgRows {
  int begin[4], end[4];
  int scan[3];  // pg_form_by_load: row tiles of 160, 224 and 256 rows of the first 64 experts, summed up to the lane's
};
__device__ __forceinline__ PgRows pg_rows(const int32_t* __restrict__ off, int L, int E) {
  const int lane = threadIdx.x & 63;
  PgRows r;
  auto load = [&](int c) {
    const int e = c * 64 + lane;
    if (e < E) r.end[c] = mi_expert_end(off, L, e);
    if (e < E && e > 0) r.begin[c] = off[e - 1];
  };
#pragma unroll
  for (int c = 0; c < 4; ++c) r.begin[c] = r.end[c] = 0;
  load(0);
  if (E > 64) {
#pragma unroll
    for (int c = 1; c < 4; ++c) load(c);
  }
  return r;
}
template <int BM, bool SCANNED = false> __device__ __forceinline__ void pg_table(const PgRows& r, int E, PgTable& tb) {
  auto tiles = [&](int c) { return pg_wave_scan((int)((uint32_t)(r.end[c] - r.begin[c] + BM - 1) / BM)); };
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    tb.incl[c] = 0;
    tb.end[c] = r.end[c];
  }
  tb.incl[0] = SCANNED ? r.scan[BM == 160 ? 0 : (BM == 224 ? 1 : 2)] : tiles(0);
  tb.total = __builtin_amdgcn_readlane(tb.incl[0], 63);
  if (E > 64) {
#pragma unroll
    for (int c = 1; c < 4; ++c) {
      tb.incl[c] = tiles(c) + tb.total;
      tb.total = __builtin_amdgcn_readlane(tb.incl[c], 63);
    }
  }
}
// The expert of a lane's row tile by binary search over the table's lanes: six exchanges, where the walk over the experts
// that this replaces took 2.2 us of a launch with 40 of them (both projections of 40 experts, 1536 / 512, 2048 tokens 112 ->
// 109 us; fp8 tiles, 64 experts, 4096 / 1408, 1024 tokens, layer 317 -> 312 us).
// EVEN: an expert's row tiles are equally high up to the last, in steps of 32 rows, and a tile ends with its own rows.
template <int BM, bool EVEN = false> __device__ __forceinline__ PgTile pg_locate(const PgTable& tb, int E, int n_tiles, int tile) {
  asm volatile("" : "+s"(n_tiles));  // (or the divisions' reciprocals stay in registers from tile to tile)
  const int q = tile / n_tiles;  // experts own contiguous tile ranges: (row tiles before) * n_tiles
  // the 64 experts that hold it, and what lies before them
  int chunk = 0, first = 0, prev = 0;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    if ((c + 1) * 64 >= E) continue;
    const int s = __builtin_amdgcn_readlane(tb.incl[c], 63), en = __builtin_amdgcn_readlane(tb.end[c], 63);
    const bool past = q >= s;
    chunk = past ? c + 1 : chunk;
    first = past ? s : first;
    prev = past ? en : prev;
  }
  auto from = [&](const int (&v)[4], int l) {
    int r = __shfl(v[0], l, 64);
#pragma unroll
    for (int c = 1; c < 4; ++c) {
      if (c * 64 >= E) continue;
      const int w = __shfl(v[c], l, 64);
      r = chunk == c ? w : r;
    }
    return r;
  };
  int l = 0;                     // the first lane whose sum exceeds q
#pragma unroll
  for (int step = 32; step > 0; step >>= 1) l += from(tb.incl, l + step - 1) <= q ? step : 0;
  const int incl = from(tb.incl, l), rend = from(tb.end, l);
  const int before = l > 0 ? l - 1 : 0;
  const int s = from(tb.incl, before), en = from(tb.end, before);
  first = l > 0 ? s : first;
  prev = l > 0 ? en : prev;
  const int tile_band = n_tiles < 8 ? n_tiles : 8;
  const int local = tile - first * n_tiles, per_band = (incl - first) * tile_band;
  const int band = local / per_band;
  const int rem = local - band * per_band;
  const int left = n_tiles - band * tile_band;
  const int width = left < tile_band ? left : tile_band;
  const int mt = rem / width;
  PgTile t;
  t.expert = chunk * 64 + l;
  t.nt = band * tile_band + rem - mt * width;
  if (EVEN) {
    const int n = incl - first, h = (rend - prev + 32 * n - 1) / (32 * n) * 32;
    t.row_begin = prev + mt * h;
    t.row_end = t.row_begin + h < rend ? t.row_begin + h : rend;
  } else {
    t.row_begin = prev + mt * BM;
    t.row_end = rend;
  }
  return t;
}
// The form that is the fastest for the experts' rows as they are: lane i has form i.  This is a chain in front of the launch's
// first load, and its instructions come from memory where a layer's weights have gone through the caches, so it is kept short: no
// division, no branch, what is the load's only, and the sums are the tile table's too.  Whole numbers of 64 bits and a branch for every
// choice took 0.8 us of a launch, floats with the host's part among them 0.4, this 0.2; with cold caches the last two 1.1 - 1.5 and
// 0 - 1.6.
__device__ __forceinline__ int pg_form_by_load(const GemmArgs& a, PgRows& r, int form, int slots) {
  const int lane = threadIdx.x & 63;
  uint32_t n[3];
  auto tiles = [&](int c, int b) {
    const uint32_t rows = (uint32_t)(r.end[c] - r.begin[c]);
    return b == 0 ? (rows + 159) / 160 : (b == 1 ? (rows + 223) / 224 : (rows + 255) / 256);
  };
#pragma unroll
  for (int b = 0; b < 3; ++b) {
    r.scan[b] = pg_wave_scan((int)tiles(0, b));
    n[b] = (uint32_t)__builtin_amdgcn_readlane(r.scan[b], 63);
  }
  if (__builtin_expect(a.E > 64, 0)) {
#pragma unroll
    for (int b = 0; b < 3; ++b)
      n[b] += (uint32_t)__builtin_amdgcn_readlane(pg_wave_scan((int)(tiles(1, b) + tiles(2, b) + tiles(3, b))), 63);
  }
  const int i = lane < PERSIST_FORMS ? lane : 0, bm = persist_form_rows(i);
  const float t = persist_time(a, form, i, bm == 160 ? n[0] : (bm == 224 ? n[1] : n[2]), slots);
  int best = 0;
  uint32_t least = 0;  // (positive floats are ordered as their bits)
#pragma unroll
  for (int j = 0; j < PERSIST_FORMS; ++j) {
    if (form == PG_WEIGHT_KN && persist_form_blocks(j) != 8) continue;
    const uint32_t tj = (uint32_t)__builtin_amdgcn_readlane((int)__float_as_uint(t), j);
    if (j == 0 || tj < least) {
      least = tj;
      best = j;
    }
  }
  return __builtin_amdgcn_readfirstlane(best);
}
// pairs of 16-row blocks of a tile
__device__ __forceinline__ int pg_row_pairs(const PgTile& t) { return (t.row_end - t.row_begin + 31) >> 5; }
