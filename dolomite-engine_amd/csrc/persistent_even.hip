// The persistent grouped GEMM (persistent_gemm.hip) in forms for middling loads, where 256 x 256 tiles are padding or leave most
// of a round's CUs without one: an expert's row tiles are equally high, in steps of 32 rows, matrix instructions are left out for
// the pairs of row blocks that a low tile does not have, and there are four sizes of tiles.
//
//   tile        ring                   a slice of 64, by the matrix instructions (us at 2.1 GHz) and measured
//   256 x 256   five units of 32 KB    0.98 / 1.2     (1: 410 rows per expert, 224 high: 0.85 / 1.16)
//   160 x 256   three whole slices     0.61 / 0.90
//   224 x 192   three whole slices     0.64 / 1.0
//   256 x 128   three whole slices     0.49 / 0.78
//
// What bounds a slice beside its matrix instructions is the trip of the DMA: 0.3 us are in none of the pipes.  In the ring of
// five units activations have half a slice to land, which a low or narrow tile does not last; a ring of three whole slices gives
// them one more (8 experts, 14336 -> 4096, 1000 tokens 299 -> 247 us, 32 experts, 1024 -> 512 SwiGLU, 2048 tokens 46.5 -> 40.8).
// It fits the LDS for tiles of up to 416 rows and columns together.
//
// 256 x 256 tiles / the form the rule picks, us, cold weights (SwiGLU up, then down): 40 experts, 1536 / 512: 500 tokens 37.6 ->
// 31.6 and 19.7 -> 17.9, 1000 tokens 40.5 -> 36.8 and 21.3 -> 21.2, 2048 tokens 68.6 -> 58.8 and 34.5 -> 34.1, 4096 tokens 103.8 ->
// 99.8 and 61.5 -> 59.5; 32 experts, 1024 / 512: 509 tokens 25.8 -> 20.1 and 15.5 -> 11.8, 2048 tokens 47.5 -> 40.8 and 29.0 -> 22.2;
// 8 experts, 14336 -> 4096, 1000 tokens 307 -> 247.
#include "persistent_even.h"

#include <cmath>

// Row tiles of bm rows of an expert on average: as many experts lie beyond each multiple of bm as a normal load around avg has, with
// its square root.  Only the multiples within reach of the average are summed, so that the host's time does not grow with the load
// (summed from the first one on, three experts of 90000 rows took 9.5 us a launch, of 2^28 rows 34 ms): those 8.5 deviations below
// it count one to double precision, and where many lie within a deviation the sum is its mean.
static double normal_row_tiles(double avg, int bm) {
  const double sd = std::sqrt(avg);
  if (sd > 2.0 * bm) return avg / bm + 0.5;
  const int first = avg > 8.5 * sd ? (int)((avg - 8.5 * sd) / bm) : 0;
  double n = 1.0 + first;
  for (int j = first + 1; j * bm < avg + 4.0 * sd; ++j) n += 0.5 * std::erfc((j * bm - avg) / (sd * 1.41421356));
  return n;
}

// Time of a launch by the model below, us.  A round is a tile on every CU; a slice takes 0.35 us and 0.013 us for each 16 x 16
// block of a wave, a tile's ends 1.5 us and 0.035 us for each.  The model orders the forms above as they were measured, and is
// within a fifth of most times.  What is known here of the experts' rows is their average.
static double tile_cost(const GemmArgs& a, int form, int nb, int bm, bool even, int cus) {
  const bool glu = form == PG_SWIGLU || form == PG_SWIGLU_KEEP;
  const double avg = (double)a.L / a.E, sd = a.E > 1 ? std::sqrt(avg) : 0.0;
  const double row_tiles = a.E > 1 ? normal_row_tiles(avg, bm) : std::ceil(avg / bm);
  const int cols = mi_ceil_div(a.N, (glu ? 16 : 32) * nb);
  const double all = a.E * row_tiles * cols / cus;
  double rounds = std::ceil(all);
  // (a last round that the plan cuts along K: 8 experts, 5120 -> 4096, 1000 tokens, whose two halves it refuses, 102.6 us with the
  // credit for them, 76.4 without)
  if (!even && a.ws != nullptr && mi_gemm_persistent_splits(a.K) && form != PG_SWIGLU_KEEP && rounds > all)
    rounds += 1.0 / persist_parts(cus, (int)std::ceil((all - std::floor(all)) * cus), mi_ceil_div(a.K, PG_BK)) - 1.0;
  double pairs = bm / 32;
  if (even) pairs = std::fmax(4.0, std::fmin(pairs, std::ceil((avg + 0.5 * sd) / row_tiles / 32.0)));
  const int slices = mi_ceil_div(a.K, PG_BK) < 2 ? 2 : mi_ceil_div(a.K, PG_BK);
  return rounds * (slices * (0.35 + 0.013 * pairs * nb) + 1.5 + (form == PG_SWIGLU_KEEP ? 0.07 : 0.035) * pairs * nb);
}

int mi_gemm_even_pick(const GemmArgs& a, int form) {
  int cus = 0;
  if (mi_cu_count(&cus) != MI_MOE_OK) return EVEN_NONE;
  const struct { int tile, nb, bm; } forms[] = {{EVEN_160x256, 8, 160}, {EVEN_256x256, 8, 256}, {EVEN_224x192, 6, 224}, {EVEN_256x128, 4, 256}};
  int best = EVEN_NONE;
  double least = 0.97 * tile_cost(a, form, 8, 256, false, cus);  // (the plain form's loop has no branches)
  for (const auto& f : forms) {
    if (form == PG_WEIGHT_KN && f.nb != 8) continue;
    const double c = tile_cost(a, form, f.nb, f.bm, true, cus);
    if (c < least) {
      least = c;
      best = f.tile;
    }
  }
  return best;
}

int mi_gemm_even(const GemmArgs& a, int dtype, int form, int tile, hipStream_t s) {
  if (!mi_gemm_persistent_ok(a)) return MI_MOE_EUNSUPPORTED;
  if (dtype != MI_MOE_BF16 && dtype != MI_MOE_F16) return MI_MOE_EDTYPE;
  const bool bf = dtype == MI_MOE_BF16;
  switch (form) {
    case PG_PLAIN: return bf ? launch_even_tile<bf16_t, PG_PLAIN>(a, tile, s) : launch_even_tile<f16_t, PG_PLAIN>(a, tile, s);
    case PG_SWIGLU: return bf ? launch_even_tile<bf16_t, PG_SWIGLU>(a, tile, s) : launch_even_tile<f16_t, PG_SWIGLU>(a, tile, s);
  }
  return mi_gemm_even_train(a, dtype, form, tile, s);
}

static int tile_choice(int L, int K, int N, int E, int form, bool ws) {
  if (L < 1 || K < 1 || N < 1 || E < 1 || E > PERSIST_MAX_E || form < PG_PLAIN || form > PG_WEIGHT_KN) return MI_MOE_ESHAPE;
  GemmArgs a = {};
  a.L = L; a.K = K; a.N = N; a.E = E;
  a.ws = ws ? &a : nullptr;  // (whether there is one)
  return mi_gemm_even_pick(a, form);
}

extern "C" int mi_moe_grouped_gemm_tile_choice(int L, int K, int N, int E, int form) { return tile_choice(L, K, N, E, form, false); }
extern "C" int mi_moe_grouped_gemm_tile_choice_ws(int L, int K, int N, int E, int form) { return tile_choice(L, K, N, E, form, true); }
