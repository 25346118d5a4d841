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
// 256 x 256 tiles / the fastest form, us, cold weights, experts with about as many rows each (SwiGLU up, then down): 40 experts, 1536 / 512: 500 tokens 37.6 ->
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

// Loads in the shape of a power law, rows of an expert ~ (place in the order)^-p: the relative rows at sixteen places.
struct LoadShapes {
  static constexpr int N = 4, PLACES = 16;
  double rows[N][PLACES];
  LoadShapes() {
    for (int n = 0; n < N; ++n) {
      double sum = 0.0;
      for (int i = 0; i < PLACES; ++i) sum += rows[n][i] = std::pow((i + 0.5) / PLACES, -0.2 * (n + 1));
      for (double& r : rows[n]) r *= PLACES / sum;
    }
  }
};
static const LoadShapes load_shapes;

// Row tiles of 160, 224 and 256 rows where L rows are spread in shape n over a.E experts (-1: normally around their average)
struct RowTiles {
  uint32_t n[3];
  uint32_t of(int i) const { return n[persist_form_rows(i) == 160 ? 0 : (persist_form_rows(i) == 224 ? 1 : 2)]; }
};
static RowTiles row_tiles_of(const GemmArgs& a, int n) {
  const double avg = (double)a.L / a.E;
  RowTiles r;
  for (int b = 0; b < 3; ++b) {
    const int bm = b == 0 ? 160 : (b == 1 ? 224 : 256);
    if (a.E == 1) {
      r.n[b] = (uint32_t)mi_ceil_div(a.L, bm);
    } else if (n < 0) {
      r.n[b] = (uint32_t)std::lround(a.E * normal_row_tiles(avg, bm));
    } else {
      long tiles = 0;
      const double per = avg / bm;
      for (const double rows : load_shapes.rows[n]) {
        const long whole = (long)(per * rows);
        tiles += whole + (per * rows > (double)whole);
      }
      r.n[b] = (uint32_t)((tiles * a.E + LoadShapes::PLACES / 2) / LoadShapes::PLACES);
    }
  }
  return r;
}
// The fastest form for so many row tiles; t: time of each
static int form_of(const GemmArgs& a, int form, int slots, const RowTiles& r, float (&t)[PERSIST_FORMS]) {
  int best = 0;
  for (int i = 0; i < PERSIST_FORMS; ++i) {
    if (form == PG_WEIGHT_KN && persist_form_blocks(i) != 8) continue;
    t[i] = persist_time(a, form, i, r.of(i), slots);
    if (t[i] < t[best]) best = i;
  }
  return best;
}

// The tiles that are the fastest, or hardly less, whatever the load, as far as the model goes: 732 of 976 problems of 64 to 6000 tokens
// in 8 to 64 experts, among them all loads of many rounds.  For the others there is pg_form_by_load, which costs a launch 0.2 us, and
// 1 us where its instructions come from memory: that is worth a loss of more than a twentieth over the loads or a fifth in one of
// them (lines at 2 % in each: 584 problems, and 0.1 % faster as far as the pick itself goes; at 12 %: 708).
int mi_gemm_tiles_of_any_load(const GemmArgs& args, int form) {
  GemmArgs a = args;
  int cus = 0;
  if (mi_cu_count(&cus) != MI_MOE_OK) return EVEN_NONE;
  if (!mi_gemm_persistent_splits(a.K)) a.ws = nullptr;
  persist_cost(a, form, cus);
  float t[PERSIST_FORMS];
  const int best = form_of(a, form, cus, row_tiles_of(a, -1), t);
  float loss = 0.0f;
  for (int n = 0; a.E > 1 && n < LoadShapes::N; ++n) {
    const int other = form_of(a, form, cus, row_tiles_of(a, n), t);
    const float more = t[best] / t[other] - 1.0f;
    loss += more;
    if (more > 0.2f || loss > 0.05f * (LoadShapes::N + 1)) return EVEN_BY_LOAD;
  }
  return persist_form_tile(best);
}

static int tile_choice(int L, int K, int N, int E, int form, bool ws) {
  if (L < 1 || K < 1 || N < 1 || E < 1 || E > PERSIST_MAX_E || form < PG_PLAIN || form > PG_WEIGHT_KN) return MI_MOE_ESHAPE;
  GemmArgs a = {};
  a.L = L; a.K = K; a.N = N; a.E = E;
  a.ws = ws && mi_gemm_persistent_splits(K) ? &a : nullptr;  // (whether there is one)
  int cus = 0;
  if (mi_cu_count(&cus) != MI_MOE_OK) return EVEN_NONE;
  persist_cost(a, form, cus);
  float t[PERSIST_FORMS];
  return persist_form_tile(form_of(a, form, cus, row_tiles_of(a, -1), t));
}

extern "C" int mi_moe_grouped_gemm_tile_choice(int L, int K, int N, int E, int form) { return tile_choice(L, K, N, E, form, false); }
extern "C" int mi_moe_grouped_gemm_tile_choice_ws(int L, int K, int N, int E, int form) { return tile_choice(L, K, N, E, form, true); }

extern "C" int mi_moe_grouped_gemm_tile_choice_load(const int32_t* ends, int K, int N, int E, int form, int ws) {
  if (K < 1 || N < 1 || E < 1 || E > PERSIST_MAX_E || form < PG_PLAIN || form > PG_WEIGHT_KN) return MI_MOE_ESHAPE;
  if (!ends) return MI_MOE_ENULL;
  GemmArgs a = {};
  a.L = ends[E - 1]; a.K = K; a.N = N; a.E = E;
  if (a.L < 1) return MI_MOE_ESHAPE;
  a.ws = ws ? &a : nullptr;
  int slots = 0;
  const int rc = by_load_prepare(a, form, &slots);
  if (rc != MI_MOE_OK) return rc;
  RowTiles r = {};
  for (int e = 0; e < E; ++e) {
    const int rows = ends[e] - (e > 0 ? ends[e - 1] : 0);
    r.n[0] += (uint32_t)mi_ceil_div(rows, 160);
    r.n[1] += (uint32_t)mi_ceil_div(rows, 224);
    r.n[2] += (uint32_t)mi_ceil_div(rows, 256);
  }
  float t[PERSIST_FORMS];
  return persist_form_tile(form_of(a, form, slots, r, t));
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
