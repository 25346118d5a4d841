// Types shared by the grouped-GEMM kernels: the register-staged and DMA-staged tiles of grouped_gemm.hip and the
// persistent kernel of persistent_gemm.hip.
#pragma once

#include "common.h"

// Tiles picked by the load: what the experts' rows have no part in (persist_cost; with it goes n_tiles, of the first form)
struct PersistCost {
  float ends, pair;  // ns of a tile without its matrix instructions, and for a pair of row blocks and one of columns
  float per_slot;    // rounds for a tile
  uint32_t cols6;    // column tiles of tiles of 192 weight rows
};

struct GemmArgs {
  const void* in;
  const void* w;
  void* out;
  const int32_t* sorted_scattered;
  const int32_t* expert_offsets;  // null: one expert that owns all L rows
  int L;        // rows of the sorted order
  int K;        // contraction length
  int N;        // output columns (SwiGLU: I, with 2N weight rows per expert)
  int E;
  int kdiv;     // gather divisor (top-k) for scattered inputs
  int kshift;   // log2(kdiv) if kdiv is a power of two, else -1 (set by the persistent launch)
  int n_tiles;  // column tiles per row tile
  int gather;   // input row of sorted row i is sorted_scattered[i] / kdiv (else i)
  int scatter;  // output row of sorted row i is sorted_scattered[i] (else i)
  int remap;    // XCD-aware tile order
  void* ws;     // persistent kernel: workspace for splitting the last round of tiles along K (or null)
  void* pre;    // persistent SwiGLU kernel: (L, 2N) pre-activation output next to the activation (or null)
  int out_nt;   // SwiGLU on 256 x 256 tiles, fp8 persistent tiles: store the output non-temporal (persistent_out_nt)
  uint32_t out_window;  // persistent kernel: rows of the output that 32-bit byte offsets reach (set by the launch)
  // fp8 weights (register-staged kernel, W8 form): w holds e4m3fn bytes, row-major (E, rows, K) or in the streamed-tile
  // layout of decode_fp8.hip; wscale (E, rows) fp32 is applied to the accumulators in the epilogue
  // (16-bit weights: the costs in their place.  The arguments fill two lines of 64 bytes with what the compiler adds to them; a third,
  // fetched by every launch, cost 0.2 us of it)
  union {
    struct {
      const float* wscale;
      int w_tiled;
    };
    PersistCost cost;
  };
};

// ---- persistent_gemm.hip ---------------------------------------------------------------------------------------------
#define PERSIST_REMAP_INTERLEAVE 2
#define PERSIST_REMAP_FIXED 4  // the caller chose the form (cfg 8 / 9): the host does not apply its own rule
#define PERSIST_MAX_E 256
#define PERSIST_WS_TILE_BYTES (256 * 256 * 4)
#define PERSIST_PRE_MAX_I (1 << 22)  // 256 rows of a pre-activation this wide (2I elements of 16 bits) are 4 GiB

enum { PG_PLAIN = 0, PG_SWIGLU = 1, PG_SWIGLU_KEEP = 2, PG_WEIGHT_KN = 3 };
// K % 8 == 0 and N % 8 == 0, at most PERSIST_MAX_E experts, 16-byte aligned output
bool mi_gemm_persistent_ok(const GemmArgs& a);
// whether a contraction of length K can be cut along K (the only calls that use a workspace)
bool mi_gemm_persistent_splits(int K);
int mi_gemm_persistent(const GemmArgs& a, int dtype, int form, hipStream_t s);

// ---- persistent_even.hip: the same with an expert's row tiles equally high, and other tiles (rows x columns) -----------------
enum { EVEN_NONE = 0, EVEN_256x128 = 14, EVEN_160x256 = 15, EVEN_224x192 = 16, EVEN_256x256 = 18, EVEN_BY_LOAD = 19 };
// the tiles that are the fastest for this problem whatever its load, 256 x 256 (EVEN_NONE) or these, or EVEN_BY_LOAD: as it is
int mi_gemm_tiles_of_any_load(const GemmArgs& a, int form);
int mi_gemm_even(const GemmArgs& a, int dtype, int form, int tile, hipStream_t s);
int mi_gemm_even_train(const GemmArgs& a, int dtype, int form, int tile, hipStream_t s);
// ---- persistent_load.hip: those tiles or 256 x 256 ones, by the experts' rows --------------------------------------------
int mi_gemm_by_load(const GemmArgs& a, int dtype, int form, hipStream_t s);
int mi_gemm_by_load_train(const GemmArgs& a, int dtype, int form, hipStream_t s);
// the launch that adds the parts of tiles cut along K: of 8 nslot workgroups; by_load: unless even tiles were picked
int mi_gemm_split_finish(const GemmArgs& a, int dtype, int form, int nslot, bool by_load, hipStream_t s);

// ---- persistent_fp8.hip: fp8 weights (wscale, w_tiled); K % 16 == 0, K > 256, N % 8 == 0, at most PERSIST_MAX_E experts,
// 16-byte aligned output ----------------------------------------------------------------------------------------------
enum { FP8_BY_SHAPE = 1, FP8_PERSISTENT = 3, FP8_STAGED = 4 };  // forms of mi_gemm_fp8_tiled
bool mi_gemm_fp8_persistent_ok(const GemmArgs& a);
// whether they are the faster form than the register-staged tiles
bool mi_gemm_fp8_persistent_pick(int L, int K, int N, int E, bool glu);
int mi_gemm_fp8_persistent(const GemmArgs& a, int dtype, bool glu, hipStream_t s);

// ---- stream_gemm.hip: K a multiple of one 16-byte chunk, N % 4 == 0 ------------------------------------------------------
// whether the stream is the faster form for this problem (elt: bytes of an element)
bool mi_gemm_stream_pick(const GemmArgs& a, bool glu, int elt);
// form: 10 x row blocks of 16 per unit (1, 2, 4) + waves that split the contraction (1, 2, 4; row blocks 4: 1, 2); below 10: by
// the rule, which is
int mi_gemm_stream_form(const GemmArgs& a, bool glu, int elt);
int mi_gemm_stream(const GemmArgs& a, int dtype, bool glu, int form, hipStream_t s);

// ---- grouped_gemm.hip: one expert that owns every row, rows in place (no index arrays): out = in @ W^T, or with SwiGLU ------
int mi_gemm_one_expert_wt(const void* in, const void* w_kn, void* out, int L, int K, int N, int dtype, mi_moe_stream_t stream);
int mi_gemm_one_expert(const void* in, const void* w, void* out, int L, int K, int N, bool glu, int dtype, mi_moe_stream_t stream);

// end of expert e's rows
__device__ __forceinline__ int mi_expert_end(const int32_t* __restrict__ off, int L, int e) { return off ? off[e] : L; }
