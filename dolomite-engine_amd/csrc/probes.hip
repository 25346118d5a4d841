// Diagnostic kernels: the pieces of the persistent grouped GEMM's inner loop (persistent_gemm.hip) run in isolation, so that a
// benchmark can put measured rates of the matrix cores, the LDS and the DMA next to the grouped GEMM's figure on the same GPU in
// the same process.  Nothing in the layer calls these; they compute nothing useful.
//
// One workgroup of four waves per compute unit works through `slices` K slices, 32 wide, of a 256 x 256 bf16 tile (wave tile
// 128 x 128; per wave and slice 64 v_mfma_f32_16x16x32, sixteen 16-byte fragment reads and eight 1 KiB DMA instructions of whole
// 128-byte lines, ring of five 32 KiB units, one barrier for two slices), with parts switched off:
//   mode 0   matrix instructions only (operands read once): what the matrix cores sustain on this data at the
//            clock the chip settles at
//   mode 1   + the LDS fragment reads of every slice (no DMA: the ring keeps its first contents)
//   mode 2   DMA only: L2 -> LDS fill rate of one workgroup per CU (addresses walk an L2-resident span)
//   mode 3   everything, spread between the matrix instructions as in the GEMM
// `data` supplies the bytes (the caller chooses them: random bf16 values draw more power than zeros and lower the
// clock).  flops per slice and workgroup: 2 * 256 * 256 * 32; DMA bytes per slice and workgroup: 32 KiB.
#include "mfma_core.h"

#define PROBE_U 32768   // bytes of a ring unit
#define PROBE_LDS (5 * PROBE_U)

template <int MODE>
__global__ __launch_bounds__(256, 1) void probe_kloop_kernel(const unsigned char* __restrict__ data, uint32_t data_bytes,
                                                             uint32_t span, int slices, float* __restrict__ sink) {
  constexpr bool MM = MODE != 2, READ = MODE == 1 || MODE == 3, DMA = MODE >= 2;
  typedef __attribute__((address_space(3))) unsigned char* lds_ptr_t;
  typedef __attribute__((address_space(3))) const u32x4* frag_ptr_t;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  const uint32_t lds0 = (uint32_t)(size_t)(lds_ptr_t)smem;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave & 1, wn = wave >> 1;

  // DMA sources: instruction j of this wave fills rows 8 (4 j + wave) .. + 8 of a unit, lane -> row lane / 8, 16-byte piece
  // lane % 8 of a 128-byte line; rows 3072 bytes apart like the rows of a (tokens, 1536) matrix
  uint32_t goff[8];
  const uint32_t blk = (uint32_t)(((uint64_t)(blockIdx.x >> 3) * 7919u * 65536u) % span);
#pragma unroll
  for (int j = 0; j < 8; ++j)
    goff[j] = ((blk + (uint32_t)((4 * j + wave) * 8 + (lane >> 3)) * 3072u + (uint32_t)(lane & 7) * 16u) % span) & ~15u;
  const u32x4 srd = pg_srd(data, data_bytes);
  const uint32_t dma0 = lds0 + wave * 1024;

  // fragment reads as in the GEMM: row lane % 16 of a 16-row block, k chunk lane / 16, slot chunk ^ ((row >> 1) & 7)
  const int frow = lane & 15, fq = lane >> 4;
  const uint32_t fx = (wm * 128 + frow) * 128, fw = (wn * 128 + frow) * 128;
  const uint32_t fc0 = lds0 + ((fq ^ ((frow >> 1) & 7)) * 16), fc1 = lds0 + (((fq + 4) ^ ((frow >> 1) & 7)) * 16);
  auto read = [&](uint32_t base, int b) -> u32x4 { return *(frag_ptr_t)(size_t)(base + b * 2048); };
  u32x4 wf[2][8], xf[2][8];

  // the ring's first contents
#pragma unroll
  for (int u = 0; u < 5; ++u)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      pg_dma_dst(dma0 + u * PROBE_U, j * 4096);
      asm volatile("s_nop 0");
      pg_dma(goff[j], srd, __builtin_amdgcn_readfirstlane(u * 128));
    }
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    wf[0][i] = read(fc0 + fw + PROBE_U, i);
    xf[0][i] = read(fc0 + fx, i);
  }

  uint32_t p0 = 0, p1 = PROBE_U, p2 = 2 * PROBE_U, p3 = 3 * PROBE_U, p4 = 4 * PROBE_U;
  uint32_t rw, rx;                                  // addresses of the next slice's fragments
  auto read_bases = [&](uint32_t fc, uint32_t ps_w, uint32_t ps_x) {
    rw = fc + fw + ps_w;
    rx = fc + fx + ps_x;
    asm volatile("" : "+v"(rw), "+v"(rx));
  };
  read_bases(fc1, p1, p0);
  auto slice = [&](auto btag, auto ftag, uint32_t dst, uint32_t soff) {
    constexpr int B = decltype(btag)::value;
    constexpr int SET = READ ? B : 0;
    if constexpr (MM) pg_own_agprs();
#pragma unroll
    for (int m = 0; m < 64; ++m) {
      const int nb = m & 7, mb = m >> 3;
      if constexpr (MM && decltype(ftag)::value) pg_mfma_first<bf16_t>(m * 4, wf[SET][nb], xf[SET][mb]);
      else if constexpr (MM) pg_mfma<bf16_t>(m * 4, wf[SET][nb], xf[SET][mb]);
      if (READ && m % 2 == 0 && m < 32) {
        const int q = m / 2;
        PG_SCHED();
        if (q < 8) wf[B ^ 1][q] = read(rw, q);
        else xf[B ^ 1][q - 8] = read(rx, q - 8);
        PG_SCHED();
      }
      if (DMA && m % 8 == 1) {
        PG_SCHED();
        pg_dma_dst(dst, m / 8 * 4096);
        if (!MM) asm volatile("s_nop 0");
        PG_SCHED();
      }
      if (DMA && m % 8 == 3) {
        PG_SCHED();
        pg_dma(goff[m / 8], srd, soff);
        PG_SCHED();
      }
    }
  };
  for (int s = 0; s < slices; s += 2) {
    const uint32_t soff = __builtin_amdgcn_readfirstlane(((s >> 1) & 15) * 128);
    if (s == 0) slice(std::integral_constant<int, 0>{}, std::true_type{}, dma0 + p4, soff);
    else slice(std::integral_constant<int, 0>{}, std::false_type{}, dma0 + p4, soff);
    if (s + 1 >= slices) break;
    if constexpr (DMA) {
      __builtin_amdgcn_s_waitcnt(pg_wait(8, 0));
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      PG_SCHED();
    }
    read_bases(fc0, p3, p2);
    slice(std::integral_constant<int, 1>{}, std::false_type{}, dma0 + p0, soff);
    const uint32_t t0 = p0, t1 = p1;
    p0 = p2;
    p1 = p3;
    p2 = p4;
    p3 = t0;
    p4 = t1;
    if constexpr (MODE == 3) asm volatile("" : "+s"(p0), "+s"(p1), "+s"(p2), "+s"(p3), "+s"(p4));
    read_bases(fc1, p1, p0);
  }
  __builtin_amdgcn_s_waitcnt(pg_wait(0, 0));  // no DMA may outlive the workgroup's LDS
  float r[2] = {0.f, 0.f};
  if constexpr (MM) {
    pg_acc_settle();
#pragma unroll
    for (int i = 0; i < 256; ++i) {
      if (i % 32 == 0) pg_own_agprs();
      r[i / 128] += pg_acc(i);
    }
  } else {
    r[0] = r[1] = (float)smem[tid];
  }
  sink[(size_t)blockIdx.x * 512 + tid] = r[0];
  sink[(size_t)blockIdx.x * 512 + 256 + tid] = r[1];
}

extern "C" size_t mi_moe_probe_sink_bytes(void) {
  int cus = 0;
  if (mi_cu_count(&cus) != MI_MOE_OK) return 0;
  return (size_t)cus * 512 * sizeof(float);
}

extern "C" int mi_moe_probe_kloop(int mode, const void* data, size_t data_bytes, int slices, void* sink,
                                  size_t sink_bytes, mi_moe_stream_t stream) {
  if (mode < 0 || mode > 3 || slices < 1) return MI_MOE_ESHAPE;
  // the walk needs a span of at least the 256 rows x 3072 bytes one unit touches, plus the slice offsets
  if (data_bytes < (2u << 20) + 4096 || data_bytes >= (1ull << 32)) return MI_MOE_ESHAPE;
  if (!data || !sink) return MI_MOE_ENULL;
  if (!mi_aligned(data, 16)) return MI_MOE_EALIGN;
  int cus = 0;
  int rc = mi_cu_count(&cus);
  if (rc != MI_MOE_OK) return rc;
  if (sink_bytes < (size_t)cus * 512 * sizeof(float)) return MI_MOE_EWORKSPACE;
  const uint32_t span = (uint32_t)((data_bytes - 4096) & ~(size_t)0xffff);  // room for the slice offsets behind it
  hipStream_t s = static_cast<hipStream_t>(stream);
  const size_t lds = PROBE_LDS;
  const unsigned char* d = static_cast<const unsigned char*>(data);
  float* out = static_cast<float*>(sink);
  static std::atomic<uint64_t> lds_ok[4];
#define PROBE_LAUNCH(M)                                                                                       \
  {                                                                                                           \
    auto kern = probe_kloop_kernel<M>;                                                                        \
    if ((rc = mi_allow_lds_once(reinterpret_cast<const void*>(kern), (int)lds, lds_ok[M])) != MI_MOE_OK) return rc; \
    hipLaunchKernelGGL(kern, dim3(cus), dim3(256), lds, s, d, (uint32_t)data_bytes, span, slices, out); \
  }
  switch (mode) {
    case 0: PROBE_LAUNCH(0) break;
    case 1: PROBE_LAUNCH(1) break;
    case 2: PROBE_LAUNCH(2) break;
    default: PROBE_LAUNCH(3) break;
  }
#undef PROBE_LAUNCH
  return mi_launch_status();
}
