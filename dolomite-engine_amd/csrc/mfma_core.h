// The pieces of the 256 x 256 matrix kernels that are written in assembly: accumulators that fill the AGPR half of the
// register file (persistent_gemm.hip, grouped_wgrad.hip), and DMA from memory to LDS.
//
// The accumulators are addressed by number.  As C++ values they would be 64 four-register tuples that fill the AGPR file
// to the last register, and the compiler moved and spilled them at every tile boundary.  To the compiler all of them are
// lost at every pg_own_agprs and pg_acc_settle: nothing of its own can live there from one of these to behind the next.
// They stand at the start of each half slice, at the end of a tile, and between the groups of accumulators that an
// epilogue reads.  Between two of them it could still place a value that lives no longer than that; what the built
// kernels do with a0 .. a255 is checked on the built code (tests/test_built_kernels.py).
#pragma once

#include "common.h"

#include <type_traits>

// Byte offset past every buffer: such a lane of the DMA writes zeros.  (A 16-bit operand of the accepted sizes, under
// 2^31 elements in whole 16-byte chunks, ends here at the latest; the range check does not wrap with the scalar offset.)
#define PG_OOB 0xfffffff0u
#define PG_SCHED() __builtin_amdgcn_sched_barrier(0)

#define ALL_AGPRS \
    "a0", "a1", "a2", "a3", "a4", "a5", "a6", "a7", "a8", "a9", "a10", "a11", "a12", "a13", "a14", "a15", \
    "a16", "a17", "a18", "a19", "a20", "a21", "a22", "a23", "a24", "a25", "a26", "a27", "a28", "a29", "a30", "a31", \
    "a32", "a33", "a34", "a35", "a36", "a37", "a38", "a39", "a40", "a41", "a42", "a43", "a44", "a45", "a46", "a47", \
    "a48", "a49", "a50", "a51", "a52", "a53", "a54", "a55", "a56", "a57", "a58", "a59", "a60", "a61", "a62", "a63", \
    "a64", "a65", "a66", "a67", "a68", "a69", "a70", "a71", "a72", "a73", "a74", "a75", "a76", "a77", "a78", "a79", \
    "a80", "a81", "a82", "a83", "a84", "a85", "a86", "a87", "a88", "a89", "a90", "a91", "a92", "a93", "a94", "a95", \
    "a96", "a97", "a98", "a99", "a100", "a101", "a102", "a103", "a104", "a105", "a106", "a107", "a108", "a109", "a110", "a111", \
    "a112", "a113", "a114", "a115", "a116", "a117", "a118", "a119", "a120", "a121", "a122", "a123", "a124", "a125", "a126", "a127", \
    "a128", "a129", "a130", "a131", "a132", "a133", "a134", "a135", "a136", "a137", "a138", "a139", "a140", "a141", "a142", "a143", \
    "a144", "a145", "a146", "a147", "a148", "a149", "a150", "a151", "a152", "a153", "a154", "a155", "a156", "a157", "a158", "a159", \
    "a160", "a161", "a162", "a163", "a164", "a165", "a166", "a167", "a168", "a169", "a170", "a171", "a172", "a173", "a174", "a175", \
    "a176", "a177", "a178", "a179", "a180", "a181", "a182", "a183", "a184", "a185", "a186", "a187", "a188", "a189", "a190", "a191", \
    "a192", "a193", "a194", "a195", "a196", "a197", "a198", "a199", "a200", "a201", "a202", "a203", "a204", "a205", "a206", "a207", \
    "a208", "a209", "a210", "a211", "a212", "a213", "a214", "a215", "a216", "a217", "a218", "a219", "a220", "a221", "a222", "a223", \
    "a224", "a225", "a226", "a227", "a228", "a229", "a230", "a231", "a232", "a233", "a234", "a235", "a236", "a237", "a238", "a239", \
    "a240", "a241", "a242", "a243", "a244", "a245", "a246", "a247", "a248", "a249", "a250", "a251", "a252", "a253", "a254", "a255"

// ---- the accumulators: a0 .. a255, addressed by number -------------------------------
// Block (nb, mb) of a wave -- 16 weight rows x 16 activation rows -- lives in a[4 (8 mb + nb) ..]: register i of a
// lane is output column 16 nb + 4 (lane / 16) + i of activation row 16 mb + lane % 16.
template <typename T> __device__ __forceinline__ void pg_mfma(int acc, u32x4 w, u32x4 x) {
  if constexpr (std::is_same<T, bf16_t>::value)
    asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, a[%0:%1]" : : "i"(acc), "i"(acc + 3), "v"(w), "v"(x));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 a[%0:%1], %2, %3, a[%0:%1]" : : "i"(acc), "i"(acc + 3), "v"(w), "v"(x));
}
// first half slice of a tile: onto zero, so that the accumulators need not be cleared
template <typename T> __device__ __forceinline__ void pg_mfma_first(int acc, u32x4 w, u32x4 x) {
  if constexpr (std::is_same<T, bf16_t>::value)
    asm volatile("v_mfma_f32_16x16x32_bf16 a[%0:%1], %2, %3, 0" : : "i"(acc), "i"(acc + 3), "v"(w), "v"(x));
  else
    asm volatile("v_mfma_f32_16x16x32_f16 a[%0:%1], %2, %3, 0" : : "i"(acc), "i"(acc + 3), "v"(w), "v"(x));
}
__device__ __forceinline__ float pg_acc(int acc) {
  float v;
  asm volatile("v_accvgpr_read_b32 %0, a[%1]" : "=v"(v) : "i"(acc));
  return v;
}
// (a wait inside the statement: the matrix instructions that wrote a register take up to 19 issue slots to do so)
__device__ __forceinline__ void pg_acc_settle() { asm volatile("s_nop 15\n\ts_nop 7" : : : "memory", ALL_AGPRS); }
__device__ __forceinline__ void pg_own_agprs() { asm volatile("" : : : "memory", ALL_AGPRS); }

// ---- DMA: M0 = LDS byte address of the wave's 1 KB piece, then 16 bytes per lane from buffer + lane offset + scalar
// offset; a lane whose offset lies past the buffer writes zeros.  Inline assembly, because the compiler makes every
// later LDS read wait for a DMA it knows of; the waits are written by hand here.
__device__ __forceinline__ void pg_dma_dst(uint32_t lds, int bytes) {
  asm volatile("s_add_u32 m0, %0, %1" : : "s"(lds), "i"(bytes) : "scc");
}
__device__ __forceinline__ void pg_dma(uint32_t off, u32x4 srd, uint32_t soff) {
  asm volatile("buffer_load_dwordx4 %0, %1, %2 offen lds" : : "v"(off), "s"(srd), "s"(soff) : "memory");
}
__device__ __forceinline__ uint32_t pg_srd_bytes(uint64_t bytes) { return bytes < (uint64_t)PG_OOB ? (uint32_t)bytes : PG_OOB; }
__device__ __forceinline__ u32x4 pg_srd(const void* base, uint64_t bytes) {
  const uint64_t b = (uint64_t)base;
  return (u32x4){(uint32_t)b, (uint32_t)(b >> 32) & 0xffffu, pg_srd_bytes(bytes), 0x00020000u};
}
__device__ __forceinline__ constexpr int pg_wait(int vm, int lgkm) {
  // gfx9 encoding: vmcnt = {imm[15:14], imm[3:0]}, expcnt = imm[6:4] (7 = no wait), lgkmcnt = imm[11:8]
  return (vm & 15) | ((vm >> 4) << 14) | (7 << 4) | ((lgkm & 15) << 8);
}
