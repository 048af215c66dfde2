// The LDS-DMA pieces shared by the MFMA GEMMs of 16-byte aligned operands:
// the persistent 256x256 kernel (gemm_pers.h: whole tiles) and the ring
// kernel (gemm_ring.h: any shape).
//
// Operands travel global -> LDS with buffer_load ... lds (LDS DMA): no
// staging registers.  K is consumed in steps of BK = 64 so that every
// K-contiguous row segment a DMA instruction fetches is one whole 128-byte
// line (with BK = 32 the L2 served twice the requests for the same bytes
// and ran 93% busy at half the needed rate).  A stage holds
//   * a K-contiguous operand as [rows][8 chunks of 8 k], 16-byte chunk
//     index XOR-swizzled by row so the ds_read_b128 of 16 consecutive rows
//     covers all banks;
//   * an M/N-contiguous operand (row-major [K,N] B, or a transposed A) as
//     [64 k][rows / 8 chunks of 8 rows], read with ds_read_b64_tr_b16, which
//     transposes 16-bit data across each 16-lane group (lane i gets element
//     i of four rows); an XOR by k keeps the rows read together on distinct
//     banks.
// A DMA instruction writes 64 lanes x 16 bytes contiguously, so the
// swizzle is applied by choosing, per lane, which global chunk to fetch.
//
// The 256x256 tile's constants below are the persistent kernel's: four
// wave64s in a 2x2 grid each own 128x128 of the output as 4x4 tiles of
// v_mfma_f32_32x32x16 (256 accumulation registers), issued with B as the
// first operand so each lane accumulates four consecutive output columns
// and the epilogue writes them with one vector store; two LDS stages of
// 64 KB.
#pragma once

#include "gemm_common.h"

namespace nova_hip {
namespace dma {

using namespace gemm;

constexpr int BM = 256, BN = 256;
#ifndef NOVA_DMA_BK
#define NOVA_DMA_BK 64
#endif
constexpr int BK = NOVA_DMA_BK;
constexpr int kChunks = BK / 8;              // 16-byte chunks per K-contiguous row
constexpr int kSlots = BM * BK / 8;          // 16-byte slots per operand per stage
constexpr int kLoads = kSlots / kThreads;    // DMA instructions per thread per operand
constexpr int kStages = 2;
// The DMA of a tile is spread over this many k16 steps (see the main loop).
#ifndef NOVA_DMA_SPREAD
#define NOVA_DMA_SPREAD 2
#endif
constexpr int kSpread = NOVA_DMA_SPREAD;
constexpr int kPerStep = (2 * kLoads + kSpread - 1) / kSpread;  // DMA loads per k16 step
constexpr int TM = 4, TN = 4;  // 32x32 tiles per wave (128 x 128)
static_assert(kStages * 2 * kSlots * 16 <= 160 * 1024, "LDS budget");
static_assert(kPerStep <= TM * TN && TM + TN <= TM * TN &&
                  kSpread <= BK / 16,
              "one DMA load and one fragment read per MFMA at most");

typedef __attribute__((address_space(3))) void lds_void;

// vmcnt(n) with expcnt and lgkmcnt left free; lgkmcnt(0) with the others
// free (gfx9 encodings).
#define NOVA_WAIT_VMCNT(n) __builtin_amdgcn_s_waitcnt((((n) & 15) | (((n) >> 4) << 14)) | 0x0F70)
#define NOVA_WAIT_LGKMCNT0() __builtin_amdgcn_s_waitcnt(0xC07F)

// Swizzles, conflict-free whether the LDS serves 8 or 16 lanes of a
// ds_read_b128 per cycle (16 or 32 lanes of a ds_read_b64_tr_b16):
//   K-contiguous: chunk c of row r at c ^ f(r)
//   M/N-contiguous: 16-byte chunk c of k-row k at c ^ (2(k&3) ^ 4(k&3))
__device__ __forceinline__ int kc_swz(int row) {
  if constexpr (kChunks == 8) return (row ^ (row >> 3)) & 7;
  else return ((row >> 1) ^ (row >> 2)) & 3;
}
__device__ __forceinline__ int kc_slot(int row, int c) { return row * kChunks + (c ^ kc_swz(row)); }
__device__ __forceinline__ int mn_swz(int k) { return ((k & 3) << 1) ^ ((k & 3) << 2); }
__device__ __forceinline__ int mn_slot(int k, int c16) { return k * 32 + (c16 ^ mn_swz(k)); }

// LDS reads as inline assembly.  Written as intrinsics or plain loads, the
// compiler assumes they may read what any in-flight LDS DMA writes and
// drains the DMA queue (vmcnt) before them; it cannot tell the two ring
// stages apart.  As assembly they are invisible to that analysis, and the
// kernel places the lgkmcnt waits for them itself.
__device__ __forceinline__ uint32_t lds_addr(const void *p) {
  return (uint32_t)(uintptr_t)(const lds_void *)p;
}
typedef uint32_t u32x2v __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u32x4 lds_read_b128(uint32_t addr) {
  u32x4 v;
  asm volatile("ds_read_b128 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}
__device__ __forceinline__ u32x2v lds_read_tr(uint32_t addr) {
  u32x2v v;
  asm volatile("ds_read_b64_tr_b16 %0, %1" : "=v"(v) : "v"(addr));
  return v;
}

__device__ __forceinline__ u32x2v lds_read_tr_hi(uint32_t addr) {
  u32x2v v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:2048" : "=v"(v) : "v"(addr));
  return v;
}
// Byte offset, from the stage base, of this lane's read of fragment
// row_base for k16-step kk (the second transposing read is 2048 bytes on).
template <bool KC>
__device__ __forceinline__ uint32_t frag_ofs(int row_base, int kk, int lane) {
  if constexpr (KC) {
    const int row = row_base + (lane & 31);
    return (uint32_t)kc_slot(row, kk * 2 + (lane >> 5)) * 16u;
  } else {
    const int g = lane >> 4, p = lane & 15;
    const int n = row_base + 16 * (g & 1) + 4 * (p & 3);
    const int kb = kk * 16 + 8 * (g >> 1) + (p >> 2);
    return (uint32_t)(mn_slot(kb, n >> 3) * 8 + (n & 7)) * 2u;
  }
}
template <bool KC>
__device__ __forceinline__ u32x4 read_frag_at(uint32_t addr) {
  if constexpr (KC) {
    return lds_read_b128(addr);
  } else {
    const u32x2v lo = lds_read_tr(addr);
    const u32x2v hi = lds_read_tr_hi(addr);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
}

}  // namespace dma
}  // namespace nova_hip
