// Host side of the persistent LDS-DMA GEMM (gemm_pers.h): which problems it
// takes, the round size of its tile order, and dispatch to the
// per-output-dtype translation units gemm_dma_out_{f32,bf16,f16}.hip, each
// of which instantiates the kernel for its output dtype (compiled in
// parallel).
#include "gemm_common.h"

namespace nova_hip {

namespace {
constexpr int kBM = 256, kBN = 256, kBK = 64;  // the tile of gemm_pers.h
}  // namespace

// Whole tiles, vector stores (16-byte aligned output rows) and two K steps
// or more.  Whether it is the faster kernel is choose()'s to say
// (gemm_ring.hip).
bool gemm_dma_applicable(const gemm::GemmArgs &a) {
  const int cus = device_cu_count();
  const bool c_ok = (reinterpret_cast<uintptr_t>(a.C) & 15u) == 0 && a.scm % 8 == 0 &&
                    a.scb % 8 == 0;
  return c_ok && a.M % kBM == 0 && a.N % kBN == 0 && a.K % kBK == 0 && a.K >= 2 * kBK &&
         cus > 0 && cus % 8 == 0 &&
         (int64_t)a.batch * (a.M / kBM) * (a.N / kBN) <= 0x7fffffff;
}

int32_t launch_gemm_dma(const gemm::GemmArgs &a_in, int in_dt, bool akc, bool bkc, hipStream_t s) {
  gemm::GemmArgs a = a_in;
  a.tiles_m = a.M / kBM;
  a.tiles_n = a.N / kBN;
  // 146 KB of LDS allow one workgroup per CU: a round is one workgroup per
  // CU of the current device (8 XCDs, so a multiple of 8), and the kernel
  // launches at most one round.
  a.round = device_cu_count();
  if (a.out_dt == NOVA_HIP_DT_F32) return launch_gemm_dma_f32out(a, in_dt, akc, bkc, s);
  if (a.out_dt == NOVA_HIP_DT_BF16) return launch_gemm_dma_bf16out(a, in_dt, akc, bkc, s);
  return launch_gemm_dma_f16out(a, in_dt, akc, bkc, s);
}

}  // namespace nova_hip
