// MFMA GEMM / batch GEMM for gfx950: bf16 or f16 inputs, f32 accumulate,
// f32 / bf16 / f16 output, optional bias and GELU(tanh) epilogue.
//
// Replaces the NVPTX code generation of nova-gpu-optimized-pipeline for
// linalg.matmul / linalg.batch_matmul (lib/Transforms/LLVMGPU/Passes.cpp:
// 115-372: tile+distribute, pad, promote to shared memory, mma.sync,
// 3-stage cp.async).  The kernels, chosen per problem by launch_gemm_mfma:
//
//  * operands with 16-byte aligned rows: gemm_pers.h (whole 256x256 tiles)
//    or gemm_ring.h (any shape), by estimated time;
//  * unaligned rows: gemm_small.hip when the whole K of a tile fits LDS, else
//    the kernel in this file.
//
// gemm_unaligned_kernel: rows at any 2-byte alignment.  What bounded its
// predecessor was its loads, one element each.  LDS DMA cannot shift, so each
// 16-byte chunk goes through registers: the four dwords that hold its first
// byte and the dword behind them (both dword-aligned, so legal for any
// element), shifted together by the row's odd half dword.  The chunk's shift
// is the same in every K step, as a step is a multiple of four bytes in
// either layout.  Stages, swizzles and fragment reads are those of
// gemm_ring.h, two stages deep with the next step's loads in registers; tile
// 64 T x 64 T, four waves.  Edge tiles as there: rows past M or N feed only
// outputs that are not stored (the resource covers the slice, out to dword
// boundaries), k past K reads zero.
#include "gemm_ring.h"

namespace nova_hip {
namespace {

using namespace gemm;

constexpr int kBK = 64;  // K per LDS stage

struct Chunk {
  u32x4 lo;
  uint32_t hi;
};

// The 16 goes into the address (the instruction's own offset, which the range
// check counts), not into the scalar offset operand, which it need not.
__device__ __forceinline__ Chunk load_chunk(__amdgpu_buffer_rsrc_t r, uint32_t off) {
  return Chunk{__builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0),
               (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(r, off + 16u, 0, 0)};
}

// The chunk's eight elements, with only the first `left` kept.
__device__ __forceinline__ u32x4 shifted(const Chunk &c, uint32_t shift, int left) {
  u32x4 v;
#pragma unroll
  for (int d = 0; d < 4; ++d) {
    const uint32_t w = __builtin_amdgcn_alignbyte(d < 3 ? c.lo[d < 3 ? d + 1 : 3] : c.hi, c.lo[d], shift);
    v[d] = 2 * d + 1 < left ? w : 2 * d < left ? w & 0xffffu : 0u;
  }
  return v;
}

// A fragment of gemm_ring.h's stages (rows row_base + lane % 32, k16 step kk).
template <bool KC, int R>
__device__ __forceinline__ u32x4 read_frag(const char *stage, int row_base, int kk, int lane) {
  const char *p = stage + ring::frag_offset<KC, R>(row_base, kk, lane);
  if constexpr (KC) {
    return *reinterpret_cast<const u32x4 *>(p);
  } else {
    typedef __attribute__((address_space(3))) i16x4 lds_i16x4;
    const i16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)p);
    const i16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_i16x4 *)(p + 4 * R * 2));
    const u32x2 l = __builtin_bit_cast(u32x2, lo), h = __builtin_bit_cast(u32x2, hi);
    return u32x4{l[0], l[1], h[0], h[1]};
  }
}

// One operand's loads: chunk i of a thread is slot (i * 256 + tid) of the
// stage.  off: byte offset at k = 0 from the dword that holds the slice's
// first element.
template <bool KC, int R>
struct Loader {
  static constexpr int kN = R * 8 / kThreads, CH = R / 8;
  __amdgpu_buffer_rsrc_t rsrc;
  uint32_t off[kN];
  uint32_t step;
  Chunk c[kN];

  __device__ __forceinline__ static int k_of(int i) {  // the chunk's k within a step
    const int s = i * kThreads + (int)threadIdx.x;
    if constexpr (KC) {
      const int row = s >> 3;
      return ((s & 7) ^ ((row ^ (row >> 3)) & 7)) * 8;
    } else {
      return s / CH;
    }
  }
  __device__ __forceinline__ void init(const uint16_t *p, uint32_t bytes, int row0, int64_t s_outer) {
    const uint32_t mis = (uint32_t)(reinterpret_cast<uintptr_t>(p) & 2u);
    rsrc = make_rsrc(reinterpret_cast<const uint16_t *>(reinterpret_cast<uintptr_t>(p) - mis),
                     bytes ? (bytes + mis + 3u) & ~3u : 0u);
    step = KC ? kBK * 2u : (uint32_t)(kBK * s_outer * 2);
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int s = i * kThreads + (int)threadIdx.x, k = k_of(i);
      const int64_t e = KC ? (int64_t)(row0 + (s >> 3)) * s_outer + k
                           : (int64_t)k * s_outer + row0 +
                                 (((s % CH) ^ ring::line_swz<CH>(k)) * 8);
      off[i] = mis + (uint32_t)(e * 2);
    }
  }
  __device__ __forceinline__ void load(int kt, int K) {
#pragma unroll
    for (int i = 0; i < kN; ++i)
      c[i] = load_chunk(rsrc, k_of(i) < K - kt * kBK ? (off[i] & ~3u) + (uint32_t)kt * step : kOOB);
  }
  __device__ __forceinline__ void store(char *stage, int kt, int K) const {
#pragma unroll
    for (int i = 0; i < kN; ++i) {
      const int left = KC ? K - kt * kBK - k_of(i) : 8;
      reinterpret_cast<u32x4 *>(stage)[i * kThreads + threadIdx.x] = shifted(c[i], off[i] & 2u, left);
    }
  }
};

template <int DT, bool AKC, bool BKC, int T>
__global__ __launch_bounds__(kThreads) void gemm_unaligned_kernel(GemmArgs a, int vec_out) {
  constexpr int B = 64 * T, kStageA = B * kBK * 2, kStage = 2 * kStageA;
  __shared__ __attribute__((aligned(16))) char smem[2 * kStage];
  __shared__ __attribute__((aligned(16))) float bias_s[B];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int am = (wave >> 1) * 32 * T, bn = (wave & 1) * 32 * T;
  int bidx, tm, tn;
  tile_of(blockIdx.x, a, bidx, tm, tn);
  const int m0 = tm * B, n0 = tn * B;
  const bool has_bias = (a.epi == NOVA_HIP_EPI_BIAS || a.epi == NOVA_HIP_EPI_BIAS_GELU);
  const bool has_gelu = (a.epi == NOVA_HIP_EPI_BIAS_GELU || a.epi == NOVA_HIP_EPI_GELU);
  if (has_bias && tid < B) bias_s[tid] = n0 + tid < a.N ? bias_at(a.bias, a.bias_dt, n0 + tid) : 0.f;

  Loader<AKC, B> la;
  Loader<BKC, B> lb;
  la.init(a.A + (int64_t)bidx * a.sab, a.a_bytes, m0, a.sa_outer);
  lb.init(a.B + (int64_t)bidx * a.sbb, a.b_bytes, n0, a.sb_outer);

  f32x16 acc[T][T];
#pragma unroll
  for (int i = 0; i < T; ++i)
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;

  const int nk = (a.K + kBK - 1) / kBK;
  la.load(0, a.K);
  lb.load(0, a.K);
  la.store(smem, 0, a.K);
  lb.store(smem + kStageA, 0, a.K);
  la.load(1, a.K);
  lb.load(1, a.K);
  __syncthreads();
  for (int kt = 0; kt < nk; ++kt) {
    const char *cur = smem + (kt & 1) * kStage;
    char *nxt = smem + ((kt & 1) ^ 1) * kStage;
    // The step after this one, loaded a step ago, into the other stage (free
    // since the last barrier), and the loads of the one after that.
    if (kt + 1 < nk) {
      la.store(nxt, kt + 1, a.K);
      lb.store(nxt + kStageA, kt + 1, a.K);
      la.load(kt + 2, a.K);
      lb.load(kt + 2, a.K);
    }
#pragma unroll
    for (int kk = 0; kk < kBK / 16; ++kk) {
      u32x4 fa[T], fb[T];
#pragma unroll
      for (int i = 0; i < T; ++i) fa[i] = read_frag<AKC, B>(cur, am + i * 32, kk, lane);
#pragma unroll
      for (int j = 0; j < T; ++j) fb[j] = read_frag<BKC, B>(cur + kStageA, bn + j * 32, kk, lane);
#pragma unroll
      for (int i = 0; i < T; ++i)
#pragma unroll
        for (int j = 0; j < T; ++j) acc[i][j] = mfma_32x32x16<DT>(fb[j], fa[i], acc[i][j]);
    }
    __syncthreads();
  }

  char *stg = smem + wave * (32 * 32 * T * 4);
  const float *bias_w = has_bias ? bias_s + bn : nullptr;
  const int lr = lane & 31, lh = lane >> 5;
#pragma unroll
  for (int i = 0; i < T; ++i) {
#pragma unroll
    for (int j = 0; j < T; ++j)
#pragma unroll
      for (int g = 0; g < 4; ++g)
        *ring::stage_chunk<32 * T>(stg, lr, 8 * j + 2 * g + lh) = f32x4{
            acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    const int mb = m0 + am + 32 * i, nw = n0 + bn;
    const int64_t at = (int64_t)bidx * a.scb + (int64_t)mb * a.scm + nw;
    if (a.out_dt == NOVA_HIP_DT_F32)
      ring::store_f32<32, 32 * T, 64, 1>(stg, 0, lane, static_cast<float *>(a.C) + at, a.scm,
                                         a.M - mb, a.N - nw, bias_w, has_gelu);
    else
      ring::store_16<32, 32 * T, 64, 1>(stg, 0, lane, static_cast<uint16_t *>(a.C) + at, a.scm,
                                        a.M - mb, a.N - nw, vec_out, bias_w, has_gelu,
                                        a.out_dt == NOVA_HIP_DT_BF16);
  }
}

template <int DT, int T>
int32_t launch_cfg(const GemmArgs &a, int vec_out, bool akc, bool bkc, hipStream_t s) {
  const int64_t total = (int64_t)a.batch * a.tiles_m * a.tiles_n;
  if (total > 0x7fffffff) return fail(NOVA_HIP_ERANGE, "gemm: grid too large");
  const dim3 g((unsigned)total), b(kThreads);
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<DT, true, true, T>), g, b, 0, s, a, vec_out);
  else if (akc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<DT, true, false, T>), g, b, 0, s, a, vec_out);
  else if (bkc)
    hipLaunchKernelGGL((gemm_unaligned_kernel<DT, false, true, T>), g, b, 0, s, a, vec_out);
  else
    hipLaunchKernelGGL((gemm_unaligned_kernel<DT, false, false, T>), g, b, 0, s, a, vec_out);
  return check_hip(hipGetLastError(), "gemm_unaligned launch");
}

bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

}  // namespace

int32_t launch_gemm_mfma(const GemmProblem &p, hipStream_t s) {
  if (p.batch == 0 || p.M == 0 || p.N == 0) return NOVA_HIP_SUCCESS;
  if (p.M > 0x7fffffff || p.N > 0x7fffffff || p.K > 0x7fffffff)
    return fail(NOVA_HIP_ERANGE, "gemm: dimension exceeds 2^31-1");

  GemmArgs a;
  a.A = static_cast<const uint16_t *>(p.A);
  a.B = static_cast<const uint16_t *>(p.B);
  a.C = p.C;
  a.bias = p.bias;
  a.sab = p.sab;
  a.sa_outer = p.sa_outer;
  a.sbb = p.sbb;
  a.sb_outer = p.sb_outer;
  a.scb = p.scb;
  a.scm = p.scm;
  a.M = (int)p.M;
  a.N = (int)p.N;
  a.K = (int)p.K;
  a.batch = (int)p.batch;
  a.out_dt = p.out_dt;
  a.bias_dt = p.bias_dt;
  a.epi = p.epi;
  a.round = 0;

  // Byte extent of one batch slice of each operand: the buffer range the
  // kernel's loads are checked against.  Buffer offsets are 32-bit.
  const int64_t a_ext = p.a_kcontig ? (p.M - 1) * p.sa_outer + p.K : (p.K - 1) * p.sa_outer + p.M;
  const int64_t b_ext = p.b_kcontig ? (p.N - 1) * p.sb_outer + p.K : (p.K - 1) * p.sb_outer + p.N;
  if (a_ext * 2 > 0x7fffffff || b_ext * 2 > 0x7fffffff)
    return fail(NOVA_HIP_ERANGE, "gemm: an operand's batch slice exceeds 2 GiB");
  a.a_bytes = p.K > 0 ? (uint32_t)(a_ext * 2) : 0u;
  a.b_bytes = p.K > 0 ? (uint32_t)(b_ext * 2) : 0u;

  // 16-byte global loads need aligned bases, outer strides that keep every
  // row aligned, and whole 8-element chunks along the contiguous dim.
  bool vec = aligned16(p.A) && aligned16(p.B) && (p.sa_outer % 8 == 0) &&
             (p.sb_outer % 8 == 0) && (p.sab % 8 == 0) && (p.sbb % 8 == 0);
  vec = vec && (p.a_kcontig ? (p.K % 8 == 0) : (p.M % 8 == 0));
  vec = vec && (p.b_kcontig ? (p.K % 8 == 0) : (p.N % 8 == 0));

  if (vec) return launch_gemm_aligned(a, p.in_dt, p.a_kcontig, p.b_kcontig, s);
  // Rows without 16-byte alignment would cost the tiled kernel 2-byte loads;
  // with a small K the staged kernel copies them whole instead.
  if (gemm_small_applicable(a, p.a_kcontig, p.b_kcontig))
    return launch_gemm_small(a, p.in_dt, p.a_kcontig, p.b_kcontig, s);

  // 128 x 128 tiles when they fill the chip (two workgroups fit a CU), else
  // 64 x 64.
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const bool big = p.batch * ((p.M + 127) / 128) * ((p.N + 127) / 128) >= cus;
  const int t = big ? 128 : 64;
  a.tiles_m = (int)((p.M + t - 1) / t);
  a.tiles_n = (int)((p.N + t - 1) / t);
  const int vec_out = aligned16(a.C) && a.N % 8 == 0 && a.scm % 8 == 0 && a.scb % 8 == 0;
  if (p.in_dt == NOVA_HIP_DT_BF16)
    return big ? launch_cfg<NOVA_HIP_DT_BF16, 2>(a, vec_out, p.a_kcontig, p.b_kcontig, s)
               : launch_cfg<NOVA_HIP_DT_BF16, 1>(a, vec_out, p.a_kcontig, p.b_kcontig, s);
  return big ? launch_cfg<NOVA_HIP_DT_F16, 2>(a, vec_out, p.a_kcontig, p.b_kcontig, s)
             : launch_cfg<NOVA_HIP_DT_F16, 1>(a, vec_out, p.a_kcontig, p.b_kcontig, s);
}

}  // namespace nova_hip
