// f32 GEMM on the matrix cores: products and sums carry f32 precision, but
// the accumulation order is the MFMA's and the tile loop's, not the
// reference's sequential k.  The result is therefore not bit-identical to
// Nova's CPU pipeline (the exact kernel in gemm_f32.hip is), but it is within
// the f32 parity bar (1e-4 relative): the error is the ordinary rounding of
// an f32 dot product.  It is what a GPU lowering of an f32 linalg.matmul
// would run (the reference's NVPTX path uses tf32 mma.sync, which is not
// within 1e-4); a caller opts in with NOVA_HIP_GEMM_F32_MFMA.
//
// The kernel is gemm_f32_split.h (each f32 value as three bf16 values, on
// the bf16 MFMA).  This file chooses its tile form and the number of K
// splits, and adds the splits' partial sums in split order, so the result is
// the same on every run.
//
// Against v_mfma_f32_32x32x2_f32 in 128 x 128 tiles, us on one MI355X:
// 8192 x 50304 x 384 2649 -> 1678, 8192 x 384 x 50304 2414 -> 1549,
// 384 x 50304 x 8192 2543 -> 1602, 8192 x 1536 x 384 87 -> 57,
// 384 x 1536 x 8192 141 -> 69, 2000 x 50304 x 32 137 -> 124, 256^3 24.1 -> 10.0.
#include "gemm_f32_split.h"

namespace nova_hip {
namespace split {
namespace {

// Measured on one MI355X (us): `step`, one 32-deep K step of a workgroup
// alone on its CU with the chip full; `more`, what each further workgroup on
// the CU adds; `fixed`, a unit's start and outputs.  Fitted to 120 shapes (K
// from 32 to 2000, 1 to 6300 tiles) run on every form in one split: the form
// of least estimate is within 0.4% of the best of the six in the geometric
// mean and 7% at worst.
constexpr Form kForm[kForms] = {
    {4, 3, 2, 1, 3.58f, 0.0f, 8.8f},   // 256 x 192
    {3, 4, 2, 1, 3.85f, 0.0f, 7.4f},   // 192 x 256
    {3, 3, 2, 1, 3.05f, 0.0f, 6.0f},   // 192 x 192
    {4, 2, 2, 1, 2.64f, 0.0f, 10.9f},  // 256 x 128
    {2, 2, 2, 2, 1.27f, 1.44f, 4.8f},  // 128 x 128
    {1, 1, 3, 3, 0.68f, 0.38f, 2.9f},  // 64 x 64
};

// The chunks that a split's sum is taken in.
int chunks_of(const SplitArgs &a, int sp) { return (int)((min_parts(a.K) + sp - 1) / sp); }

int64_t tiles_of(const SplitArgs &a, const Form &f) {
  const int64_t bm = 64 * f.tm, bn = 64 * f.tn;
  return a.batch * ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
}

// Estimated time with K in sp splits: rounds of resident workgroups (the
// last, partial one and a chip that is not full run their steps up to 30%
// faster where a workgroup has its CU to itself), each chunk of a tile a unit
// with a start and outputs of its own, and, with splits, the partials' traffic
// and the second launch.
float estimate(const SplitArgs &a, const Form &f, int sp, int cus) {
  const float q = (float)tiles_of(a, f) * sp / cus;
  const int nk = (a.K + BK - 1) / BK, steps = (nk + sp - 1) / sp;
  float step, rounds = 1.0f;
  if (q <= 1.0f) {
    step = f.step * (f.per_cu == 1 ? 0.7f + 0.3f * q : 1.0f);
  } else if (q <= f.per_cu) {
    step = f.step + f.more * (ceilf(q) - 1.0f);
  } else {
    step = f.step + f.more * (f.per_cu - 1);
    const float r = q / f.per_cu, whole = floorf(r), part = r - whole;
    rounds = f.per_cu > 1 ? r + 0.25f : part > 0.0f ? whole + 0.7f + 0.3f * part : whole;
  }
  float us = rounds * (steps * step + chunks_of(a, sp) * f.fixed);
  if (sp > 1) us += 4.0f + (2 * sp + 1) * (4.0f * a.batch * a.M * a.N) / 6e6f;
  return us;
}

typedef float f32x4u1 __attribute__((ext_vector_type(4), aligned(4)));

// C = epilogue(sum of the split partials, in split order), W columns of a
// row per thread (W = 4 where N is a multiple of 4).
template <int W>
__global__ __launch_bounds__(256) void split_reduce_kernel(const float *part, int splits,
                                                           int64_t per_split, int M, int N,
                                                           float *C, int64_t scb, int64_t scm,
                                                           int gelu) {
  const int64_t i = ((int64_t)blockIdx.x * 256 + threadIdx.x) * W;
  if (i >= per_split) return;
  float s[W];
#pragma unroll
  for (int e = 0; e < W; ++e) s[e] = 0.0f;
  for (int k = 0; k < splits; ++k) {
    const float *p = part + k * per_split + i;
    if constexpr (W == 4) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(p);
#pragma unroll
      for (int e = 0; e < 4; ++e) s[e] = k ? s[e] + v[e] : v[e];
    } else {
      s[0] = k ? s[0] + p[0] : p[0];
    }
  }
  if (gelu) {
#pragma unroll
    for (int e = 0; e < W; ++e) s[e] = gelu_tanh(s[e]);
  }
  const int64_t mn = (int64_t)M * N;
  const int64_t b = i / mn;
  const int64_t r = i - b * mn;
  const int64_t m = r / N, n = r - m * N;
  float *dst = C + b * scb + m * scm + n;
  if constexpr (W == 4) *reinterpret_cast<f32x4u1 *>(dst) = f32x4{s[0], s[1], s[2], s[3]};
  else dst[0] = s[0];
}

}  // namespace
}  // namespace split

int32_t launch_gemm_f32_mfma(const GemmProblem &p, hipStream_t s) {
  using namespace split;
  if (p.batch == 0 || p.M == 0 || p.N == 0) return NOVA_HIP_SUCCESS;
  if (p.M > 0x7fffffff || p.N > 0x7fffffff || p.K > 0x7fffffff || p.batch > 0x7fffffff)
    return fail(NOVA_HIP_ERANGE, "gemm_f32_mfma: dimension exceeds 2^31-1");
  if (p.out_dt != NOVA_HIP_DT_F32 || p.in_dt != NOVA_HIP_DT_F32)
    return fail(NOVA_HIP_EDTYPE, "gemm_f32_mfma: f32 inputs and output only");
  SplitArgs a;
  a.A = static_cast<const float *>(p.A);
  a.B = static_cast<const float *>(p.B);
  a.C = static_cast<float *>(p.C);
  a.bias = p.bias;
  a.part = nullptr;
  a.sab = p.sab;
  a.sa_outer = p.sa_outer;
  a.sbb = p.sbb;
  a.sb_outer = p.sb_outer;
  a.scb = p.scb;
  a.scm = p.scm;
  // Byte extent of one batch slice of each operand (the buffer range).
  const int64_t a_ext = p.K == 0 ? 0 : p.a_kcontig ? (p.M - 1) * p.sa_outer + p.K
                                                   : (p.K - 1) * p.sa_outer + p.M;
  const int64_t b_ext = p.K == 0 ? 0 : p.b_kcontig ? (p.N - 1) * p.sb_outer + p.K
                                                   : (p.K - 1) * p.sb_outer + p.N;
  if (a_ext * 4 > 0x7fffffff || b_ext * 4 > 0x7fffffff)
    return fail(NOVA_HIP_ERANGE, "gemm_f32_mfma: an operand's batch slice exceeds 2 GiB");
  a.a_bytes = (uint32_t)(a_ext * 4);
  a.b_bytes = (uint32_t)(b_ext * 4);
  a.M = (int)p.M;
  a.N = (int)p.N;
  a.K = (int)p.K;
  a.batch = (int)p.batch;
  a.bias_dt = p.bias_dt;
  a.epi = p.epi;

  // The form and, when K is long enough to share, the number of splits (up
  // to 8 of at least 1024, their partials at most 1 GiB) of least estimated
  // time.  A stream under capture whose workspace cannot hold the partials
  // takes one split: which calls want several is this choice's affair.
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const double out_bytes = (double)p.batch * p.M * p.N * 4.0;
  const int64_t per_split = p.batch * p.M * p.N;
  int form = 0, splits = 1;
  for (int most = 8;; most = 1) {
    float best = 0.0f;
    for (int f = 0; f < kForms; ++f)
      for (int sp = 1; sp <= most && (sp == 1 || (p.K >= 2048 && p.K / sp >= 1024 &&
                                                  sp * out_bytes <= 1073741824.0));
           ++sp) {
        const float us = estimate(a, kForm[f], sp, cus);
        if ((f == 0 && sp == 1) || us < best) {
          best = us;
          form = f;
          splits = sp;
        }
      }
    if (splits == 1 || !WorkspaceLease::refused_by_capture(s, (size_t)(splits * per_split) * 4)) break;
  }
  const Form &f = kForm[form];
  a.tiles_m = (int)((p.M + 64 * f.tm - 1) / (64 * f.tm));
  a.tiles_n = (int)((p.N + 64 * f.tn - 1) / (64 * f.tn));
  a.splits = splits;
  const int nk = (a.K + BK - 1) / BK;
  a.chunks = chunks_of(a, splits);
  const int64_t units = tiles_of(a, f) * splits;
  if (units * a.chunks > 0x7fffffff) return fail(NOVA_HIP_ERANGE, "gemm_f32_mfma: grid too large");
  a.round = cus % 8 == 0 ? cus * f.per_cu : 0;
  // One workgroup per resident slot, as long as every unit has more K steps
  // than the kernel fetches ahead; else one per tile and split (where there
  // is more than one chunk, each has at least 512 / 32 / 3 steps).
  static_assert(512 / BK / 3 > 3, "chunks longer than the ring");
  const int64_t grid =
      nk / (splits * a.chunks) > f.stages && units > cus * f.per_cu ? cus * f.per_cu : units;

  WorkspaceLease lease;  // the partials, held until their reduction is enqueued
  if (splits > 1) {
    a.part = static_cast<float *>(lease.acquire(s, (size_t)(splits * per_split) * 4));
    if (!a.part) return NOVA_HIP_ENOMEM;
  }
  const int32_t rc = p.a_kcontig ? launch_a_kcontig(form, a, p.b_kcontig, (unsigned)grid, s)
                                 : launch_a_mcontig(form, a, p.b_kcontig, (unsigned)grid, s);
  if (rc || splits == 1) return rc;
  const int gelu = (p.epi == NOVA_HIP_EPI_BIAS_GELU || p.epi == NOVA_HIP_EPI_GELU) ? 1 : 0;
  const int w = a.N % 4 == 0 ? 4 : 1;
  const dim3 rg((unsigned)((per_split / w + 255) / 256));
  if (w == 4)
    hipLaunchKernelGGL(split_reduce_kernel<4>, rg, dim3(256), 0, s, a.part, splits, per_split, a.M,
                       a.N, a.C, p.scb, p.scm, gelu);
  else
    hipLaunchKernelGGL(split_reduce_kernel<1>, rg, dim3(256), 0, s, a.part, splits, per_split, a.M,
                       a.N, a.C, p.scb, p.scm, gelu);
  return check_hip(hipGetLastError(), "gemm_f32_mfma split reduce launch");
}

}  // namespace nova_hip
