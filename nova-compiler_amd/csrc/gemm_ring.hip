// Host side of the GEMMs of 16-byte aligned operands: which tile form of the
// ring kernel (gemm_ring.h) a problem runs on, or the persistent kernel, and
// the launch.
#include "gemm_ring.h"

namespace nova_hip {
namespace ring {
namespace {

// Measured on one MI355X (bf16, all layouts):
//   step   time of one K step of a workgroup alone on its CU, chip full
//   more   what each further workgroup on the CU adds to it
//   fixed  a workgroup's launch, first loads and epilogue
// The first six forms' constants are from 56 shapes, 8 x 136 x 64 to 4096^3,
// each on every form.
//
// The last two are for short sums, where outputs and the first loads are the
// time: two stages instead of three, so one less to fill and more workgroups
// per CU.  Fitted, beside the others, to 220 shapes of K up to 512.  Against
// the better of the same tiles with three stages they take 0.85 of the time at
// one K step and more than three 64 x 64 tiles per CU (96 x [200 x 64] x
// [64 x 200] 7.8 us, 9.7 with three; 2 x [1968 x 64] x [64 x 2656] 12.4 and
// 13.9) and 0.87 at two; the gain goes down to 0.95 at eight steps, and from
// 32 on they are behind (1.25 where a workgroup has its CU to itself).  With a
// CU to each they gain nothing at any length, and are not considered.
constexpr int kAny = 0x7fffffff;
constexpr Form kForm[kForms] = {
    {4, 3, 1, 1, 1.30f, 0.0f, 6.4f, kAny},   // 256 x 192: the least operand traffic
    {4, 2, 1, 1, 0.926f, 0.0f, 4.7f, kAny},  // 256 x 128, three stages
    {2, 2, 1, 2, 1.154f, 0.0f, 3.2f, kAny},  // 128 x 128, two K groups
    {1, 2, 2, 1, 0.42f, 0.25f, 2.7f, kAny},  // 64 x 128
    {1, 1, 3, 1, 0.30f, 0.12f, 2.7f, kAny},  // 64 x 64
    {1, 1, 1, 2, 0.465f, 0.0f, 2.7f, kAny},  // 64 x 64, two K groups: few tiles
    {1, 1, 4, 1, 0.44f, 0.09f, 1.8f, 2},     // 64 x 64, two stages
    {1, 2, 3, 1, 0.61f, 0.17f, 2.1f, 2},     // 64 x 128, two stages
};
// The persistent kernel's 256 x 256 tiles.  From a full round on it is the
// faster one (4096^3: 114 us a round against 129 for 256 x 128); below, where
// the ring's forms divide the chip badly (3072 x 4096 x 4096: 192 of its
// tiles 102 us, 384 of 256 x 128 112 us), but not where they fit
// (1024 x 11008 x 4096: 172 tiles 110 us, 232 of 256 x 192 88 us).
constexpr Form kPersistent = {4, 4, 1, 1, 1.62f, 0.0f, 6.0f, kAny};

int64_t tiles_of(const GemmArgs &a, const Form &f) {
  const int64_t bm = 64 * f.tm, bn = 64 * f.tn;
  return a.batch * ((a.M + bm - 1) / bm) * ((a.N + bn - 1) / bn);
}

// Estimated time: rounds of resident workgroups, each of which runs its K
// steps.  A chip that is not full runs its steps faster (up to 30%: less
// contention in L2, a higher clock), and so does the last, partial round;
// where several workgroups share a CU the next tile starts as one ends, so
// rounds need not be whole.  GELU of f32 outputs is tanhf on the ring kernel,
// kGelu us for each output of a thread (192 of them in a 256 x 192 tile): with
// it, 3434 x 1776 x 432 takes 43 us in that form and 20 in 64 x 64 tiles, which
// several workgroups per CU share in time.  (The persistent kernel's GELU is
// gelu_tanh_fast: a tenth.)
constexpr float kGelu = 0.1f;
float estimate(const GemmArgs &a, const Form &f, int cus) {
  const float q = (float)tiles_of(a, f) / cus;
  const int nk = (a.K + BK - 1) / BK, steps = (nk + f.kg - 1) / f.kg;
  const float share = q <= 1.0f ? 1.0f : q <= f.per_cu ? ceilf(q) : f.per_cu;  // of a CU
  const bool gelu = a.out_dt == NOVA_HIP_DT_F32 &&
                    (a.epi == NOVA_HIP_EPI_BIAS_GELU || a.epi == NOVA_HIP_EPI_GELU);
  const float fixed =
      f.fixed + (gelu ? (&f == &kPersistent ? 0.1f : 1.0f) * kGelu * (16 * f.tm * f.tn / f.kg) : 0.0f);
  float step, rounds = 1.0f;
  if (q <= 1.0f) {
    step = f.step * (0.7f + 0.3f * q);
  } else {
    step = f.step + f.more * (share - 1.0f);
  }
  if (q > f.per_cu) {
    const float r = q / f.per_cu, whole = floorf(r), part = r - whole;
    rounds = f.per_cu > 1 ? r + 0.25f : part > 0.0f ? whole + 0.7f + 0.3f * part : whole;
  }
  return rounds * (steps * step + fixed);
}

// The form of least estimated time; kForms: the persistent kernel.
int choose(const GemmArgs &a, int cus) {
  const bool whole = gemm_dma_applicable(a);
  int best = -1;
  float t = 0.0f;
  for (int i = 0; i < kForms + (whole ? 1 : 0); ++i) {
    const Form &f = i < kForms ? kForm[i] : kPersistent;
    const float e = estimate(a, f, cus);
    if (f.most < kAny && ((a.K + BK - 1) / BK > f.most || tiles_of(a, f) <= cus)) continue;
    if (best < 0 || e < t) {
      t = e;
      best = i;
    }
  }
  return best;
}

}  // namespace
}  // namespace ring

int32_t launch_gemm_aligned(const gemm::GemmArgs &a, int in_dt, bool akc, bool bkc, hipStream_t s) {
  const int cus = device_cu_count() > 0 ? device_cu_count() : 256;
  const int form = ring::choose(a, cus);
  if (form == ring::kForms) return launch_gemm_dma(a, in_dt, akc, bkc, s);
  const ring::Form &f = ring::kForm[form];
  ring::RingArgs r;
  r.g = a;
  if (ring::tiles_of(a, f) > 0x7fffffff) return fail(NOVA_HIP_ERANGE, "gemm: grid too large");
  r.g.tiles_m = (a.M + 64 * f.tm - 1) / (64 * f.tm);
  r.g.tiles_n = (a.N + 64 * f.tn - 1) / (64 * f.tn);
  r.g.round = cus % 8 == 0 ? cus * f.per_cu : 0;
  r.vec_out = (reinterpret_cast<uintptr_t>(a.C) & 15u) == 0 && a.N % 8 == 0 && a.scm % 8 == 0 &&
              a.scb % 8 == 0;
  return in_dt == NOVA_HIP_DT_BF16 ? ring::launch_bf16(form, r, akc, bkc, s)
                                   : ring::launch_f16(form, r, akc, bkc, s);
}

}  // namespace nova_hip
