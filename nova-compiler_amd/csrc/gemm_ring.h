// MFMA GEMM for operands with 16-byte aligned rows and any M, N, K: bf16 or
// f16 in, f32 accumulate, f32 / bf16 / f16 out.  The ring of gemm_dma.h
// (operands global -> LDS by DMA, XOR-swizzled stages, hand-ordered issue)
// with the tile and the number of stages as template parameters, edges, and
// K shared by several groups of waves where a shape has few tiles.
//
// What bounds it: large tiles by MFMA issue and the board's power limit, as
// gemm_pers.h; small ones by the latency of the DMA a stage ahead, which
// is why the small tiles have more stages and several workgroups per CU.
//
// Four wave64s in a 2 x 2 grid own (32 TM) x (32 TN) outputs each, so the
// tile is BM = 64 TM by BN = 64 TN.  K is consumed 64 at a time.  With KG
// groups of four waves, group g takes K steps g, g + KG, ... through a ring
// of its own and the groups' sums are added in group order at the end: a
// shape with fewer tiles than compute units then has KG times the loads and
// MFMAs in flight on each, without partial sums in memory.
//
// Edges.  Rows of A past M and columns of B past N feed only outputs that
// are not stored, so they need no mask: the operand's buffer range keeps
// every load inside its batch slice (or returns zero).  Only k >= K must
// read zero in both operands; each DMA load compares its lane's k with K
// (16-byte chunks never straddle K: K % 8 == 0 for a K-contiguous operand,
// and a chunk of the other layout lies on one k-line).
//
// Epilogue.  Each wave writes 32 rows of its accumulators at a time to its
// part of the (then free) ring and reads them back as row segments, so that
// global stores cover whole lines; bias, GELU and the output conversion are
// applied on the way out, edges are masked per 16-byte chunk.
#pragma once

#include "gemm_dma.h"

namespace nova_hip {
namespace ring {

using namespace gemm;
using dma::lds_addr;
using dma::lds_void;

constexpr int BK = 64;

struct RingArgs {
  GemmArgs g;
  int vec_out;  // a 16-bit output takes 16-byte stores (aligned rows of whole chunks)
};

// LDS chunk swizzles.  K-contiguous rows are those of gemm_dma.h.  A k-line
// of an M/N-contiguous operand of R rows is R / 8 chunks: the transposing
// reads of four lines at once (64 bytes each) fall on disjoint banks when
// the lines' chunks differ by 0, 4, 8 and 12 mod 16.  At a pitch of 16 or 32
// chunks all of that comes from the XOR; at 8 or 24 the pitch itself gives
// every second line 8, the XOR the rest.
template <int CH>
__device__ __forceinline__ int line_swz(int k) {
  if constexpr (CH % 16 == 0) return ((k & 3) << 1) ^ ((k & 3) << 2);
  else return ((k >> 1) & 1) << 2;
}

// Fragment byte offset from the operand's stage base of k16-step kk for the
// 32-row block at row_base.
template <bool KC, int R>
__device__ __forceinline__ uint32_t frag_offset(int row_base, int kk, int lane) {
  if constexpr (KC) {
    const int row = row_base + (lane & 31), c = kk * 2 + (lane >> 5);
    return (uint32_t)(row * 8 + (c ^ ((row ^ (row >> 3)) & 7))) * 16u;
  } else {
    constexpr int CH = R / 8;
    const int g = lane >> 4, p = lane & 15;
    const int n = row_base + 16 * (g & 1) + 4 * (p & 3);
    const int k = kk * 16 + 8 * (g >> 1) + (p >> 2);
    return (uint32_t)((k * CH + ((n >> 3) ^ line_swz<CH>(k))) * 8 + (n & 7)) * 2u;
  }
}

// The transposing read's second half, four k-lines on: line_swz(k + 4) =
// line_swz(k), so it is a fixed distance away.
template <bool KC, int R>
__device__ __forceinline__ u32x4 read_fragment(uint32_t addr) {
  if constexpr (KC) {
    return dma::lds_read_b128(addr);
  } else {
    static_assert(R == 64 || R == 128 || R == 192 || R == 256, "4 lines of R elements");
    const dma::u32x2v lo = dma::lds_read_tr(addr);
    dma::u32x2v hi;
    if constexpr (R == 64) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:512" : "=v"(hi) : "v"(addr));
    if constexpr (R == 128) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:1024" : "=v"(hi) : "v"(addr));
    if constexpr (R == 192) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:1536" : "=v"(hi) : "v"(addr));
    if constexpr (R == 256) hi = dma::lds_read_tr_hi(addr);
    return u32x4{lo[0], lo[1], hi[0], hi[1]};
  }
}

// 16 bytes per lane from byte offset `off` of the operand slice to LDS at
// base (wave-uniform) + 16 * lane.
__device__ __forceinline__ void dma16(const uint16_t *p, uint32_t bytes, char *base, uint32_t off) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(make_rsrc(p, bytes), (lds_void *)base, 16, off, 0, 0, 0);
}

// Workgroup id -> tile: the hardware deals ids to the 8 XCDs in turn, so in
// each round of `round` resident workgroups XCD x takes one contiguous run of
// the round's tiles (see round_tile_of), here for any number of tiles.
__device__ __forceinline__ int xcd_order(int id, int total, int round) {
  const int r = id / round, q = id - r * round;
  const int n = min(round, total - r * round);
  const int per = n >> 3, rem = n & 7, x = q & 7;
  return r * round + x * per + min(x, rem) + (q >> 3);
}

// Staging of rows of COLS f32: 16-byte chunk c of row R sits at c ^ (R & 7),
// conflict-free for the column-wise writes and the row-wise reads.
template <int COLS>
__device__ __forceinline__ f32x4 *stage_chunk(char *stg, int R, int c) {
  return reinterpret_cast<f32x4 *>(stg + R * (COLS * 4) + ((c ^ (R & 7)) << 4));
}

// Chunk c of staged row R, summed over KG staged copies `dist` bytes apart.
template <int COLS, int KG>
__device__ __forceinline__ f32x4 staged_sum(char *stg, int dist, int R, int c) {
  f32x4 x = *stage_chunk<COLS>(stg, R, c);
#pragma unroll
  for (int g = 1; g < KG; ++g) x = x + *stage_chunk<COLS>(stg + g * dist, R, c);
  return x;
}

// The bf16 / f16 bits of a value.
__device__ __forceinline__ uint16_t narrow(float x, bool bf16) {
  return bf16 ? to_bf16(x) : to_f16(x);
}

// 16 bytes at any 4-byte alignment.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// A staged ROWS x COLS block to C (its element (0, 0); `rows`, `cols` left
// in the matrix) by NT threads, this one number tid.  All of a thread's
// chunks are read before the first is used.  f32 rows need no alignment
// beyond their own 4 bytes: 16-byte stores take any (element-by-element
// stores of odd rows took 93.3 us where this takes 58.6 at 48x[997x64]x[64x997],
// 59.5 against 50.6 at 4000x3002x1024; aligned rows the same either way).
// f32 with GELU (tanhf is large) goes two chunks at a time in a rolled loop.
template <int ROWS, int COLS, int NT, int KG>
__device__ __forceinline__ void store_f32(char *stg, int dist, int tid, float *C, int64_t ld,
                                          int rows, int cols, const float *bias, bool gelu) {
  constexpr int CR = COLS / 4, kIt = ROWS * CR / NT;  // 4-column chunks per row, per thread
  static_assert(ROWS * CR % NT == 0, "whole rounds");
  // 16 bytes at once where the chunk is whole.
  auto put = [&](int it, f32x4 x) __attribute__((always_inline)) {
    const int q = it * NT + tid, R = q / CR, n = 4 * (q - R * CR);
    if (R < rows && n + 4 <= cols) {
      *reinterpret_cast<f32x4u *>(C + R * ld + n) = x;
    } else if (R < rows) {
#pragma unroll
      for (int e = 0; e < 3; ++e)
        if (n + e < cols) C[R * ld + n + e] = x[e];
    }
  };
  if (gelu) {
    constexpr int kU = kIt % 2 == 0 ? 2 : 1;
#pragma unroll 1
    for (int it = 0; it < kIt; it += kU) {
      f32x4 x[kU];
#pragma unroll
      for (int u = 0; u < kU; ++u) {
        const int q = (it + u) * NT + tid, R = q / CR, c = q - R * CR;
        x[u] = staged_sum<COLS, KG>(stg, dist, R, c);
        if (bias) x[u] = x[u] + *reinterpret_cast<const f32x4 *>(bias + 4 * c);
      }
#pragma unroll
      for (int u = 0; u < kU; ++u)
#pragma unroll
        for (int e = 0; e < 4; ++e) x[u][e] = gelu_tanh(x[u][e]);
#pragma unroll
      for (int u = 0; u < kU; ++u) put(it + u, x[u]);
    }
    return;
  }
  f32x4 x[kIt];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int q = it * NT + tid, R = q / CR;
    x[it] = staged_sum<COLS, KG>(stg, dist, R, q - R * CR);
  }
  if (bias) {
#pragma unroll
    for (int it = 0; it < kIt; ++it)
      x[it] = x[it] + *reinterpret_cast<const f32x4 *>(bias + 4 * ((it * NT + tid) % CR));
  }
#pragma unroll
  for (int it = 0; it < kIt; ++it) put(it, x[it]);
}

template <int ROWS, int COLS, int NT, int KG>
__device__ __forceinline__ void store_16(char *stg, int dist, int tid, uint16_t *C, int64_t ld,
                                         int rows, int cols, bool vec, const float *bias, bool gelu,
                                         bool bf16) {
  if (!vec) {
    constexpr int CR = COLS / 4;
#pragma unroll 1
    for (int it = 0; it < ROWS * CR / NT; ++it) {
      const int q = it * NT + tid, R = q / CR, c = q - R * CR;
      f32x4 x = staged_sum<COLS, KG>(stg, dist, R, c);
      if (bias) x = x + *reinterpret_cast<const f32x4 *>(bias + 4 * c);
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (R < rows && 4 * c + e < cols)
          C[R * ld + 4 * c + e] = narrow(gelu ? gelu_tanh_fast(x[e]) : x[e], bf16);
    }
    return;
  }
  constexpr int CR = COLS / 8, kAll = ROWS * CR;  // 8-column chunks per row
  constexpr int kIt = kAll >= NT ? kAll / NT : 1;
  static_assert(kAll % NT == 0 || kAll < NT, "whole rounds");
  if (kAll < NT && tid >= kAll) return;
  f32x4 x[kIt][2];
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int q = it * NT + tid, R = q / CR, c = q - R * CR;
#pragma unroll
    for (int h = 0; h < 2; ++h) x[it][h] = staged_sum<COLS, KG>(stg, dist, R, 2 * c + h);
  }
  if (bias) {
#pragma unroll
    for (int it = 0; it < kIt; ++it)
#pragma unroll
      for (int h = 0; h < 2; ++h)
        x[it][h] = x[it][h] +
                   *reinterpret_cast<const f32x4 *>(bias + 8 * ((it * NT + tid) % CR) + 4 * h);
  }
  if (gelu) {
#pragma unroll
    for (int it = 0; it < kIt; ++it)
#pragma unroll
      for (int e = 0; e < 8; ++e) x[it][e >> 2][e & 3] = gelu_tanh_fast(x[it][e >> 2][e & 3]);
  }
#pragma unroll
  for (int it = 0; it < kIt; ++it) {
    const int q = it * NT + tid, R = q / CR, n = 8 * (q - R * CR);
    const f32x4 lo = x[it][0], hi = x[it][1];
    const u32x4 w = bf16 ? u32x4{pack_bf16(lo[0], lo[1]), pack_bf16(lo[2], lo[3]),
                                 pack_bf16(hi[0], hi[1]), pack_bf16(hi[2], hi[3])}
                         : u32x4{pack_f16(lo[0], lo[1]), pack_f16(lo[2], lo[3]),
                                 pack_f16(hi[0], hi[1]), pack_f16(hi[2], hi[3])};
    if (R < rows && n < cols) *reinterpret_cast<u32x4 *>(C + R * ld + n) = w;
  }
}

template <int DT, bool AKC, bool BKC, int TM, int TN, int S, int KG>
__global__ __launch_bounds__(kThreads * KG) void gemm_ring_kernel(RingArgs ra) {
  const GemmArgs &a = ra.g;
  constexpr int BM = 64 * TM, BN = 64 * TN;
  constexpr int LA = 2 * TM, LB = 2 * TN;  // DMA loads per thread and stage
  constexpr int kStageA = BM * BK * 2, kStage = (BM + BN) * BK * 2;
  constexpr int kSteps = BK / 16;
  constexpr int kM = TM * TN, kF = TM + TN;
  constexpr int kReads = (kF + kM - 1) / kM;  // fragment reads per MFMA
  constexpr int kDmaA = (LA + kM - 1) / kM, kDmaB = (LB + kM - 1) / kM;
  static_assert((S - 2) * (LA + LB) + LA < 64, "vmcnt range");
  static_assert((KG > 1 ? BM : 128) * BN * 4 / (KG > 1 ? 1 : 2) <= S * kStage,
                "a group's part of the epilogue fits its ring");

  __shared__ __attribute__((aligned(16))) char smem[KG * S * kStage];
  __shared__ __attribute__((aligned(16))) float bias_s[BN];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane((tid >> 6) & 3);
  const int grp = KG > 1 ? __builtin_amdgcn_readfirstlane(tid >> 8) : 0;
  char *const ring = smem + grp * (S * kStage);
  const int am = (wave >> 1) * 32 * TM, bn = (wave & 1) * 32 * TN;

  const int tiles = a.batch * a.tiles_m * a.tiles_n;
  const int id = a.round > 0 ? xcd_order(blockIdx.x, tiles, a.round) : blockIdx.x;
  int bidx, tm, tn;
  {
    // Bands of G tile rows swept column by column (near-square blocks of
    // the tiles an XCD runs at once share their panels in its L2).
    constexpr int G = TM == 4 ? 4 : 8;
    const int per_batch = a.tiles_m * a.tiles_n;
    bidx = id / per_batch;
    const int t = id - bidx * per_batch;
    const int band = t / (G * a.tiles_n), first = band * G;
    const int gsz = min(a.tiles_m - first, G), in = t - band * G * a.tiles_n;
    tm = __builtin_amdgcn_readfirstlane(first + in % gsz);
    tn = __builtin_amdgcn_readfirstlane(in / gsz);
    bidx = __builtin_amdgcn_readfirstlane(bidx);
  }
  const int m0 = tm * BM, n0 = tn * BN;
  const int nk = (a.K + BK - 1) / BK, nt = (nk + KG - 1) / KG;

  const bool has_bias = (a.epi == NOVA_HIP_EPI_BIAS || a.epi == NOVA_HIP_EPI_BIAS_GELU);
  if (has_bias && tid < BN) bias_s[tid] = n0 + tid < a.N ? bias_at(a.bias, a.bias_dt, n0 + tid) : 0.f;

  const uint16_t *Ab = a.A + (int64_t)bidx * a.sab, *Bb = a.B + (int64_t)bidx * a.sbb;
  // DMA load i of wave w fills slots [(i*4 + w) * 64, +64) of its operand's
  // stage; the lane fetches the chunk the swizzle puts into its slot.
  // off: byte offset at k = 0; kl: the chunk's k within a K step.
  auto setup = [&](auto kc, auto rows, int row0, int64_t s_outer, int i, uint32_t &off, int &kl)
                   __attribute__((always_inline)) {
    constexpr bool KC = decltype(kc)::value;
    constexpr int CH = decltype(rows)::value / 8;
    const int s = (i * 4 + wave) * 64 + lane;
    if constexpr (KC) {
      const int row = s >> 3, c = (s & 7) ^ ((row ^ (row >> 3)) & 7);
      kl = c * 8;
      off = (uint32_t)(((int64_t)(row0 + row) * s_outer + c * 8) * 2);
    } else {
      const int k = s / CH, c = (s - k * CH) ^ line_swz<CH>(k);
      kl = k;
      off = (uint32_t)(((int64_t)k * s_outer + row0 + c * 8) * 2);
    }
  };
  uint32_t oa[LA], ob[LB];
  int ka[LA], kb[LB];
#pragma unroll
  for (int i = 0; i < LA; ++i)
    setup(std::integral_constant<bool, AKC>{}, std::integral_constant<int, BM>{}, m0, a.sa_outer, i,
          oa[i], ka[i]);
#pragma unroll
  for (int i = 0; i < LB; ++i)
    setup(std::integral_constant<bool, BKC>{}, std::integral_constant<int, BN>{}, n0, a.sb_outer, i,
          ob[i], kb[i]);
  const uint32_t step_a = AKC ? BK * 2u : (uint32_t)(BK * a.sa_outer * 2);
  const uint32_t step_b = BKC ? BK * 2u : (uint32_t)(BK * a.sb_outer * 2);

  // DMA load q (A's first, then B's) of this group's K step t into stage st;
  // nothing is read past the last step or for k >= K.
  auto dma = [&](int q, int st, int t) __attribute__((always_inline)) {
    const int kt = t * KG + grp;
    const int left = kt < nk ? a.K - kt * BK : 0;
    char *base = ring + st * kStage;
    if (q < LA)
      dma16(Ab, a.a_bytes, base + (q * 4 + wave) * 1024,
            ka[q] < left ? oa[q] + (uint32_t)kt * step_a : kOOB);
    else
      dma16(Bb, a.b_bytes, base + kStageA + ((q - LA) * 4 + wave) * 1024,
            kb[q - LA] < left ? ob[q - LA] + (uint32_t)kt * step_b : kOOB);
  };

  uint32_t fofs[kSteps][kF];
#pragma unroll
  for (int kk = 0; kk < kSteps; ++kk)
#pragma unroll
    for (int f = 0; f < kF; ++f)
      fofs[kk][f] = f < TM ? frag_offset<AKC, BM>(am + f * 32, kk, lane)
                           : kStageA + frag_offset<BKC, BN>(bn + (f - TM) * 32, kk, lane);
  const uint32_t lds0 = lds_addr(ring);

  f32x16 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
  u32x4 fa[2][TM], fb[2][TN];

  auto read_one = [&](int f, int buf, uint32_t stage, int kk) __attribute__((always_inline)) {
    if (f < TM) fa[buf][f] = read_fragment<AKC, BM>(stage + fofs[kk][f]);
    else fb[buf][f - TM] = read_fragment<BKC, BN>(stage + fofs[kk][f]);
  };
  // MFMA m of a k16 step (B first, so a lane holds four consecutive columns
  // of a row) and the reads that go out behind it.
  auto mfma_read = [&](int m, int buf, bool read, uint32_t stage, int kk)
                       __attribute__((always_inline)) {
    const int i = m / TN, j = m % TN;
    acc[i][j] = mfma_32x32x16<DT>(fb[buf][j], fa[buf][i], acc[i][j]);
    if (read) {
#pragma unroll
      for (int f = m * kReads; f < (m + 1) * kReads && f < kF; ++f) read_one(f, buf ^ 1, stage, kk);
    }
  };

  // Prologue: steps 0 .. S - 2 and A of the next one in flight, the first
  // landed and its first fragments read.
#pragma unroll
  for (int st = 0; st < S - 1; ++st)
#pragma unroll
    for (int q = 0; q < LA + LB; ++q) dma(q, st, st);
#pragma unroll
  for (int q = 0; q < LA; ++q) dma(q, S - 1, S - 1);
  NOVA_WAIT_VMCNT((S - 2) * (LA + LB) + LA);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int f = 0; f < kF; ++f) read_one(f, 0, lds0, 0);
  __builtin_amdgcn_sched_barrier(0);

  // K step t: the fragments of k16 step s + 1 are read under the MFMAs of
  // step s.  B of step t + S - 1 goes out in k16 step 0 and, once the
  // barrier has freed stage t, A of step t + S in the last one.  The wait
  // ahead of the barrier leaves the S - 2 newest steps' loads in flight.
  int cur = 0;
  for (int t = 0; t < nt; ++t) {
    const int prv = cur == 0 ? S - 1 : cur - 1, nxt = cur == S - 1 ? 0 : cur + 1;
    const uint32_t stage = lds0 + cur * kStage, next = lds0 + nxt * kStage;
#pragma unroll
    for (int s = 0; s < kSteps - 1; ++s) {
      NOVA_WAIT_LGKMCNT0();
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int m = 0; m < kM; ++m) {
        mfma_read(m, s & 1, true, stage, s + 1);
        if (s == 0) {
#pragma unroll
          for (int q = m * kDmaB; q < (m + 1) * kDmaB && q < LB; ++q) dma(LA + q, prv, t + S - 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    NOVA_WAIT_LGKMCNT0();
    NOVA_WAIT_VMCNT((S - 2) * (LA + LB));
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int m = 0; m < kM; ++m) {
      mfma_read(m, (kSteps - 1) & 1, true, next, 0);
#pragma unroll
      for (int q = m * kDmaA; q < (m + 1) * kDmaA && q < LA; ++q) dma(q, cur, t + S);
      __builtin_amdgcn_sched_barrier(0);
    }
    cur = nxt;
  }
  // No DMA may still target the ring, and the reads past the last step must
  // have landed, before the epilogue reuses it.  Those reads' registers are
  // named after the wait: dead, they could be given to the epilogue's
  // address arithmetic while the reads are still on their way into them.
  __builtin_amdgcn_sched_barrier(0);
  NOVA_WAIT_VMCNT(0);
  NOVA_WAIT_LGKMCNT0();
  __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int i = 0; i < TM; ++i) asm volatile("" : : "v"(fa[0][i]));
#pragma unroll
  for (int j = 0; j < TN; ++j) asm volatile("" : : "v"(fb[0][j]));
  __syncthreads();

  const bool has_gelu = (a.epi == NOVA_HIP_EPI_BIAS_GELU || a.epi == NOVA_HIP_EPI_GELU);
  const int lr = lane & 31, lh = lane >> 5;
  if constexpr (KG == 1) {
    char *stg = smem + wave * (32 * 32 * TN * 4);
    const float *bias_w = has_bias ? bias_s + bn : nullptr;
#pragma unroll
    for (int i = 0; i < TM; ++i) {
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *stage_chunk<32 * TN>(stg, lr, 8 * j + 2 * g + lh) = f32x4{
              acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
      const int mb = m0 + am + 32 * i, nw = n0 + bn;
      const int64_t at = (int64_t)bidx * a.scb + (int64_t)mb * a.scm + nw;
      if (a.out_dt == NOVA_HIP_DT_F32)
        store_f32<32, 32 * TN, 64, 1>(stg, 0, lane, static_cast<float *>(a.C) + at, a.scm, a.M - mb,
                                      a.N - nw, bias_w, has_gelu);
      else
        store_16<32, 32 * TN, 64, 1>(stg, 0, lane, static_cast<uint16_t *>(a.C) + at, a.scm,
                                     a.M - mb, a.N - nw, ra.vec_out, bias_w, has_gelu,
                                     a.out_dt == NOVA_HIP_DT_BF16);
    }
  } else {
    // Every group stages its whole tile in its ring; all waves then share
    // the outputs, adding the groups' values in group order.
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *stage_chunk<BN>(ring, am + 32 * i + lr, bn / 4 + 8 * j + 2 * g + lh) = f32x4{
              acc[i][j][4 * g], acc[i][j][4 * g + 1], acc[i][j][4 * g + 2], acc[i][j][4 * g + 3]};
    __syncthreads();
    const int64_t at = (int64_t)bidx * a.scb + (int64_t)m0 * a.scm + n0;
    const float *bias_w = has_bias ? bias_s : nullptr;
    if (a.out_dt == NOVA_HIP_DT_F32)
      store_f32<BM, BN, kThreads * KG, KG>(smem, S * kStage, tid, static_cast<float *>(a.C) + at,
                                           a.scm, a.M - m0, a.N - n0, bias_w, has_gelu);
    else
      store_16<BM, BN, kThreads * KG, KG>(smem, S * kStage, tid, static_cast<uint16_t *>(a.C) + at,
                                          a.scm, a.M - m0, a.N - n0, ra.vec_out, bias_w, has_gelu,
                                          a.out_dt == NOVA_HIP_DT_BF16);
  }
}

// One launch of a tile config; g.tiles_m, g.tiles_n and g.round set by the
// caller.
template <int DT, int TM, int TN, int S, int KG>
int32_t launch_tile(const RingArgs &r, bool akc, bool bkc, hipStream_t s) {
  const dim3 grid((unsigned)(r.g.batch * r.g.tiles_m * r.g.tiles_n)), block(kThreads * KG);
  if (akc && bkc)
    hipLaunchKernelGGL((gemm_ring_kernel<DT, true, true, TM, TN, S, KG>), grid, block, 0, s, r);
  else if (akc)
    hipLaunchKernelGGL((gemm_ring_kernel<DT, true, false, TM, TN, S, KG>), grid, block, 0, s, r);
  else if (bkc)
    hipLaunchKernelGGL((gemm_ring_kernel<DT, false, true, TM, TN, S, KG>), grid, block, 0, s, r);
  else
    hipLaunchKernelGGL((gemm_ring_kernel<DT, false, false, TM, TN, S, KG>), grid, block, 0, s, r);
  return check_hip(hipGetLastError(), "gemm_ring launch");
}

// The tile forms, and what choose() (gemm_ring.hip) needs to know of each.
struct Form {
  int tm, tn, per_cu;  // tile 64 tm x 64 tn; workgroups that fit one CU's LDS
  int kg;
  float step, more, fixed;  // us: see choose()
  int most;                 // K steps up to which it is considered
};
constexpr int kForms = 8;

template <int DT>
int32_t launch_form(int form, const RingArgs &r, bool akc, bool bkc, hipStream_t s) {
  switch (form) {
    case 0: return launch_tile<DT, 4, 3, 2, 1>(r, akc, bkc, s);
    case 1: return launch_tile<DT, 4, 2, 3, 1>(r, akc, bkc, s);
    case 2: return launch_tile<DT, 2, 2, 2, 2>(r, akc, bkc, s);
    case 3: return launch_tile<DT, 1, 2, 3, 1>(r, akc, bkc, s);
    case 4: return launch_tile<DT, 1, 1, 3, 1>(r, akc, bkc, s);
    case 5: return launch_tile<DT, 1, 1, 4, 2>(r, akc, bkc, s);
    case 6: return launch_tile<DT, 1, 1, 2, 1>(r, akc, bkc, s);
    default: return launch_tile<DT, 1, 2, 2, 1>(r, akc, bkc, s);
  }
}

int32_t launch_bf16(int form, const RingArgs &r, bool akc, bool bkc, hipStream_t s);
int32_t launch_f16(int form, const RingArgs &r, bool akc, bool bkc, hipStream_t s);

}  // namespace ring
}  // namespace nova_hip
