// f32 GEMM on the bf16 matrix cores: each f32 value is the exact sum of
// three bf16 values, x = h + m + l (8 + 8 + 8 significand bits; h and m are
// rounded to nearest, so each remainder is at most 2^-9 of what it is a
// remainder of), and a product a b is summed from six of the nine partial
// products, h h, h m, m h, m m, h l, l h, on v_mfma_f32_32x32x16_bf16 with
// f32 accumulation.  The three left out are below 2^-26 of the product, a
// quarter of the rounding of an f32 multiply, and sixteen terms are summed
// per accumulation instead of two, so the result is no further from the
// exact sum than the f32 MFMA's.  Six bf16 MFMAs of this shape take 2.7
// times fewer cycles than the eight v_mfma_f32_32x32x2_f32 they replace.
//
// Signs.  Where products reach below the accumulator's last bits (the small
// partial products mostly do), the bf16 MFMA drops what is under its guard
// bits towards minus infinity: a bias of one sign in every output (measured
// mean -1.1e-6 of the outputs' scale at K = 50304 where plain bf16 operands
// give -3e-9), harmless in an output but not in a sum of many outputs, such as
// a bias gradient.  So every other unit of work, tiles and K splits counted
// like the squares of a chess board, splits one operand with its sign changed,
// sums the negated result and negates that.
//
// Length of a sum.  The MFMA also drops from each product what lies 2^-27 and
// more below the accumulator, so where a few terms dwarf the others (a
// one-hot gradient), small products lose bits that the f32 MFMA's fused
// multiply-adds round in, the same way in every row.  So from K = 512 on a sum
// is taken in at least three parts, of at most 3200 k: the K splits, and
// within a split in chunks, each added in f32 to the output (or the split's
// partial sum) by the workgroup that wrote it.  A sum over the rows of a loss
// gradient times the head's weights, against 64 bits: 1.5e-6 off at 1000
// classes in one part and 5.8e-7 in three (5.4e-7 on the f32 MFMA), 3.7e-6 at
// 50304 classes in 8 parts and 1.1e-6 in 16 (1.5e-6 in 8 on the f32 MFMA).
//
// What bounds it: MFMA issue and the board's power limit.  A K step moves as
// many bytes through LDS as a bf16 GEMM's and multiplies three times as long
// on them, so two stages hide the DMA.  The splitting is VALU work (13
// operations per pair of values) beside the MFMAs of the step before: it is
// done as fragments are read, once per wave that needs one, which is why the
// wave tiles are as large as the registers allow.
//
// Stages are those of gemm_ring.h with 32 f32 in place of 64 16-bit values:
// a K-contiguous operand as [rows][8 chunks of 4 k], an M/N-contiguous one
// as [32 k][rows / 4 chunks of 4 rows].  The latter is read with 4-byte
// reads down the k-lines; its chunks are XOR-swizzled so that the two lane
// halves, eight k-lines apart, fall on different banks.  Rows need only be
// 4-byte aligned.
//
// Range.  Every value is split times 2^24, so that the lowest bit of the
// smallest f32 subnormal, 2^-149, is a normal bf16's (and nothing depends on
// how the MFMA takes subnormal inputs), and outputs are scaled back by 2^-48:
// exact but where an output is subnormal, and the same bits as without for
// ordinary operands.  What is too small for the accumulator is then under
// 2^-173 in the output, below the smallest subnormal.  What is too large, an operand
// from 2^104 on (its first piece is infinite and the next one NaN, whatever
// it multiplies; infinities and NaNs likewise) or a sum from 2^80 on, leaves
// outputs that are not finite: a wave computes such a block of its columns
// again on v_mfma_f32_32x32x2_f32 straight from memory, so that infinities,
// NaNs and overflow come out as f32 arithmetic gives them.  That costs the
// blocks it happens to more than twice their time: 8192 x 8192 x 384 takes 408
// us, 413 with a NaN in one row and 952 of nothing but NaNs.  The scaling costs
// nothing where the MFMAs are the bound, and up to 7% of the 64 x 64 form, whose
// bound is the splitting (256^3 9.4 -> 10.0 us).
#pragma once

#include "gemm_ring.h"

namespace nova_hip {
namespace split {

using namespace gemm;
using dma::lds_addr;

constexpr int BK = 32;
// Parts that a sum of K terms is taken in, at least.
inline int64_t min_parts(int64_t K) {
  const int64_t n = (K + 3199) / 3200;
  return K < 512 ? 1 : n < 3 ? 3 : n;
}

struct SplitArgs {
  const float *A;
  const float *B;
  float *C;
  const void *bias;
  float *part;  // split-K partials [splits][batch][M][N], or null
  int64_t sab, sa_outer, sbb, sb_outer, scb, scm;
  uint32_t a_bytes, b_bytes;
  int M, N, K;
  int tiles_m, tiles_n, batch;
  int splits, chunks;    // K in splits (workgroups) of chunks (units in turn)
  int round;             // workgroups resident at once
  int bias_dt, epi;
};

struct Pieces {
  u32x4 p[3];  // h, m, l: eight bf16 each
};

// The eight values of a fragment (issued, not yet landed).
struct Raw {
  f32x4 v[2];
};

__device__ __forceinline__ float flip(float x, uint32_t sign) {
  return __uint_as_float(__float_as_uint(x) ^ sign);
}

constexpr float kUp = 0x1p24f, kDown = 0x1p-48f;  // see Range, at the top

// Half of the splitting of values 2 q and 2 q + 1: h and the remainder
// (unit 0), then m and l (unit 1).  FLIP: of the values with `sign` changed.
template <bool FLIP>
__device__ __forceinline__ void split_unit(Pieces &p, Raw &r, int q, int unit, uint32_t sign) {
  float a = r.v[q >> 1][2 * (q & 1)], b = r.v[q >> 1][2 * (q & 1) + 1];
  if (unit == 0) {
    const float up = FLIP ? flip(kUp, sign) : kUp;
    a = a * up;
    b = b * up;
  }
  const uint32_t w = pack_bf16(a, b);
  a = a - __uint_as_float(w << 16);
  b = b - __uint_as_float(w & 0xffff0000u);
  p.p[unit][q] = w;
  if (unit == 0) {
    r.v[q >> 1][2 * (q & 1)] = a;
    r.v[q >> 1][2 * (q & 1) + 1] = b;
  } else {
    p.p[2][q] = pack_bf16(a, b);
  }
}
template <bool FLIP>
__device__ __forceinline__ Pieces split8(Raw r, uint32_t sign) {
  Pieces p;
#pragma unroll
  for (int u = 0; u < 8; ++u) split_unit<FLIP>(p, r, u >> 1, u & 1, sign);
  return p;
}

// XOR of a chunk index of k-line k of an M/N-contiguous stage.
__device__ __forceinline__ int line_swz(int k) { return (k & 8); }

// Fragment f of a wave (rows row_base + 32 f + lane % 32, k = 16 kk + 8
// (lane / 32) ... + 7) is read at frag_base of parity frag_parity(f, kk),
// frag_fixed bytes on: 32 rows on, a K-contiguous row's swizzle has its bit 2
// changed, as it has at the other kk, and the swizzle of an M/N-contiguous
// line turns the step of 8 chunks round in the lanes of one half.  Two
// registers per operand hold all of a wave's offsets.
template <bool KC, int R>
__device__ __forceinline__ uint32_t frag_base(int row_base, int parity, int lane) {
  const int h = lane >> 5;
  if constexpr (KC) {
    const int row = row_base + (lane & 31);
    return (uint32_t)(row * 8 + ((parity * 4 + h * 2) ^ ((row ^ (row >> 3)) & 7))) * 16u;
  } else {
    const int row = row_base + 32 * parity + (lane & 31), k = h * 8;
    return (uint32_t)(k * R + ((((row >> 2) ^ line_swz(k)) << 2) | (row & 3))) * 4u;
  }
}
template <bool KC>
constexpr int frag_parity(int f, int kk) {
  return KC ? (f ^ kk) & 1 : f & 1;
}
template <bool KC, int R>
constexpr int frag_fixed(int f, int kk) {
  return KC ? f * 32 * 128 : (f >> 1) * 64 * 4 + kk * 16 * R * 4;
}

typedef float f32x2 __attribute__((ext_vector_type(2)));
template <int O0, int O1>
__device__ __forceinline__ f32x2 lds_read2st64(uint32_t addr) {
  f32x2 v;
  asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(v) : "v"(addr), "n"(O0), "n"(O1));
  return v;
}
template <int O>
__device__ __forceinline__ f32x4 lds_read_b128_at(uint32_t addr) {
  f32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(O));
  return v;
}
// The fragment O bytes past addr.
template <bool KC, int R, int O>
__device__ __forceinline__ Raw read_raw(uint32_t addr) {
  Raw r;
  if constexpr (KC) {
    static_assert(O < 65536, "offset range");
    r.v[0] = lds_read_b128_at<O>(addr);
    r.v[1] = lds_read_b128_at<O>(addr ^ 16u);
  } else {
    constexpr int P = R / 64, Q = O / 256;  // a k-line, the offset in units of 64 dwords
    static_assert(O % 256 == 0 && Q + 7 * P < 256, "offset range");
    const f32x2 a = lds_read2st64<Q, Q + P>(addr), b = lds_read2st64<Q + 2 * P, Q + 3 * P>(addr);
    const f32x2 c = lds_read2st64<Q + 4 * P, Q + 5 * P>(addr);
    const f32x2 d = lds_read2st64<Q + 6 * P, Q + 7 * P>(addr);
    r.v[0] = f32x4{a[0], a[1], b[0], b[1]};
    r.v[1] = f32x4{c[0], c[1], d[0], d[1]};
  }
  return r;
}

// In which phase of a k16 step (one per column block) each fragment of the
// next step is read and split: about the same number in each, and B's block
// j only after phase j has used its registers (the last goes to a spare set).
template <int TM, int TN>
constexpr int phase_of(int f) {
  const int p = f >= TM ? f - TM + 1 : f < 2 ? 0 : f - 1;
  return p < TN ? p : TN - 1;
}
// How many fragments phase j has, and which is its n-th.
template <int TM, int TN>
constexpr int phase_count(int j) {
  int n = 0;
  for (int f = 0; f < TM + TN; ++f) n += phase_of<TM, TN>(f) == j;
  return n;
}
template <int TM, int TN>
constexpr int phase_frag(int j, int n) {
  for (int f = 0; f < TM + TN; ++f)
    if (phase_of<TM, TN>(f) == j && n-- == 0) return f;
  return -1;
}

// f(0), ..., f(N - 1) with constant arguments (a loop of this size is not
// unrolled before the arrays in it must be registers).
template <int N, typename Fn>
__device__ __forceinline__ void static_for(Fn &&f) {
  if constexpr (N > 0) {
    static_for<N - 1>(f);
    f(std::integral_constant<int, N - 1>{});
  }
}

__device__ __forceinline__ f32x16 mfma_bf16(u32x4 a, u32x4 b, f32x16 c) {
  return mfma_32x32x16<NOVA_HIP_DT_BF16>(a, b, c);
}
__device__ __forceinline__ void dma16(const float *p, uint32_t bytes, char *base, uint32_t off) {
  ring::dma16(reinterpret_cast<const uint16_t *>(p), bytes, base, off);
}
// Sixteen consecutive k of an operand's row straight from memory, the first
// `left` of them: zero beyond, except that a K-contiguous row's last chunk of
// four may go on into the next row.  (Offsets of what is read are below 2^31;
// a negative left - 1 - e sets the bit that takes the others out of range.)
template <bool KC>
__device__ __forceinline__ void load_row(float (&v)[16], const float *p, uint32_t bytes, int left,
                                         uint32_t row, uint32_t s_bytes, uint32_t k) {
  const __amdgpu_buffer_rsrc_t rsrc = make_rsrc(reinterpret_cast<const uint16_t *>(p), bytes);
  auto at = [&](uint32_t off, int e) __attribute__((always_inline)) {
    return off | ((uint32_t)(left - 1 - e) & kOOB);
  };
  if constexpr (KC) {
    const uint32_t off = row * s_bytes + k * 4u;
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      const f32x4 q = __builtin_bit_cast(
          f32x4, __builtin_amdgcn_raw_buffer_load_b128(rsrc, at(off + 16u * c, 4 * c), 0, 0));
#pragma unroll
      for (int e = 0; e < 4; ++e) v[4 * c + e] = q[e];
    }
  } else {
    uint32_t off = k * s_bytes + row * 4u;
#pragma unroll
    for (int e = 0; e < 16; ++e, off += s_bytes)
      v[e] = __builtin_bit_cast(float, __builtin_amdgcn_raw_buffer_load_b32(rsrc, at(off, e), 0, 0));
  }
}

// One unit of work: an output tile and the K steps [kt0, kt1) summed into it
// (wave-uniform).  A tile's chunks of a split are consecutive units of one
// workgroup.
struct Tile {
  int bidx, m0, n0, split, chunk, kt0, kt1;
  uint32_t sign;  // the sign bit where the negated sum is taken, else 0
};

template <int BM, int BN>
__device__ __forceinline__ Tile tile_at(const SplitArgs &a, int u) {
  constexpr int G = 4;  // bands of G tile rows, swept column by column
  const int tiles = a.batch * a.tiles_m * a.tiles_n;
  const int ti = u / a.chunks, chunk = u - ti * a.chunks;
  int id = blockIdx.x + ti * gridDim.x;
  if (a.round > 0) id = ring::xcd_order(id, tiles * a.splits, a.round);
  const int split = id / tiles;
  id -= split * tiles;
  const int per_batch = a.tiles_m * a.tiles_n;
  const int bidx = id / per_batch;
  const int t = id - bidx * per_batch;
  const int band = t / (G * a.tiles_n), first = band * G;
  const int gsz = min(a.tiles_m - first, G), in = t - band * G * a.tiles_n;
  Tile r;
  r.bidx = __builtin_amdgcn_readfirstlane(bidx);
  r.m0 = __builtin_amdgcn_readfirstlane((first + in % gsz) * BM);
  r.n0 = __builtin_amdgcn_readfirstlane(in / gsz * BN);
  r.split = __builtin_amdgcn_readfirstlane(split);
  r.chunk = __builtin_amdgcn_readfirstlane(chunk);
  // K steps dealt out evenly over the splits' chunks.
  const int64_t nk = (a.K + BK - 1) / BK, part = r.split * a.chunks + r.chunk;
  const int64_t parts = (int64_t)a.splits * a.chunks;
  r.kt0 = __builtin_amdgcn_readfirstlane((int)(part * nk / parts));
  r.kt1 = __builtin_amdgcn_readfirstlane((int)((part + 1) * nk / parts));
  r.sign = (uint32_t)__builtin_amdgcn_readfirstlane(
      (int)((uint32_t)(first + in % gsz + in / gsz + split + chunk) << 31));
  return r;
}

// 16 bytes to a row of any 4-byte alignment.
typedef float f32x4u __attribute__((ext_vector_type(4), aligned(4)));

// Persistent: workgroup g of G computes tiles g, g + G, ... with the K steps
// of all their units as one stream through the ring, so that the next
// unit's first S steps are on their way (and its first fragments split)
// before this one's outputs are written.  With more than one unit per
// workgroup every unit has more than S steps (the steps being fetched when a
// unit ends are then the next one's).
template <bool AKC, bool BKC, int TM, int TN, int S, int PER_CU>
__global__ __launch_bounds__(kThreads, PER_CU) void gemm_f32_split_kernel(SplitArgs a) {
  constexpr int BM = 64 * TM, BN = 64 * TN;
  constexpr int LA = 2 * TM, LB = 2 * TN, L = LA + LB;
  constexpr int kStageA = BM * BK * 4, kStage = (BM + BN) * BK * 4;
  constexpr int F = TM + TN;
  constexpr bool kFlipB = TN <= TM;  // the operand whose sign changes: the smaller
  static_assert((S - 1) * L < 64, "vmcnt range");

  __shared__ __attribute__((aligned(128))) char smem[S * kStage];
  // One 32 x 32 block per wave; the smallest tile's one block fits registers.
  constexpr bool kGeluLds = TM * TN > 1;
  __shared__ f32x4 gelu_s[kGeluLds ? 4 : 1][kGeluLds ? 256 : 1];
  static_assert(sizeof(smem) + sizeof(gelu_s) <= 160 * 1024, "LDS");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int am = (wave >> 1) * 32 * TM, bn = (wave & 1) * 32 * TN;

  const int total = a.batch * a.tiles_m * a.tiles_n * a.splits;
  const int units = (total - (int)blockIdx.x + (int)gridDim.x - 1) / (int)gridDim.x * a.chunks;

  // As in gemm_ring.h: byte offset (at k = 0, from the tile's first row) and
  // k within a K step of the chunk this lane's DMA load i fetches.  The
  // pattern repeats after 64 rows (two loads) of a K-contiguous operand and
  // after 16 k-lines (TM or TN loads) of the other: a lane keeps one period,
  // and what later loads add is the same for all lanes.
  auto setup = [&](auto kc, auto rows, int64_t s_outer, int i, uint32_t &off, int &kl)
                   __attribute__((always_inline)) {
    constexpr bool KC = decltype(kc)::value;
    constexpr int CH = decltype(rows)::value / 4;
    const int s = (i * 4 + wave) * 64 + lane;
    if constexpr (KC) {
      const int row = s >> 3, c = (s & 7) ^ ((row ^ (row >> 3)) & 7);
      kl = c * 4;
      off = (uint32_t)(((int64_t)row * s_outer + c * 4) * 4);
    } else {
      const int k = s / CH, c = (s - k * CH) ^ line_swz(k);
      kl = k;
      off = (uint32_t)(((int64_t)k * s_outer + c * 4) * 4);
    }
  };
  constexpr int PA = AKC ? 2 : TM, PB = BKC ? 2 : TN;
  uint32_t oa[PA], ob[PB];
  int ka[PA], kb[PB];
#pragma unroll
  for (int i = 0; i < PA; ++i)
    setup(std::integral_constant<bool, AKC>{}, std::integral_constant<int, BM>{}, a.sa_outer, i,
          oa[i], ka[i]);
#pragma unroll
  for (int i = 0; i < PB; ++i)
    setup(std::integral_constant<bool, BKC>{}, std::integral_constant<int, BN>{}, a.sb_outer, i,
          ob[i], kb[i]);
  // The next K step to fetch: S steps ahead of the one being multiplied.
  struct {
    const float *A, *B;   // batch slices
    uint32_t at_a, at_b;  // byte offsets of the tile's K step
    int left;             // K - k, or 0 with nothing to fetch
    int steps;            // this unit's steps yet to fetch
    int unit;
    Tile t;
  } next;
  const uint32_t row_a = (uint32_t)(a.sa_outer * 4), row_b = (uint32_t)(a.sb_outer * 4);
  const uint32_t step_a = AKC ? BK * 4u : BK * row_a;
  const uint32_t step_b = BKC ? BK * 4u : BK * row_b;
  auto next_unit = [&](int u) __attribute__((always_inline)) {
    next.unit = u;
    next.left = next.steps = 0;
    if (u >= units) return;
    const Tile t = tile_at<BM, BN>(a, u);
    next.t = t;
    next.A = a.A + (int64_t)t.bidx * a.sab;
    next.B = a.B + (int64_t)t.bidx * a.sbb;
    next.at_a = (uint32_t)((AKC ? (int64_t)t.m0 * a.sa_outer : (int64_t)t.m0) * 4) + t.kt0 * step_a;
    next.at_b = (uint32_t)((BKC ? (int64_t)t.n0 * a.sb_outer : (int64_t)t.n0) * 4) + t.kt0 * step_b;
    next.steps = t.kt1 - t.kt0;
    next.left = next.steps > 0 ? a.K - t.kt0 * BK : 0;
  };
  auto advance = [&]() __attribute__((always_inline)) {
    next.at_a += step_a;
    next.at_b += step_b;
    next.left -= BK;
    if (--next.steps <= 0) next_unit(next.unit + 1);
  };
  // DMA load q (A's first, then B's) of that step into stage st; nothing is
  // read for k >= K.
  auto dma = [&](int q, int st) __attribute__((always_inline)) {
    char *base = smem + st * kStage;
    if (q < LA) {
      const int p = q / PA;
      const uint32_t at = next.at_a + (uint32_t)(p * (AKC ? 64 : 16)) * row_a;
      dma16(next.A, a.a_bytes, base + (q * 4 + wave) * 1024,
            ka[q % PA] < next.left - (AKC ? 0 : 16 * p) ? oa[q % PA] + at : kOOB);
    } else {
      const int r = q - LA, p = r / PB;
      const uint32_t at = next.at_b + (uint32_t)(p * (BKC ? 64 : 16)) * row_b;
      dma16(next.B, a.b_bytes, base + kStageA + (r * 4 + wave) * 1024,
            kb[r % PB] < next.left - (BKC ? 0 : 16 * p) ? ob[r % PB] + at : kOOB);
    }
  };
  // With K not a multiple of 4, the last chunk of a K-contiguous row holds
  // values of the next row: zero them once the K step holding it has landed.
  const bool tail = (AKC || BKC) && (a.K & 3) != 0;
  auto zero_tail = [&](int st) __attribute__((always_inline)) {
    const int kend = a.K & (BK - 1);
    for (int r = tid; r < (AKC ? BM : 0) + (BKC ? BN : 0); r += kThreads) {
      const int row = AKC && r >= BM ? r - BM : r;
      float *base = reinterpret_cast<float *>(smem + st * kStage + ((AKC && r < BM) ? 0 : kStageA));
      for (int k = kend; k & 3; ++k)
        base[row * 32 + (((k >> 2) ^ ((row ^ (row >> 3)) & 7)) << 2) + (k & 3)] = 0.0f;
    }
    __syncthreads();
  };

  uint32_t fofs_a[2], fofs_b[2];
#pragma unroll
  for (int p = 0; p < 2; ++p) {
    fofs_a[p] = frag_base<AKC, BM>(am, p, lane);
    fofs_b[p] = kStageA + frag_base<BKC, BN>(bn, p, lane);
  }
  const uint32_t lds0 = lds_addr(smem);
  // Fragment f (A's first, then B's) of k16 step kk of the stage at `stage`.
  auto read_one = [&](auto fc, uint32_t stage, auto kkc) __attribute__((always_inline)) {
    constexpr int f = decltype(fc)::value, kk = decltype(kkc)::value;
    if constexpr (f < TM)
      return read_raw<AKC, BM, frag_fixed<AKC, BM>(f, kk)>(stage + fofs_a[frag_parity<AKC>(f, kk)]);
    else
      return read_raw<BKC, BN, frag_fixed<BKC, BN>(f - TM, kk)>(
          stage + fofs_b[frag_parity<BKC>(f - TM, kk)]);
  };

  f32x16 acc[TM][TN];
  Pieces pa[2][TM], pb[TN], spare;

  const int last_kt = (a.K + BK - 1) / BK - 1;  // the K step that may hold a tail

  // Prologue: the first S steps in flight, the first landed and split.
  next_unit(0);
  Tile tc = next.t;
#pragma unroll
  for (int st = 0; st < S; ++st) {
#pragma unroll
    for (int q = 0; q < L; ++q) dma(q, st);
    if (st < tc.kt1 - tc.kt0) advance();
  }
  NOVA_WAIT_VMCNT((S - 1) * L);
  __builtin_amdgcn_s_barrier();
  if (tail && tc.kt0 == last_kt) zero_tail(0);
  static_for<F>([&](auto f) __attribute__((always_inline)) {
    __builtin_amdgcn_sched_barrier(0);
    const Raw r = read_one(f, lds0, std::integral_constant<int, 0>{});
    NOVA_WAIT_LGKMCNT0();
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (f < TM) pa[0][f] = split8<!kFlipB>(r, tc.sign);
    else pb[f - TM] = split8<kFlipB>(r, tc.sign);
  });

  // One k16 step with A's pieces in pa[KK]: the MFMAs of column block j are
  // phase j, the six partial products of each of its TM tiles, the smallest
  // first; beside them the next step's fragments (k16 step KK ^ 1 at stage
  // `from`) are read and split, the one operand with `sign` changed.  With
  // KK = 1, the next K step is fetched into stage st meanwhile.
  constexpr int kProd[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};
  auto step = [&](auto kkc, uint32_t from, int st, uint32_t sign)
                  __attribute__((always_inline)) {
    constexpr int KK = decltype(kkc)::value;
    static_for<TN>([&](auto jc) __attribute__((always_inline)) {
      constexpr int j = decltype(jc)::value;
      constexpr int NF = phase_count<TM, TN>(j);
      __builtin_amdgcn_sched_barrier(0);
      Raw raw[NF];
      static_for<NF>([&](auto n) __attribute__((always_inline)) {
        raw[n] = read_one(std::integral_constant<int, phase_frag<TM, TN>(j, n)>{}, from,
                          std::integral_constant<int, KK ^ 1>{});
      });
      if constexpr (KK == 1) {
        constexpr int kPer = (L + TN - 1) / TN;
        static_for<kPer>([&](auto q) __attribute__((always_inline)) {
          if constexpr (j * kPer + q < L) dma(j * kPer + q, st);
        });
      }
      // MFMA m of the phase.
      auto mfma_one = [&](int m) __attribute__((always_inline)) {
        acc[m % TM][j] = mfma_bf16(pb[j].p[kProd[m / TM][1]], pa[KK][m % TM].p[kProd[m / TM][0]],
                                   acc[m % TM][j]);
      };
      static_for<2 * TM>([&](auto m) __attribute__((always_inline)) { mfma_one(m); });
      __builtin_amdgcn_sched_barrier(0);
      NOVA_WAIT_LGKMCNT0();
      __builtin_amdgcn_sched_barrier(0);
      // The splitting goes out in units of five or six operations, spread
      // evenly behind the 4 TM remaining MFMAs and fenced there.
      constexpr int kMfma = 4 * TM, kUnits = 8 * NF;
      Pieces nw[NF];
      static_for<kMfma>([&](auto m) __attribute__((always_inline)) {
        mfma_one(2 * TM + m);
        constexpr int first = (m * kUnits + kMfma - 1) / kMfma;
        constexpr int end = ((m + 1) * kUnits + kMfma - 1) / kMfma;
        static_for<end - first>([&](auto v) __attribute__((always_inline)) {
          constexpr int u = first + v;
          constexpr bool isb = phase_frag<TM, TN>(j, u / 8) >= TM;
          split_unit<isb == kFlipB>(nw[u / 8], raw[u / 8], (u % 8) >> 1, u & 1, sign);
        });
        __builtin_amdgcn_sched_barrier(0);
      });
      static_for<NF>([&](auto n) __attribute__((always_inline)) {
        constexpr int f = phase_frag<TM, TN>(j, n);
        // Opaque here: the compiler otherwise moves the whole step's
        // splitting to the top of the next step, ahead of its MFMAs.
        asm volatile("" : "+v"(nw[n].p[0]), "+v"(nw[n].p[1]), "+v"(nw[n].p[2]));
        if constexpr (f < TM) pa[KK ^ 1][f] = nw[n];
        else if constexpr (f - TM == j) spare = nw[n];
        else pb[f - TM] = nw[n];
      });
    });
    pb[TN - 1] = spare;
  };

  int cur = 0;
  for (int ti = 0; ti < units; ++ti) {
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int v = 0; v < 16; ++v) acc[i][j][v] = 0.0f;
    for (int t = tc.kt0; t < tc.kt1; ++t) {
      const int nxt = cur == S - 1 ? 0 : cur + 1;
      step(std::integral_constant<int, 0>{}, lds0 + cur * kStage, 0, tc.sign);
      // The next K step has landed for every wave, and nobody reads this
      // one's stage any more: the step S on may go there.
      __builtin_amdgcn_sched_barrier(0);
      NOVA_WAIT_VMCNT((S - 2) * L);
      __builtin_amdgcn_s_barrier();
      if (tail && t + 1 == last_kt) zero_tail(nxt);
      __builtin_amdgcn_sched_barrier(0);
      step(std::integral_constant<int, 1>{}, lds0 + nxt * kStage, cur,
           t + 1 < tc.kt1 ? tc.sign : next.t.sign);
      advance();
      cur = nxt;
    }
    __builtin_amdgcn_sched_barrier(0);

    // Outputs straight from the accumulators, one column block at a time: lane
    // l holds columns 8 g + 4 (l / 32) ... + 3 of row l % 32 of a block, 16
    // bytes.  (The lane is opaque here: what is computed from it below is not
    // kept in registers through the K loops.)
    const bool has_bias =
        (a.epi == NOVA_HIP_EPI_BIAS || a.epi == NOVA_HIP_EPI_BIAS_GELU) && tc.kt0 == 0;
    const bool has_gelu = (a.epi == NOVA_HIP_EPI_BIAS_GELU || a.epi == NOVA_HIP_EPI_GELU) &&
                          !a.part && tc.kt1 * BK >= a.K;
    float *Cb = a.part ? a.part + ((int64_t)tc.split * a.batch + tc.bidx) * a.M * a.N
                       : a.C + (int64_t)tc.bidx * a.scb;
    const int64_t ldc = a.part ? a.N : a.scm;
    int lr = lane & 31, lh = lane >> 5;
    asm volatile("" : "+v"(lr), "+v"(lh));
    auto store_column = [&](int j, f32x16 (&x)[TM]) __attribute__((always_inline)) {
      const int n = tc.n0 + bn + 32 * j + 4 * lh;
      if (has_bias) {
#pragma unroll
        for (int g = 0; g < 4; ++g)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const float b = n + 8 * g + e < a.N ? bias_at(a.bias, a.bias_dt, n + 8 * g + e) : 0.0f;
#pragma unroll
            for (int i = 0; i < TM; ++i) x[i][4 * g + e] += b;
          }
      }
#pragma unroll
      for (int i = 0; i < TM; ++i) {
        const int m = tc.m0 + am + 32 * i + lr;
        float *row = Cb + (int64_t)m * ldc;
        if (tc.chunk > 0 && m < a.M) {
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const int c = n + 8 * g;
            if (c + 4 <= a.N) {
              const f32x4 old = *reinterpret_cast<const f32x4u *>(row + c);
#pragma unroll
              for (int e = 0; e < 4; ++e) x[i][4 * g + e] += old[e];
            } else {
#pragma unroll
              for (int e = 0; e < 3; ++e)
                if (c + e < a.N) x[i][4 * g + e] += row[c + e];
            }
          }
        }
        if (has_gelu && !kGeluLds) {
#pragma unroll
          for (int v = 0; v < 16; ++v) x[i][v] = gelu_tanh(x[i][v]);
        }
        if (has_gelu && kGeluLds) {  // tanhf is large: in a rolled loop, through LDS
          f32x4 *blk = gelu_s[wave];
#pragma unroll
          for (int g = 0; g < 4; ++g)
            blk[g * 64 + lane] = f32x4{x[i][4 * g], x[i][4 * g + 1], x[i][4 * g + 2], x[i][4 * g + 3]};
#pragma unroll 1
          for (int g = 0; g < 4; ++g) {
            f32x4 y = blk[g * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = gelu_tanh(y[e]);
            blk[g * 64 + lane] = y;
          }
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const f32x4 y = blk[g * 64 + lane];
#pragma unroll
            for (int e = 0; e < 4; ++e) x[i][4 * g + e] = y[e];
          }
        }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int c = n + 8 * g;
          if (m < a.M && c + 4 <= a.N) {
            *reinterpret_cast<f32x4u *>(row + c) =
                f32x4{x[i][4 * g], x[i][4 * g + 1], x[i][4 * g + 2], x[i][4 * g + 3]};
          } else if (m < a.M) {
#pragma unroll
            for (int e = 0; e < 3; ++e)
              if (c + e < a.N) row[c + e] = x[i][4 * g + e];
          }
        }
      }
    };
    // Values that are not finite keep their column block back for the loop
    // below (see Range, at the top).  Those past the matrix's edges, where
    // whatever lies in memory was multiplied, do not count.
    const float down = flip(kDown, tc.sign);
    uint32_t again = 0;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      f32x16 x[TM];
      float fin = 0.0f;  // x * 0 is 0 or NaN
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) {
          // (+ 0: a zero sum is +0 whichever sign was summed, as in f32.)
          x[i][v] = __builtin_fmaf(acc[i][j][v], down, 0.0f);
          fin = __builtin_fmaf(x[i][v], 0.0f, fin);
        }
      bool bad = __any(!(fin == 0.0f));
      if (bad) {
        const int n = tc.n0 + bn + 32 * j + 4 * lh;
        fin = 0.0f;
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (tc.m0 + am + 32 * i + lr < a.M && n + 8 * (v >> 2) + (v & 3) < a.N)
              fin = __builtin_fmaf(x[i][v], 0.0f, fin);
        bad = __any(!(fin == 0.0f));
      }
      if (bad) again |= 1u << j;
      else store_column(j, x);
    }
    // Column blocks in f32 from memory, a whole 128-byte line of K-contiguous
    // rows per step: lane half h takes the sixteen k from 16 h on.
#pragma unroll 1
    for (; again; again &= again - 1) {
      const int j = __builtin_ctz(again);
      // (Opaque: what the loop makes of them is not worked out, and spilled,
      // ahead of all units.)
      uint32_t sa = row_a, sb = row_b;
      int ml = tc.m0 + am;
      asm volatile("" : "+s"(sa), "+s"(sb), "+s"(ml));
      const float *Ab = a.A + (int64_t)tc.bidx * a.sab, *Bb = a.B + (int64_t)tc.bidx * a.sbb;
      const int kend = min(a.K, tc.kt1 * BK), n = tc.n0 + bn + 32 * j + lr;
      f32x16 x[TM];
#pragma unroll
      for (int i = 0; i < TM; ++i)
#pragma unroll
        for (int v = 0; v < 16; ++v) x[i][v] = 0.0f;
#pragma unroll 1
      for (int k = tc.kt0 * BK + 16 * lh; k - 16 * lh < kend; k += 32) {
        float fa[TM][16], fb[16];
#pragma unroll
        for (int i = 0; i < TM; ++i) {
          const int m = ml + 32 * i + lr;
          load_row<AKC>(fa[i], Ab, a.a_bytes, m < a.M ? kend - k : 0, m, sa, k);
        }
        load_row<BKC>(fb, Bb, a.b_bytes, n < a.N ? kend - k : 0, n, sb, k);
        __builtin_amdgcn_sched_barrier(0);  // else each load sinks to its use and is waited for alone
#pragma unroll
        for (int e = 0; e < 16; ++e) {
          // In a K-contiguous row the values from kend on are the next row's.
          const uint32_t in = ~(uint32_t)((kend - k - 1 - e) >> 31);
          const float b = BKC ? __uint_as_float(__float_as_uint(fb[e]) & in) : fb[e];
#pragma unroll
          for (int i = 0; i < TM; ++i)
            x[i] = __builtin_amdgcn_mfma_f32_32x32x2f32(
                b, AKC ? __uint_as_float(__float_as_uint(fa[i][e]) & in) : fa[i][e], x[i], 0, 0, 0);
        }
      }
      store_column(j, x);
    }
    tc = next.t;
  }
  NOVA_WAIT_VMCNT(0);  // no DMA may target this workgroup's LDS when it retires
}

// The tile forms (launch_form's cases, in this order) and what the choice
// between them (gemm_f32_mfma.hip) needs to know of each.  The workgroups per
// CU are the kernel's last template argument too: its launch bound, which
// keeps the registers of two 128 x 128 tiles within a CU's (206 each; 320
// without).
struct Form {
  int tm, tn, stages, per_cu;  // tile 64 tm x 64 tn; workgroups per CU
  float step, more, fixed;     // us: see estimate()
};
constexpr int kForms = 6;

template <bool AKC, bool BKC>
int32_t launch_form(int form, const SplitArgs &r, unsigned grid, hipStream_t s) {
  const dim3 g(grid), b(kThreads);
  switch (form) {
    case 0: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 4, 3, 2, 1>), g, b, 0, s, r); break;
    case 1: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 3, 4, 2, 1>), g, b, 0, s, r); break;
    case 2: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 3, 3, 2, 1>), g, b, 0, s, r); break;
    case 3: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 4, 2, 2, 1>), g, b, 0, s, r); break;
    case 4: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 2, 2, 2, 2>), g, b, 0, s, r); break;
    default: hipLaunchKernelGGL((gemm_f32_split_kernel<AKC, BKC, 1, 1, 3, 3>), g, b, 0, s, r); break;
  }
  return check_hip(hipGetLastError(), "gemm_f32_split launch");
}

// By A's layout (gemm_f32_split_{kc,mc}.hip, compiled in parallel).
int32_t launch_a_kcontig(int form, const SplitArgs &r, bool bkc, unsigned grid, hipStream_t s);
int32_t launch_a_mcontig(int form, const SplitArgs &r, bool bkc, unsigned grid, hipStream_t s);

}  // namespace split
}  // namespace nova_hip
