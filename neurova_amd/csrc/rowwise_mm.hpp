// Rowwise 2..8-bit product over a batch of activation rows on the matrix
// cores (gfx950): Y[M, N] = X[M, K] @ dequant(W)^T, replacing the reference's
// csrc/lowbit_gemv.cu:145-224 for batches (and its one-row kernels for rows
// the LDS-staged one-row kernel does not take).
//
// Arithmetic.  The code minus the zero point is exact in fp16, so v_mfma_f32_
// 16x16x32_f16 sums exact products of codes and activations in fp32; one fp32
// FMA per accumulator and scale group applies the group's scale.  No weight is
// rounded (fp16 scaled weights would be), so the result is at least as close to
// the exact sum as a scalar fp32 loop.
//
// Fragments.  The activations are the A operand (16 rows of the batch), the
// weights B (16 output rows): lane l = 16 g + nl holds 8 k values of batch row
// / output row nl.  Eight codes of BITS bits are BITS whole bytes, so a lane's
// share of a row always starts at a byte, whatever the row stride.  The loop
// runs in stages of 128 k (4 MFMA steps).  The k values a lane takes depend on
// how many scale spans a stage has (SPS), because the four lane groups of one
// MFMA are summed and must share a scale:
//   SPS = 1 (groups of a multiple of 128): lane group g takes k = 32 g .. 32 g
//            + 31 of the stage, one piece of 4 BITS bytes;
//   SPS = 2 (64):  k = 64 h + 16 g .. + 15, two pieces of 2 BITS bytes;
//   SPS = 4 (32):  k = 32 d + 8 g .. + 7, four pieces of BITS bytes.
// Decode of 8 codes: the stream is arranged in words whose 16-bit halves hold
// codes i and i + 4 at the same offset (2 to 5 VALU, none at 4 bits), one
// v_and_or_b32 puts a pair under the exponent of 1024 and one packed add or
// fma (by 2^-offset) leaves code - z: 9 to 15 VALU per 8 codes.  The
// activations are put in the same pair order (four v_perm_b32 per fragment).
//
// Measured (4 bits, g128, against the scalar-dot kernel that read and decoded
// the weights again for every four batch rows): M = 16, K = 5120, N = 17408
// 196 -> 21 us, K = 17408, N = 5120 186 -> 24 us; M = 384 at 2 bits, g64 4260 ->
// 113 us and 3960 -> 125 us (604 TFLOP/s).  Up to 32 rows the few stages a wave
// runs, their loads and the LDS traffic bound it (floor: 9.6 us of weight
// bytes), above that the VALU work of the decode and the scales beside the MFMAs.
#pragma once

#include "lb_common.hpp"
#include "rowwise_mm_run.hpp"

namespace lb {
namespace rwmm {


constexpr int kStageK = 128;

// The group of scale span t (wave-uniform).
__device__ __forceinline__ int span_group(const Params& p, int t) {
  return p.span_mul == 0 ? t : (int)__umulhi((uint32_t)t, p.span_mul);
}

struct DecodeConsts {
  uint32_t magic;  // VGPR: fp16 exponent of 1024 in both halves
};
__device__ __forceinline__ DecodeConsts decode_consts() {
  DecodeConsts c;
  asm("v_mov_b32 %0, 0x64006400" : "=v"(c.magic));
  return c;
}

// The pair at bit offset OFF of the halves of v, as fp16 (code - z).
template <int BITS, int OFF>
__device__ __forceinline__ uint32_t pair_at(uint32_t v, const DecodeConsts& c) {
  static_assert(OFF + BITS <= 10, "inside the fp16 mantissa");
  constexpr uint32_t m = ((1u << BITS) - 1u) << OFF;
  constexpr float z = (float)(1 << (BITS - 1));
  const f16x2 b = as_h2(and_or(v, m | (m << 16), c.magic));
  if constexpr (OFF == 0) {
    return as_u32(b - (f16x2){(f16)(1024.f + z), (f16)(1024.f + z)});
  } else {
    constexpr float r = 1.f / (float)(1 << OFF);
    constexpr float o = -(1024.f * r + z);  // (1024 + code * 2^OFF) * 2^-OFF + o: exact
    return as_u32(b * (f16x2){(f16)r, (f16)r} + (f16x2){(f16)o, (f16)o});
  }
}

// low half of a, high half of b
__device__ __forceinline__ uint32_t halves(uint32_t a, uint32_t b) { return (a & 0xffffu) | (b & 0xffff0000u); }

// Eight codes of a stream (w0: bits 0..31, w1: bits 32..63 of it) as a B
// fragment, in the pair order (0,4) (1,5) (2,6) (3,7); 8 bits: natural order.
template <int BITS>
__device__ __forceinline__ f16x8 decode8(uint32_t w0, uint32_t w1, const DecodeConsts& c) {
  uint32_t p0, p1, p2, p3;
  if constexpr (BITS == 8) {
    const f16x2 zb = {(f16)1152.0f, (f16)1152.0f};
    p0 = as_u32(as_h2(__builtin_amdgcn_perm(c.magic, w0, 0x05010500u)) - zb);
    p1 = as_u32(as_h2(__builtin_amdgcn_perm(c.magic, w0, 0x05030502u)) - zb);
    p2 = as_u32(as_h2(__builtin_amdgcn_perm(c.magic, w1, 0x05010500u)) - zb);
    p3 = as_u32(as_h2(__builtin_amdgcn_perm(c.magic, w1, 0x05030502u)) - zb);
  } else if constexpr (BITS <= 4) {
    uint32_t v;
    if constexpr (BITS == 2) v = __builtin_amdgcn_perm(0u, w0, 0x0c010c00u);  // bytes 0 and 1
    else if constexpr (BITS == 3) v = halves(w0, w0 << 4);                    // bits 0..11 and 12..23
    else v = w0;
    p0 = pair_at<BITS, 0>(v, c);
    p1 = pair_at<BITS, BITS>(v, c);
    if constexpr (BITS == 4) {
      p2 = pair_at<4, 0>(v >> 8, c);
      p3 = pair_at<4, 4>(v >> 8, c);
    } else {
      p2 = pair_at<BITS, 2 * BITS>(v, c);
      if constexpr (BITS == 2) p3 = pair_at<2, 6>(v, c);
      else p3 = pair_at<3, 0>(v >> 9, c);
    }
  } else {
    // codes 0, 1 | 4, 5 and codes 2, 3 | 6, 7: 2 BITS bits per half
    const uint32_t v01 = halves(w0, __builtin_amdgcn_alignbit(w1, w0, 4 * BITS - 16));
    const uint32_t v23 = halves(w0 >> (2 * BITS), __builtin_amdgcn_alignbit(w1, w0, 6 * BITS - 16));
    p0 = pair_at<BITS, 0>(v01, c);
    p2 = pair_at<BITS, 0>(v23, c);
    if constexpr (2 * BITS <= 10) {
      p1 = pair_at<BITS, BITS>(v01, c);
      p3 = pair_at<BITS, BITS>(v23, c);
    } else {
      p1 = pair_at<BITS, 0>(v01 >> BITS, c);
      p3 = pair_at<BITS, 0>(v23 >> BITS, c);
    }
  }
  return __builtin_bit_cast(f16x8, (u32x4){p0, p1, p2, p3});
}

// Eight activations in the pair order of decode8.
template <int BITS>
__device__ __forceinline__ u32x4 pair_order(u32x4 v) {
  if constexpr (BITS == 8) return v;
  return (u32x4){__builtin_amdgcn_perm(v[2], v[0], 0x05040100u), __builtin_amdgcn_perm(v[2], v[0], 0x07060302u),
                 __builtin_amdgcn_perm(v[3], v[1], 0x05040100u), __builtin_amdgcn_perm(v[3], v[1], 0x07060302u)};
}

// k (of a stage) of the eight values lane group g holds in step d.
template <int SPS>
__device__ __forceinline__ int frag_k(int g, int d) {
  constexpr int per = 4 / SPS;  // steps per span
  return (d / per) * (kStageK / SPS) + g * (8 * per) + (d % per) * 8;
}

typedef u32x4 u32x4_any __attribute__((aligned(1)));

__device__ __forceinline__ u32x4 load16(const void* base, uint32_t byte_off) {
  return *reinterpret_cast<const u32x4_any*>(reinterpret_cast<const char*>(base) + byte_off);
}
// Bytes [from, from + 16) of a row of `end` bytes, zeros past its end; nothing
// outside the row is read.  One 16-byte load that ends inside the row, shifted
// into place: the stage that ends a ragged row is a serial tail of one wave,
// and sixteen byte loads a chunk there took half of a short launch (4 bits, one
// row: K = 1144, N = 1024 9.8 -> 4.7 us, K = 2168, N = 4096 12.1 -> 5.5, K = 5240, N =
// 17408 32.6 -> 17.8).
__device__ __forceinline__ u32x4 load16_tail(const uint8_t* row, int from, int end) {
  if (end < 16) {  // (uniform) the whole row is shorter than a load
    uint32_t v[4] = {0, 0, 0, 0};
#pragma unroll
    for (int b = 0; b < 16; ++b)
      if (from + b < end) v[b >> 2] |= (uint32_t)row[from + b] << (8 * (b & 3));
    return (u32x4){v[0], v[1], v[2], v[3]};
  }
  const int at = min(from, end - 16);
  const u32x4 v = load16(row + at, 0);
  const int bits = 8 * (from - at);
  uint64_t lo = v[0] | ((uint64_t)v[1] << 32), hi = v[2] | ((uint64_t)v[3] << 32);
  if (bits >= 64) {
    lo = bits >= 128 ? 0 : hi >> (bits - 64);
    hi = 0;
  } else if (bits > 0) {
    lo = (lo >> bits) | (hi << (64 - bits));
    hi >>= bits;
  }
  return (u32x4){(uint32_t)lo, (uint32_t)(lo >> 32), (uint32_t)hi, (uint32_t)(hi >> 32)};
}

// The weight bytes of 16 NB rows of one stage, through LDS.  A load
// instruction's neighbouring lanes take neighbouring 16-byte chunks of a row
// (a row's stage is BITS chunks): with each lane loading its own fragment,
// neighbouring lanes read different rows and every lane is a cache-line access
// of its own (about 60 cycles an instruction: M = 2, K = 5120, N = 17408 at 4
// bits took 20.9 us, 50.8 us with four pieces a lane).  The LDS rows are an odd
// number of 16-byte chunks long, so that the 16 rows of a fragment read fall in
// different banks.  One wave stores and reads its own rows: no barrier.
template <int BITS, int SPS, int NB>
struct Weights {
  static constexpr int kRows = 16 * NB;
  static constexpr int kChunks = kRows * BITS;
  static constexpr int kLoads = (kChunks + kWave - 1) / kWave;
  static constexpr int kPitch = 16 * (BITS | 1);
  static constexpr int kLdsBytes = kRows * kPitch + 16;  // a fragment may be read with up to 3 bytes after it
  static constexpr int kPiece = 4 * BITS / SPS;          // bytes of one lane and span
  static constexpr int kWords = (kPiece + 3) / 4;
  static constexpr int kMis = kPiece % 4 == 0 ? 0 : kPiece % 2 == 0 ? 2 : 3;  // largest misalignment of a piece
  static constexpr int kRead = (kPiece + kMis + 3) / 4;

  uint32_t off[kLoads];  // the lane's chunks: offset in the matrix
  uint32_t at[kLoads];   // ... and in LDS

  // chunk t of this lane (past the end: the last chunk again)
  static __device__ __forceinline__ int chunk(int lane, int t) { return min(t * kWave + lane, kChunks - 1); }
  __device__ __forceinline__ void init(const Params& p, int n0, int lane) {
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const int c = chunk(lane, t), row = c / BITS, seg = c - row * BITS;
      off[t] = (uint32_t)min(n0 + row, p.rows - 1) * (uint32_t)p.packed_cols + 16u * seg;
      at[t] = row * kPitch + 16 * seg;
    }
  }
  __device__ __forceinline__ void load(u32x4 (&r)[kLoads], const uint8_t* q, int stage) const {
#pragma unroll
    for (int t = 0; t < kLoads; ++t) r[t] = load16(q + (uint32_t)stage * (16u * BITS), off[t]);
  }
  // the stage that ends the row: only bytes that hold the row's codes
  __device__ __forceinline__ void load_last(u32x4 (&r)[kLoads], const Params& p, const uint8_t* q, int stage, int n0,
                                            int lane) const {
    const int row_bytes = (int)(((int64_t)p.cols * BITS + 7) >> 3);
#pragma unroll
    for (int t = 0; t < kLoads; ++t) {
      const int c = chunk(lane, t), row = c / BITS, seg = c - row * BITS;
      r[t] = load16_tail(q + (int64_t)min(n0 + row, p.rows - 1) * p.packed_cols, stage * (16 * BITS) + 16 * seg, row_bytes);
    }
  }
  __device__ __forceinline__ void store(char* lds, const u32x4 (&r)[kLoads]) const {
#pragma unroll
    for (int t = 0; t < kLoads; ++t) *reinterpret_cast<u32x4*>(lds + at[t]) = r[t];
  }
  // Span t's piece of row 16 j + nl, lane group g.  A piece may begin inside a
  // dword (the same place in all of a lane's): it is read with the dwords it
  // touches and shifted.
  static __device__ __forceinline__ void read(uint32_t (&w)[kWords], const char* lds, int j, int t, int nl, int g) {
    const char* src = lds + (16 * j + nl) * kPitch + t * (16 * BITS / SPS) + ((g * kPiece) & ~3);
    if constexpr (kMis == 0) {
      constexpr int align = kPiece % 16 == 0 ? 16 : kPiece % 8 == 0 ? 8 : 4;
      __builtin_memcpy(w, __builtin_assume_aligned(src, align), kWords * 4);
    } else {
      uint32_t d[kRead + 1];
      __builtin_memcpy(d, __builtin_assume_aligned(src, 4), kRead * 4);
      d[kRead] = 0;
      const uint32_t sh = ((g * kPiece) & 3) * 8;
#pragma unroll
      for (int i = 0; i < kWords; ++i) w[i] = __builtin_amdgcn_alignbit(d[i + 1], d[i], sh);
    }
  }
  // Step u of a piece (4 / SPS steps) as a fragment.
  static __device__ __forceinline__ f16x8 frag(const uint32_t (&w)[kWords], int u, const DecodeConsts& c) {
    const int bit = 8 * BITS * u, lo = bit >> 5, sh = bit & 31;
    auto word = [&](int i) -> uint32_t { return i < kWords ? w[i] : 0u; };
    const uint32_t w0 = sh ? __builtin_amdgcn_alignbit(word(lo + 1), word(lo), sh) : word(lo);
    const uint32_t w1 = BITS <= 4 ? 0u : (sh ? __builtin_amdgcn_alignbit(word(lo + 2), word(lo + 1), sh) : word(lo + 1));
    return decode8<BITS>(w0, w1, c);
  }
};

// The group scales of 16 NB rows of one stage: lane l < 16 NB loads row l's,
// the fragments' lanes fetch them from there.
template <int SPS, int NB>
struct Scales {
  uint32_t off;
  __device__ __forceinline__ void init(const Params& p, int n0, int lane) {
    off = (uint32_t)min(n0 + min(lane, 16 * NB - 1), p.rows - 1) * (uint32_t)p.scale_cols * 2u;
  }
  // (`last`: the last span that holds columns; spans past it count as scale 0,
  // so that an infinity in the last group's scale stays one)
  __device__ __forceinline__ void load(uint16_t (&r)[SPS], const Params& p, const uint16_t* s, int stage, int last) const {
#pragma unroll
    for (int t = 0; t < SPS; ++t) {
      const uint16_t v = *reinterpret_cast<const uint16_t*>(
          reinterpret_cast<const char*>(s + span_group(p, min(stage * SPS + t, last))) + off);
      r[t] = stage * SPS + t <= last ? v : (uint16_t)0;
    }
  }
  static __device__ __forceinline__ float get(uint16_t r, int j, int nl) {
    return h2f((uint16_t)__builtin_amdgcn_ds_bpermute((16 * j + nl) << 2, (int)(uint32_t)r));
  }
};

// Activation rows of a stage in LDS: 17 chunks of 16 bytes a row (16 of data).
constexpr int kXPitch = 17 * 16;

// ---------------------------------------------------------------------------
// Few rows of X (M <= 16 MB per workgroup): the W waves of a workgroup share
// 16 NB output rows and take every W-th stage each, with their own rows of W
// and X in LDS; their sums meet in LDS at the end, in wave order.
// ---------------------------------------------------------------------------
template <int BITS, int SPS, int MB, int NB, int W, int DEPTH>
__global__ __launch_bounds__(W* kWave) void skinny_kernel(Params p) {
  using Wt = Weights<BITS, SPS, NB>;
  using Sc = Scales<SPS, NB>;
  constexpr int kWaveBytes = 16 * MB * kXPitch + (Wt::kLdsBytes + 15) / 16 * 16;
  constexpr int kRedBytes = MB * NB * kWave * 16;
  constexpr int kLds = W * (kWaveBytes > kRedBytes ? kWaveBytes : kRedBytes);
  __shared__ __attribute__((aligned(16))) char smem[kLds];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nl = lane & 15, g = lane >> 4;
  const int n0 = blockIdx.x * (16 * NB), m0 = blockIdx.y * (16 * MB);
  const int mat = blockIdx.z;
  const uint8_t* const q = p.q[mat];
  const uint16_t* const sp = p.s[mat];
  const DecodeConsts dc = decode_consts();
  char* const xs = smem + wave * kWaveBytes;
  char* const ws = xs + 16 * MB * kXPitch;

  Wt wt;
  Sc sc;
  wt.init(p, n0, lane);
  sc.init(p, n0, lane);
  // activations: load t of a lane is chunk lane & 15 of row 4 t + lane / 16
  uint32_t xoff[4 * MB];  // bytes; the host keeps every operand below 4 GB
#pragma unroll
  for (int t = 0; t < 4 * MB; ++t)
    xoff[t] = ((uint32_t)min(m0 + 4 * t + g, p.batch - 1) * (uint32_t)p.x_stride + 8u * nl) * 2u;
  const int mrows = min(p.batch - m0, 16 * MB);

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  u32x4 raw[DEPTH][Wt::kLoads];
  u32x4 xv[DEPTH][4 * MB];
  uint16_t sv[DEPTH][SPS];

  auto issue = [&](int slot, int stage) __attribute__((always_inline)) {
    wt.load(raw[slot], q, stage);
    sc.load(sv[slot], p, sp, stage, 0x7fffffff);
#pragma unroll
    for (int t = 0; t < 4 * MB; ++t)
      if (4 * t < mrows) xv[slot][t] = load16(p.x + (uint32_t)stage * kStageK, xoff[t]);  // (uniform)
  };
  // a slot's data into LDS; its registers are free afterwards
  auto stage_lds = [&](int slot) __attribute__((always_inline)) {
    wt.store(ws, raw[slot]);
#pragma unroll
    for (int t = 0; t < 4 * MB; ++t)
      if (4 * t < mrows)
        *reinterpret_cast<u32x4*>(xs + (4 * t + g) * kXPitch + 16 * nl) = pair_order<BITS>(xv[slot][t]);
    asm volatile("" ::: "memory");  // the reads below are of other lanes' stores
  };
  auto compute = [&](const uint16_t (&sr)[SPS]) __attribute__((always_inline)) {
    constexpr int per = 4 / SPS;
#pragma unroll
    for (int t = 0; t < SPS; ++t) {
      f32x4 sum[MB][NB];
#pragma unroll
      for (int i = 0; i < MB; ++i)
#pragma unroll
        for (int j = 0; j < NB; ++j) sum[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
      uint32_t w[NB][Wt::kWords];
#pragma unroll
      for (int j = 0; j < NB; ++j) Wt::read(w[j], ws, j, t, nl, g);
#pragma unroll
      for (int u = 0; u < per; ++u) {
        f16x8 a[MB];
#pragma unroll
        for (int i = 0; i < MB; ++i)
          a[i] = *reinterpret_cast<const f16x8*>(xs + (16 * i + nl) * kXPitch + 2 * frag_k<SPS>(g, t * per + u));
#pragma unroll
        for (int j = 0; j < NB; ++j) {
          const f16x8 b = Wt::frag(w[j], u, dc);
#pragma unroll
          for (int i = 0; i < MB; ++i) sum[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a[i], b, sum[i][j], 0, 0, 0);
        }
      }
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        const float s = Sc::get(sr[t], j, nl);
#pragma unroll
        for (int i = 0; i < MB; ++i)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(s, sum[i][j][e], acc[i][j][e]);
      }
    }
    asm volatile("" ::: "memory");  // the next stage's stores stay behind these reads
  };

  const int plain = p.cols / kStageK;           // whole stages
  const int mine = (plain - wave + W - 1) / W;  // stages wave, wave + W, ...
  if (mine > 0) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      issue(i, wave + W * min(i, mine - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int b = 0; b < mine; b += DEPTH) {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) {
        if (b + i < mine) {
          uint16_t sr[SPS];
#pragma unroll
          for (int t = 0; t < SPS; ++t) sr[t] = sv[i][t];
          stage_lds(i);
          __builtin_amdgcn_sched_barrier(0);
          issue(i, wave + W * min(b + i + DEPTH, mine - 1));  // past the end: the last stage again, not used
          __builtin_amdgcn_sched_barrier(0);
          compute(sr);
        }
      }
    }
  }
  // the stage that ends the row, where it is ragged
  if (plain * kStageK < p.cols && wave == plain % W) {
    wt.load_last(raw[0], p, q, plain, n0, lane);
    sc.load(sv[0], p, sp, plain, (p.cols - 1) / (kStageK / SPS));
#pragma unroll
    for (int t = 0; t < 4 * MB; ++t)
      if (4 * t < mrows)
        xv[0][t] = load16_tail(
            reinterpret_cast<const uint8_t*>(p.x + (int64_t)min(m0 + 4 * t + g, p.batch - 1) * p.x_stride),
            2 * (plain * kStageK + 8 * nl), 2 * p.cols);
    stage_lds(0);
    compute(sv[0]);
  }

  f32x4* const red = reinterpret_cast<f32x4*>(smem);  // [W][MB NB][64]
  __syncthreads();                                    // every wave is done with its rows
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) red[(wave * (MB * NB) + i * NB + j) * kWave + lane] = acc[i][j];
  __syncthreads();
  for (int e = tid; e < MB * NB * kWave; e += W * kWave) {
    const int blk = e >> 6, l = e & 63;
    f32x4 v = red[e];
#pragma unroll
    for (int w = 1; w < W; ++w) v += red[w * (MB * NB * kWave) + e];
    const int m = m0 + 16 * (blk / NB) + 4 * (l >> 4), n = n0 + 16 * (blk % NB) + (l & 15);
    if (n < p.rows) {
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (m + r < p.batch) p.y[mat][(int64_t)(m + r) * p.y_stride + n] = f2h(v[r]);
    }
  }
}

// ---------------------------------------------------------------------------
// Many rows of X: a workgroup tile of 16 MB batch rows x 64 NB output rows; its
// four waves take 16 NB output rows each (their own in LDS, as above) and share
// X through LDS, one stage (16 MB rows x 128 k) at a time in two buffers,
// staged through registers in decode8's pair order.
// ---------------------------------------------------------------------------
constexpr int kTileThreads = 256;

template <int BITS, int SPS, int MB, int NB, int DEPTH, int OCC>
__global__ __launch_bounds__(kTileThreads, OCC) void tile_kernel(Params p) {
  using Wt = Weights<BITS, SPS, NB>;
  using Sc = Scales<SPS, NB>;
  constexpr int BM = 16 * MB;
  constexpr int kWt = (Wt::kLdsBytes + 15) / 16 * 16;
  __shared__ __attribute__((aligned(16))) char smem[2 * BM * kXPitch + 4 * kWt];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int nl = lane & 15, g = lane >> 4;
  const int n0 = (blockIdx.x * 4 + wave) * (16 * NB), m0 = blockIdx.y * BM;
  const uint8_t* const q = p.q[0];
  const uint16_t* const sp = p.s[0];
  const DecodeConsts dc = decode_consts();
  char* const ws = smem + 2 * BM * kXPitch + wave * kWt;

  Wt wt;
  Sc sc;
  wt.init(p, n0, lane);
  sc.init(p, n0, lane);
  // staging: item t of this thread is chunk tid & 15 of row tid / 16 + 16 t
  const int xc = tid & 15, xr = tid >> 4;
  auto xrow = [&](int t) __attribute__((always_inline)) {
    return (uint32_t)min(m0 + xr + 16 * t, p.batch - 1) * (uint32_t)p.x_stride;
  };
  u32x4 xl[DEPTH][MB];
  u32x4 raw[DEPTH][Wt::kLoads];
  uint16_t sv[DEPTH][SPS];
  auto load_stage = [&](int slot, int stage) __attribute__((always_inline)) {
    wt.load(raw[slot], q, stage);
    sc.load(sv[slot], p, sp, stage, 0x7fffffff);
#pragma unroll
    for (int t = 0; t < MB; ++t) xl[slot][t] = load16(p.x + (uint32_t)stage * kStageK, (xrow(t) + 8u * xc) * 2u);
  };
  auto load_last = [&](int stage) __attribute__((always_inline)) {
    wt.load_last(raw[0], p, q, stage, n0, lane);
    sc.load(sv[0], p, sp, stage, (p.cols - 1) / (kStageK / SPS));
#pragma unroll
    for (int t = 0; t < MB; ++t)
      xl[0][t] = load16_tail(reinterpret_cast<const uint8_t*>(p.x + xrow(t)), 2 * (stage * kStageK + 8 * xc), 2 * p.cols);
  };
  auto store_x = [&](int slot, int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int t = 0; t < MB; ++t)
      *reinterpret_cast<u32x4*>(smem + (buf * BM + xr + 16 * t) * kXPitch + 16 * xc) = pair_order<BITS>(xl[slot][t]);
  };

  f32x4 acc[MB][NB];
#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) acc[i][j] = (f32x4){0.f, 0.f, 0.f, 0.f};
  auto compute = [&](int buf, const uint16_t (&sr)[SPS]) __attribute__((always_inline)) {
    constexpr int per = 4 / SPS;
    const char* xb = smem + buf * BM * kXPitch;
#pragma unroll
    for (int t = 0; t < SPS; ++t) {
      f16x8 b[per][NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) {
        uint32_t w[Wt::kWords];
        Wt::read(w, ws, j, t, nl, g);
#pragma unroll
        for (int u = 0; u < per; ++u) b[u][j] = Wt::frag(w, u, dc);
      }
      float s[NB];
#pragma unroll
      for (int j = 0; j < NB; ++j) s[j] = Sc::get(sr[t], j, nl);
#pragma unroll
      for (int i = 0; i < MB; ++i) {
        f32x4 sum[NB];
#pragma unroll
        for (int j = 0; j < NB; ++j) sum[j] = (f32x4){0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < per; ++u) {
          const f16x8 a = *reinterpret_cast<const f16x8*>(xb + (16 * i + nl) * kXPitch + 2 * frag_k<SPS>(g, t * per + u));
#pragma unroll
          for (int j = 0; j < NB; ++j) sum[j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b[u][j], sum[j], 0, 0, 0);
        }
#pragma unroll
        for (int j = 0; j < NB; ++j)
#pragma unroll
          for (int e = 0; e < 4; ++e) acc[i][j][e] = __builtin_fmaf(s[j], sum[j][e], acc[i][j][e]);
        if (i & 1) __builtin_amdgcn_sched_barrier(0);  // bounds the registers live at a time
      }
    }
  };
  // the loaded stage into LDS (buffer `buf` of X); every wave's X is there
  // after the barrier, and the buffer of the stage before it is free
  auto publish_stage = [&](int slot, int buf, uint16_t (&sr)[SPS]) __attribute__((always_inline)) {
    store_x(slot, buf);
    wt.store(ws, raw[slot]);
#pragma unroll
    for (int t = 0; t < SPS; ++t) sr[t] = sv[slot][t];
    lds_barrier();
  };

  const int plain = p.cols / kStageK;
  if (plain > 0) {
#pragma unroll
    for (int i = 0; i < DEPTH; ++i) {
      load_stage(i, min(i, plain - 1));
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int b = 0; b < plain; b += DEPTH) {
#pragma unroll
      for (int i = 0; i < DEPTH; ++i) {
        const int s = b + i;
        if (s < plain) {
          uint16_t sr[SPS];
          publish_stage(i, s & 1, sr);
          load_stage(i, min(s + DEPTH, plain - 1));  // past the end: the last stage again, not used
          __builtin_amdgcn_sched_barrier(0);
          compute(s & 1, sr);
        }
      }
    }
  }
  if (plain * kStageK < p.cols) {
    uint16_t sr[SPS];
    load_last(plain);
    publish_stage(0, plain & 1, sr);
    compute(plain & 1, sr);
  }

#pragma unroll
  for (int i = 0; i < MB; ++i)
#pragma unroll
    for (int j = 0; j < NB; ++j) {
      const int n = n0 + 16 * j + nl;
      if (n < p.rows) {
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const int m = m0 + 16 * i + 4 * g + e;
          if (m < p.batch) p.y[0][(int64_t)m * p.y_stride + n] = f2h(acc[i][j][e]);
        }
      }
    }
}

}  // namespace rwmm
}  // namespace lb
