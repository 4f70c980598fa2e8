// Marlin-layout W4A16 projection for skinny batches (decode: M <= 32) on gfx950.
//
// Reads the reference's Marlin layout (langburst/csrc/marlin_cuda_kernel.cu,
// packing in adapters/qwen36_tools/quantize.py:180-243) directly; no repack.
//
// Layout facts used (derived from quantize.py:50-76):
//   qweight int32 [K/16, 2N].  Row kb holds k = 16kb..16kb+15.  Each 64-column
//   "chunk" of a row is 128 int32 = 512 contiguous bytes = 32 16-byte slots.
//   Slot i (0..31), with c = i>>2 and q = i&3, holds 4 words j = 0..3; word j
//   covers columns 16j+c (bytes 0,2) and 16j+c+8 (bytes 1,3) of the chunk:
//   the low nibbles of bytes 0/2 are k = 2q / 2q+1, the high nibbles
//   k = 2q+8 / 2q+9.  Group scales: the 64-column chunk of group row g stores
//   column 8jj+i at 8i+jj, so the 8 scales a slot needs are the 16 bytes at 8c.
//
// Kernel.  A workgroup owns cpw chunks (64 * cpw columns, cpw = 4, 2 or 1)
// and a k range; wave w streams chunk w % cpw over share w / cpw of that k
// range (4 / cpw shares, whole scale groups), and the shares of a column are
// added in the epilogue in share order.  cpw < 4 serves narrow N: more,
// narrower tiles instead of many k splits.  The B fragment of v_mfma_f32_16x16x32_f16 (lane
// l = 16g + nl holds 8 k-values of column nl) is built in registers: with
// k-group g = (row p = g>>1, slot pair 4c+2g', 4c+2g'+1, g' = g&1) and column
// nl = 8h + c, the fragment needs the h half of every word of both slots of
// the pair: (q0 k0,k1)(q1 k0,k1)(q0 k8,k9)(q1 k8,k9) = physical k 4g'+{0..3}
// and 4g'+8+{0..3} of row p.  Lane l loads only slot 4c+2g'+h, so the 32
// lanes of a row fetch its 512 bytes once; the other slot of the pair is in
// lane l^8 and arrives by a DPP row rotation, and one v_perm_b32 gathers the
// four bytes the lane uses.  Dequant per fp16 pair: one v_and_or_b32 gives
// the biased 1024 + q (k = 0..7 of a row, low nibbles) or 1024 + 16q
// (k = 8..15, high nibbles), one packed add (or fma by 1/16) makes it the
// exact q - 8, and one packed multiply by the group's scale gives the
// reference's fp16 (q - 8) * s, rounded as marlin_cuda_kernel.cu:131-159
// rounds it; the MFMA then accumulates exact products in fp32.
//
// Latency.  A ring of kDepth weight batches (one scale group, 1 KB per wave
// each) stays in flight, with unconditional loads, so the memory counters
// never force a full drain.  The A operand comes one of three ways (the host
// planner picks per shape):
//   staged (M <= 16): the activation slice of the workgroup's k range is
//     staged once in LDS in fragment order ([k/32][4 k-groups][m] x 16 bytes,
//     SiLU-gated variant: fp16(silu(g) * u)); the staging loads are issued
//     first and the first weight batches right behind them, so the staging
//     round trip overlaps the weight fetch;
//   direct (narrow tiles, and M = 5..32 whole-K tiles; MR = 2 row blocks of 16
//     above 16 rows): each lane loads its own A fragments (16 bytes per row
//     block and step, from L2, completed by a lane swap) with the weight batch
//     they meet, in the same ring; no LDS, no barrier before the loop;
//   ring (4-chunk tiles, M <= 32): one scale group of A at a time through a
//     two-slot LDS ring shared by the four waves.

// Epilogue.  Accumulators go through an LDS tile [M][256]; for plain stores
// every thread then takes one column and every (4 / cpw)-th row of it, for
// the SiLU-gated and argmax epilogues thread t owns column t.  Under split-K
// each workgroup publishes fp32 partials to scratch [S][M][N]; the last one to
// arrive on the tile's counter (workspace, zero on entry and on exit)
// collects them in split order (deterministic), rounds to fp16 and stores or
// feeds the fused argmax.  4-chunk tiles with plain stores skip the tile: each
// wave hands off its own chunk.

#pragma once
#include "lb_common.hpp"

namespace lb {
namespace skinny {

constexpr int kWaves = 4;               // chunks (64 columns each) per workgroup
constexpr int kThreads = kWaves * kWave;
constexpr int kCols = 64 * kWaves;      // 256 columns per workgroup
constexpr int kMaxM = 16;               // rows of the MFMA tile; the staged-A modes' M limit
constexpr int kMaxMR = 2;               // A_DIRECT: 16-row blocks per MFMA tile (M <= 32)
constexpr int kSteps = 4;               // 32-k steps per batch (one scale group)
constexpr int kStageUnroll = 8;         // A staging: 16-byte items in flight per thread
constexpr int kDepth = 2;               // weight batches in flight

// A_DIRECT: plain fp16 A, not staged: fragments loaded per step (M up to 32).
// A_RING: plain fp16 A staged one batch (one scale group) at a time through a
// two-slot LDS ring, for 4-chunk tiles whose waves share it (M up to 32).
// A_WAVE: as A_DIRECT, each wave's batch of A through LDS of its own (M = 29..32).
enum AMode { A_PLAIN = 0, A_SILU_PACKED = 1, A_DIRECT = 3, A_RING = 4, A_WAVE = 5 };
constexpr int kWaveRowBytes = 17 * 16;  // A_WAVE: one LDS row of a batch, 128 k and 16 bytes of padding
// dynamic LDS of an A_WAVE workgroup of `mr` 16-row blocks
__host__ __device__ constexpr int wave_a_bytes(int mr) { return kWaves * 16 * mr * kWaveRowBytes; }
// EPI_ACT: the tile pairs gate and up chunks (gate_up projection of an MLP)
// and stores fp16(silu(g) * u) of its fp16 outputs instead of the outputs.
enum EpiMode { EPI_STORE = 0, EPI_ARGMAX = 1, EPI_ACT = 2 };

struct Params {
  const uint16_t* a;     // x [M, K] (A_PLAIN) or mixed [M, 2K] (A_SILU_PACKED)
  const uint32_t* b;     // qweight [K/16, 2N]
  const uint16_t* s;     // scales
  uint16_t* c;           // out [M, N] (EPI_STORE)
  int32_t* counters;     // workspace: [0] argmax arrival counter, [1 + tile] split-K counters
  float* partial;        // scratch: [S][M][N] fp32 partials (S > 1)
  uint64_t* tile_keys;   // scratch: [M][n_cg] argmax keys (EPI_ARGMAX)
  int64_t* argmax_state; // [M]
  int64_t* argmax_out;   // [M]
  int m, n, k;
  int splits;            // S
  int kp_total;          // K / 32
  int n_cg;              // N / (64 * cpw): column tiles
  uint32_t* act_out;     // EPI_ACT: fp16 pairs [M][N / 4] (N / 2 neurons)
  int gate_chunks;       // EPI_ACT: N / 128, chunks of the gate half
};

__device__ __forceinline__ float silu(float v) { return v / (1.0f + __expf(-v)); }

// Order-preserving key: larger value wins, then smaller column.
__device__ __forceinline__ uint64_t argmax_key(float v, uint32_t col) {
  const uint32_t bits = __builtin_bit_cast(uint32_t, v);
  const uint32_t ord = (bits & 0x80000000u) ? ~bits : (bits ^ 0x80000000u);
  return ((uint64_t)ord << 32) | (uint64_t)(0xffffffffu - col);
}

__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }

__device__ __forceinline__ uint64_t wave_max_u64(uint64_t v) {
  const int lane = __builtin_amdgcn_mbcnt_hi(~0u, __builtin_amdgcn_mbcnt_lo(~0u, 0u));
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(((lane ^ off) & 63) << 2, (int)(uint32_t)v);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(((lane ^ off) & 63) << 2, (int)(uint32_t)(v >> 32));
    v = max_u64(v, ((uint64_t)hi << 32) | lo);
  }
  return v;
}

// Splits are whole scale groups (4 k-steps of 32) balanced over S.  32-bit
// arithmetic: the host keeps groups * S below 2^32 (K <= 2^30, S <= 256).
__device__ __forceinline__ void split_range(const Params& p, int split, int& kp0, int& kp1) {
  const uint32_t groups = (uint32_t)p.kp_total >> 2;
  const uint32_t g0 = (groups * (uint32_t)split) / (uint32_t)p.splits;
  const uint32_t g1 = (groups * (uint32_t)(split + 1)) / (uint32_t)p.splits;
  kp0 = (int)(g0 << 2);
  kp1 = (int)(g1 << 2);
}

// Inverse of the per-column scale permutation (quantize.py:66-68).
__device__ __forceinline__ int per_column_scale_index(int n) {
  const int r = n & 31;
  return (n & ~31) + 8 * ((r >> 1) & 3) + ((r >> 3) << 1) + (r & 1);
}

__device__ __forceinline__ uint32_t silu_mul2(uint32_t g, uint32_t u) {
  const float g0 = h2f((uint16_t)(g & 0xffffu)), g1 = h2f((uint16_t)(g >> 16));
  const float u0 = h2f((uint16_t)(u & 0xffffu)), u1 = h2f((uint16_t)(u >> 16));
  return (uint32_t)f2h(silu(g0) * u0) | ((uint32_t)f2h(silu(g1) * u1) << 16);
}

// Global chunk (64 columns) of chunk c (0 .. CPW-1) of column tile cg.  EPI_ACT
// pairs the gate and up halves of a gate_up projection: chunks 0 .. CPW/2-1
// are gate chunks, the rest the up chunks of the same neurons.
template <int EPI, int CPW>
__device__ __forceinline__ int tile_chunk(const Params& p, int cg, int c) {
  if (EPI == EPI_ACT) {
    constexpr int h = CPW / 2;
    return c < h ? cg * h + c : p.gate_chunks + cg * h + (c - h);
  }
  return cg * CPW + c;
}

// The split-K collect of a tile: sums the T shares of columns [col0, col0 +
// 4 CQ) of every row in share order (deterministic), rounds to fp16 (the
// per-column scale after that, as the reference does) and hands each value to
// `store(row, column - col0, fp16 bits)` (the output, or the SiLU-gated
// epilogue's LDS exchange).
// Thread t (of NT) takes column quad t % CQ and rows t / CQ + (NT / CQ) i, and
// keeps every row's loads of up to kSU shares in flight together (16-byte
// device-coherent loads, at most kMaxLoads per thread): the collect costs one
// memory round trip per kSU shares, not one per four rows.
template <bool GROUPED, int CQ, int NT, int ROWS, int kMaxLoads, typename Store>
__device__ __forceinline__ void collect_store(const Params& p, int total, int col0, int t, Store store) {
  constexpr int kRowStep = NT / CQ;
  constexpr int kRowIters = (ROWS + kRowStep - 1) / kRowStep;
  constexpr int kSU = kMaxLoads / kRowIters < 1 ? 1 : kMaxLoads / kRowIters > 8 ? 8 : kMaxLoads / kRowIters;
  const int mrows = p.m;
  const int64_t share_stride = (int64_t)mrows * p.n;
  // The partials of a skinny plan stay far below 4 GB (the planner keeps
  // S * M * N small), so 32-bit buffer offsets address them.
  const __amdgpu_buffer_rsrc_t rp = buffer_of(p.partial, (uint32_t)((int64_t)total * share_stride * 4));
  const int cq = t % CQ, rs = t / CQ;
  const int ncol = col0 + 4 * cq;
  f32x4 sum[kRowIters];
#pragma unroll
  for (int i = 0; i < kRowIters; ++i) sum[i] = (f32x4){0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < total; s0 += kSU) {
    f32x4 tv[kRowIters][kSU];
#pragma unroll
    for (int i = 0; i < kRowIters; ++i)
#pragma unroll
      for (int u = 0; u < kSU; ++u) {
        const int row = rs + kRowStep * i;
        if (row < mrows) {
          const int64_t e = (int64_t)min(s0 + u, total - 1) * share_stride + (int64_t)row * p.n + ncol;
          tv[i][u] = collect16(rp, (uint32_t)(e * 4));
        }
      }
#pragma unroll
    for (int i = 0; i < kRowIters; ++i)
#pragma unroll
      for (int u = 0; u < kSU; ++u)
        if (rs + kRowStep * i < mrows && s0 + u < total) sum[i] += tv[i][u];
  }
  f16 cs[4];
#pragma unroll
  for (int e = 0; e < 4; ++e)
    cs[e] = GROUPED ? (f16)1.0f : __builtin_bit_cast(f16, p.s[per_column_scale_index(ncol + e)]);
#pragma unroll
  for (int i = 0; i < kRowIters; ++i) {
    const int row = rs + kRowStep * i;
    if (row < mrows) {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        f16 h = (f16)sum[i][e];
        if (!GROUPED) h = h * cs[e];
        store(row, ncol - col0 + e, __builtin_bit_cast(uint16_t, h));
      }
    }
  }
}

// Plain-store epilogue, one wave on its own (no LDS, no workgroup barrier).
// The wave holds the fp32 sums of one 64-column chunk over its share of K:
// acc[rb][j][i] is row 16 rb + 4 (lane >> 4) + i, column 16 j + (lane & 15)
// of the chunk.  Shares are the k splits times the k shares of a workgroup,
// T = S * ksub, numbered split-major.  T == 1: the wave rounds and stores its
// outputs.  Otherwise it publishes its partial (device-coherent stores into
// partial [T][M][N]), waits for their acknowledgement, and counts its arrival
// on the chunk's counter (workspace entry 1 + chunk); the wave that completes
// the count reads the T partials of the chunk in share order (deterministic),
// rounds, stores, and resets the counter.  Returns true in the wave that
// stored the chunk's outputs.
template <bool GROUPED, int MR>
__device__ __forceinline__ bool wave_epilogue(const Params& p, const f32x4 (&acc)[MR][4], int chunk, int share,
                                              int ksub) {
  const int lane = threadIdx.x & 63;
  const int mrows = p.m;
  const int total = p.splits * ksub;
  const int crow0 = (lane >> 4) * 4;
  const int col0 = chunk * 64;
  if (total == 1) {
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const int n = col0 + 16 * j + (lane & 15);
      const f16 cs = GROUPED ? (f16)1.0f : __builtin_bit_cast(f16, p.s[per_column_scale_index(n)]);
#pragma unroll
      for (int rb = 0; rb < MR; ++rb)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * rb + crow0 + i;
          f16 h = (f16)acc[rb][j][i];
          if (!GROUPED) h = h * cs;
          if (r < mrows) p.c[(int64_t)r * p.n + n] = __builtin_bit_cast(uint16_t, h);
        }
    }
    return true;
  }
  const int64_t share_stride = (int64_t)mrows * p.n;
  float* part = p.partial + share * share_stride + col0 + (lane & 15);
#pragma unroll
  for (int rb = 0; rb < MR; ++rb)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (16 * rb + crow0 + i < mrows) publish(part + (int64_t)(16 * rb + crow0 + i) * p.n + 16 * j, acc[rb][j][i]);
  wait_published();
  int32_t* ctr = p.counters + 1 + chunk;
  int prev = 0;
  if (lane == 0) prev = arrive(ctr);
  prev = __builtin_amdgcn_readfirstlane(prev);
  if (prev != total - 1) return false;
  after_last_arrival();
  if (lane == 0) __hip_atomic_store(ctr, 0, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  if (MR == 1 && mrows <= 4) {
    // Few rows: lane = column, the 4 rows x 8 shares of 4-byte loads in flight
    // (one round trip up to 8 shares; measured faster here than the 16-byte
    // form, which leaves 48 of the 64 lanes idle).
    const int n = col0 + lane;
    const float* src = p.partial + n;
    const f16 cs = GROUPED ? (f16)1.0f : __builtin_bit_cast(f16, p.s[per_column_scale_index(n)]);
    float sum[4] = {0.f, 0.f, 0.f, 0.f};
    for (int s0 = 0; s0 < total; s0 += 8) {
      float tv[4][8];
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < 8; ++u)
          tv[i][u] = collect(src + (int64_t)min(s0 + u, total - 1) * share_stride + (int64_t)min(i, mrows - 1) * p.n);
#pragma unroll
      for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int u = 0; u < 8; ++u) sum[i] += (s0 + u < total) ? tv[i][u] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      f16 h = (f16)sum[i];
      if (!GROUPED) h = h * cs;
      if (i < mrows) p.c[(int64_t)i * p.n + n] = __builtin_bit_cast(uint16_t, h);
    }
    return true;
  }
  // (MR = 2: fewer loads in flight, so that two workgroups still fit a CU)
  collect_store<GROUPED, 16, kWave, 16 * MR, MR == 1 ? 32 : 16>(
      p, total, col0, lane, [&](int row, int col, uint16_t v) { p.c[(int64_t)row * p.n + col0 + col] = v; });
  return true;
}

// One workgroup's share of the projection: column tile cg (64 * CPW columns),
// k split `split`.  CPW: chunks per workgroup (4, 2 or 1), a compile-time
// constant so that the wide-N instantiation (CPW = 4) carries no k-share
// arithmetic.  Uses the kernel's dynamic LDS.  Returns true in the workgroup
// that stored the tile's outputs (EPI_STORE, EPI_ACT) or ran the launch's
// final argmax reduction.
template <int AM, int EPI, bool GROUPED, int CPW, int MR = 1>
__device__ __forceinline__ bool skinny_tile(const Params p, const int cg, const int split) {
  static_assert(EPI != EPI_ACT || CPW >= 2, "EPI_ACT pairs a gate and an up chunk");
  static_assert(MR == 1 || ((AM == A_DIRECT || AM == A_RING || AM == A_WAVE) && (EPI == EPI_STORE || EPI == EPI_ACT)),
                "row blocks > 1: direct or ring A, store or SiLU-gated epilogue");
  static_assert(MR >= 1 && MR <= kMaxMR, "row blocks");
  static_assert(AM != A_RING || (CPW == kWaves && EPI != EPI_ARGMAX), "A ring: 4-chunk tiles");
  constexpr bool kDirect = AM == A_DIRECT;
  constexpr bool kRing = AM == A_RING;
  constexpr bool kWaveA = AM == A_WAVE;
  constexpr int kRows = 16 * MR;  // rows of the MFMA tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ int s_prev;
  __shared__ uint64_t s_keys[kWaves][kMaxM];
  // Every kernel argument the prologue needs, named before any other work
  // (the kernels pass them as scalar arguments, preloaded into SGPRs).
  asm volatile("" ::"s"(p.a), "s"(p.b), "s"(p.s), "s"(p.m), "s"(p.n), "s"(p.k), "s"(p.splits), "s"(p.kp_total));
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // uniform: the ring's offsets stay scalar
  const int lane = tid & 63;
  const int mrows = p.m;      // <= kRows
  constexpr int cpw = CPW;
  constexpr int ksub = kWaves / cpw;   // k shares per tile
  const int wchunk = cpw == kWaves ? wave : (wave & (cpw - 1));  // this wave's chunk of the tile ...
  const int wsub = cpw == kWaves ? 0 : wave / cpw;                // ... and its k share

  int kp0, kp1;
  split_range(p, split, kp0, kp1);  // the workgroup's k range
  const int nkp = kp1 - kp0;  // positive multiple of kSteps
  const int ngw = nkp / kSteps;  // scale groups of the workgroup
  // this wave's groups [gw0, gw0 + nb) of them (nb >= 1: the host plans at
  // least ksub groups per split)
  const int gw0 = (ngw * wsub) / ksub;
  const int nb = (ngw * (wsub + 1)) / ksub - gw0;
  const int kpw0 = kp0 + gw0 * kSteps;

  // fragment coordinates: lane = 16g + 8h + c
  const int chunk = EPI == EPI_ACT ? tile_chunk<EPI, CPW>(p, cg, wchunk) : cg * cpw + wchunk;
  const uint32_t row_bytes = (uint32_t)p.n * 8u;  // one qweight row: 2N int32
  const int g = lane >> 4;
  const int hsel = (lane >> 3) & 1;
  const int cc = lane & 7;
  const int prow = g >> 1;  // which of the two k16 rows of a 32-k step
  const int gq = g & 1;     // slot pair (q0, q1) = (2gq, 2gq+1)
  // Each lane loads one slot, 4c + 2gq + h; the pair's other slot comes from
  // lane ^ 8 (same c and g, other h) by a DPP row rotation.
  // The lane's offset into the weights and scales is a fixed 32-bit VGPR and
  // each step's row offset a wave-uniform scalar (32-bit: the host keeps the
  // weights below 4 GB), so the ring costs two VALU per 16-byte load instead
  // of a 64-bit multiply-add.  Weights and scales are read once: non-temporal
  // loads.  The scales come through a buffer descriptor (with the weights as
  // buffer loads too, the compiler drains the ring at the loop head).
  const __amdgpu_buffer_rsrc_t rbs = buffer_of(p.s, (uint32_t)(p.k >> 7) * (uint32_t)p.n * 2u);
  const uint32_t bvoff = (uint32_t)prow * row_bytes + (uint32_t)chunk * 512u + (uint32_t)(cc * 4 + gq * 2 + hsel) * 16u;
  const uint32_t svoff = (uint32_t)chunk * 128u + (uint32_t)cc * 16u;
  const uint32_t step_bytes = 2u * row_bytes;      // one 32-k step: two qweight rows
  const uint32_t group_bytes = (uint32_t)p.n * 2u;  // one row of group scales
  // Byte selection of v_perm_b32(own, partner): word = [A.b_h, B.b_h, A.b_(2+h), B.b_(2+h)]
  // with A = slot 4c+2gq (q0) and B = slot 4c+2gq+1 (q1).
  const uint32_t psel = hsel ? 0x07030501u : 0x02060004u;
  const int mrow = lane & 15;  // A fragment row
  const NibConsts nk = nib_consts();

  // LDS: staged A in fragment order, entry (kp, g, m) = 16 bytes holding
  // x[m][32kp + 16(g>>1) + 4(g&1) + {0..3}] and the same + 8, then one zero
  // entry (read by the lanes of rows >= M).
  u32x4* afr = reinterpret_cast<u32x4*>(smem);
  const int k0 = kp0 * 32;
  const int octs = nkp * 4;            // 8-half runs per row of the slice
  const int items = octs * mrows;
  const int n_frag = nkp * 4 * mrows;  // staged entries; afr[n_frag] is the zero entry
  // Item it is octet it % octs of row it / octs.  The staged slice fits LDS, so
  // it and octs stay below 2^16, where umulhi(it, ceil(2^32 / octs)) is exactly
  // it / octs (the error term it * (ceil(2^32 / octs) * octs - 2^32) / 2^32 < 1 / octs
  // never reaches the next integer); octs >= 16.
  const uint32_t oct_magic = 0xffffffffu / (uint32_t)octs + 1u;
  const int64_t a_row_stride = AM == A_SILU_PACKED ? 2 * (int64_t)p.k : (int64_t)p.k;
  uint4 gv[kStageUnroll], uv[kStageUnroll];
  auto stage_load = [&](int base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int it = min(base + u * kThreads + tid, items - 1);
      const int mm = (int)__umulhi((uint32_t)it, oct_magic);
      const int r = it - mm * octs;
      const uint16_t* src = p.a + (int64_t)mm * a_row_stride + k0 + (r << 3);
      gv[u] = *reinterpret_cast<const uint4*>(src);
      if (AM == A_SILU_PACKED) uv[u] = *reinterpret_cast<const uint4*>(src + p.k);
    }
  };
  auto stage_store = [&](int base) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kStageUnroll; ++u) {
      const int it = base + u * kThreads + tid;
      if (it < items) {
        const int mm = (int)__umulhi((uint32_t)it, oct_magic);
        const int r = it - mm * octs;  // kp = r >> 2, octet o = r & 3 = 2 prow + half
        uint4 w = gv[u];
        if (AM == A_SILU_PACKED)
          w = make_uint4(silu_mul2(w.x, uv[u].x), silu_mul2(w.y, uv[u].y), silu_mul2(w.z, uv[u].z),
                         silu_mul2(w.w, uv[u].w));
        const int fg = ((r >> 2) * 4 + ((r & 3) >> 1) * 2) * mrows + mm;  // fragment (kp, g = 2 prow)
        uint2* dst = reinterpret_cast<uint2*>(afr + fg) + (r & 1);
        dst[0] = make_uint2(w.x, w.y);          // halves 0..3 -> g = 2 prow
        dst[2 * mrows] = make_uint2(w.z, w.w);  // halves 4..7 -> g = 2 prow + 1
      }
    }
  };

  // A_DIRECT: lane (g, row mrow) of row block rb needs row min(16 rb + mrow,
  // M - 1) (rows >= M compute values that are never stored) at k offsets
  // 32 kp + 16 prow + 4 gq + {0..3} and the same + 8 (the staged entry's
  // contents).  It loads the 16 contiguous bytes at 32 kp + 16 prow + 8 gq
  // instead; the lanes of gq = 0 and gq = 1 (rows 2 prow and 2 prow + 1 of the
  // wave) then hold each other's missing halves, which two
  // v_permlane16_swap exchange at use.
  const uint16_t* arow[MR];
#pragma unroll
  for (int rb = 0; rb < MR; ++rb)
    arow[rb] = p.a + (int64_t)min(16 * rb + mrow, mrows - 1) * p.k + 16 * prow + 8 * gq;

  // A_RING: batch b of the workgroup's A (rows x 128 k, fragment order as
  // staged above) lives in LDS slot b & 1; thread t loads 16-byte items
  // t + 256 u (row it >> 4, octet it & 15) of batch b + 1 two batches ahead
  // into registers, stores them while batch b is consumed, and one LDS barrier
  // per batch publishes them (and frees the slot of batch b - 1).
  constexpr int kRingItems = (16 * kRows + kThreads - 1) / kThreads;
  const int ring_slot = 16 * mrows;  // fragment entries per slot
  const int ring_zero = 2 * ring_slot;
  u32x4 ar[kDepth][kRingItems];
  u32x4 ar0[kRingItems];
  auto ring_load = [&](u32x4(&dst)[kRingItems], int batch) __attribute__((always_inline)) {
    const int kb = 32 * (kpw0 + batch * kSteps);
#pragma unroll
    for (int u = 0; u < kRingItems; ++u) {
      const int it = tid + kThreads * u;
      const int mm = min(it >> 4, mrows - 1);
      dst[u] = *reinterpret_cast<const u32x4*>(p.a + (int64_t)mm * p.k + kb + 8 * (it & 15));
    }
  };
  auto ring_store = [&](const u32x4(&src)[kRingItems], int lslot) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < kRingItems; ++u) {
      const int it = tid + kThreads * u;
      const int mm = it >> 4, o = it & 15;  // o = 4 d + 2 prow + half
      if (mm < mrows) {
        const int fg = lslot * ring_slot + ((o >> 2) * 4 + ((o & 3) >> 1) * 2) * mrows + mm;
        uint2* dst = reinterpret_cast<uint2*>(afr + fg) + (o & 1);
        dst[0] = make_uint2(src[u][0], src[u][1]);          // halves 0..3 -> g = 2 prow
        dst[2 * mrows] = make_uint2(src[u][2], src[u][3]);  // halves 4..7 -> g = 2 prow + 1
      }
    }
  };

  // A_WAVE: with A_DIRECT's loads neighbouring lanes read different rows, and
  // every row a sixteen-lane group touches is a cache-line access of its own
  // (M = 16: 64 a load instruction).  Here load u of a lane is the 16 bytes at
  // octet lane & 15 of row 4 u + (lane >> 4) of the batch (four rows of 256
  // contiguous bytes an instruction, 8 cache lines), and the fragments come from
  // the wave's own LDS rows: halves 4 gq .. + 3 and 8 + 4 gq .. + 3 of a k16 row
  // are two 8-byte reads 16 bytes apart, which the padding spreads over all
  // banks.  No barrier: a wave reads what it stored.  The LDS round trip pays
  // near the full 32 rows (M = 32: K = 5120, N = 14336 18.5 -> 16.0 us, N = 7168
  // 14.7 -> 13.4, N = 5120 12.1 -> 11.7, K = 17408, N = 5120 22.2 -> 20.1; even from M
  // = 24 on the wide projections to 28 on the narrow ones; M = 17 4 to 8 % slower).
  char* const wa = reinterpret_cast<char*>(smem) + wave * (kRows * kWaveRowBytes);
  uint32_t aoff[4 * MR];
  if constexpr (kWaveA) {
#pragma unroll
    for (int u = 0; u < 4 * MR; ++u)
      aoff[u] = ((uint32_t)min(4 * u + g, mrows - 1) * (uint32_t)p.k + 8u * (uint32_t)mrow) * 2u;
  }
  auto wave_store = [&](const u32x4(&src)[kSteps][MR]) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 4 * MR; ++u)
      *reinterpret_cast<u32x4*>(wa + (4 * u + g) * kWaveRowBytes + 16 * mrow) = src[u / MR][u % MR];
    asm volatile("" ::: "memory");  // the reads that follow are of other lanes' stores
  };
  auto wave_frag = [&](int rb, int d) __attribute__((always_inline)) {
    const char* src = wa + (16 * rb + mrow) * kWaveRowBytes + 64 * d + 32 * prow + 8 * gq;
    const u32x2 lo = *reinterpret_cast<const u32x2*>(src), hi = *reinterpret_cast<const u32x2*>(src + 16);
    return __builtin_bit_cast(f16x8, (u32x4){lo[0], lo[1], hi[0], hi[1]});
  };

  // Ring of kDepth batches (one scale group, 1 KB per wave, each) in flight.
  u32x4 bw[kDepth][kSteps];
  u32x4 bs[kDepth];
  u32x4 aw[kDepth][kSteps][MR];  // A_DIRECT: [step][row block]; A_WAVE: load u at [u / MR][u % MR]
#pragma unroll
  for (int i = 0; i < kDepth; ++i) bs[i] = (u32x4){0, 0, 0, 0};
  auto issue_step = [&](int slot, int batch, int d) __attribute__((always_inline)) {
    const int kpf = kpw0 + batch * kSteps;
    const char* base = reinterpret_cast<const char*>(p.b) + (size_t)((uint32_t)(kpf + d) * step_bytes);  // uniform
    bw[slot][d] = __builtin_nontemporal_load(reinterpret_cast<const u32x4*>(base + bvoff));
    if constexpr (kDirect) {
#pragma unroll
      for (int rb = 0; rb < MR; ++rb) aw[slot][d][rb] = *reinterpret_cast<const u32x4*>(arow[rb] + 32 * (kpf + d));
    }
  };
  auto issue_wave_a = [&](int slot, int batch) __attribute__((always_inline)) {
    const char* base = reinterpret_cast<const char*>(p.a) + (size_t)((uint32_t)(kpw0 + batch * kSteps) * 64u);  // uniform
#pragma unroll
    for (int u = 0; u < 4 * MR; ++u) aw[slot][u / MR][u % MR] = *reinterpret_cast<const u32x4*>(base + aoff[u]);
  };
  auto issue_scale = [&](int slot, int batch) __attribute__((always_inline)) {
    const int kpf = kpw0 + batch * kSteps;
    if (GROUPED)
      bs[slot] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rbs, svoff, (uint32_t)(kpf >> 2) * group_bytes, kNonTemporal));
  };
  auto issue = [&](int slot, int batch) __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < kSteps; ++d) issue_step(slot, batch, d);
    if constexpr (kWaveA) issue_wave_a(slot, batch);
    issue_scale(slot, batch);
  };

  // ---- staging loads, then the first weight batches, then the stores ----
  // (A_DIRECT: no staging; A_RING: batch 0 of A, then per weight batch i the
  // A batch i + 1)
  if (!kDirect && !kRing && !kWaveA) stage_load(0);
  if constexpr (kRing) ring_load(ar0, 0);
  __builtin_amdgcn_sched_barrier(0);  // staging loads strictly before the weight loads
#pragma unroll
  for (int i = 0; i < kDepth; ++i) {
    issue(i, min(i, nb - 1));
    if constexpr (kRing) ring_load(ar[i], min(i + 1, nb - 1));
    __builtin_amdgcn_sched_barrier(0);  // keep slot order: the loop's waits assume it
  }
  if constexpr (kRing) {
    __builtin_amdgcn_sched_barrier(0);
    ring_store(ar0, 0);
    if (tid == 0) afr[ring_zero] = (u32x4){0, 0, 0, 0};
    lds_barrier();  // LDS only: the weight ring stays in flight
  }
  if constexpr (!kDirect && !kRing && !kWaveA) {
    __builtin_amdgcn_sched_barrier(0);
    stage_store(0);
    for (int base = kThreads * kStageUnroll; base < items; base += kThreads * kStageUnroll) {
      stage_load(base);
      stage_store(base);
    }
    if (tid == 0) afr[n_frag] = (u32x4){0, 0, 0, 0};
    lds_barrier();  // LDS only: the weight ring stays in flight
  }

  // A fragment address: rows >= M read the zero entry.
  const bool a_live = mrow < mrows;
  const int a_step = a_live ? 4 * mrows : 0;
  const int a_base = a_live ? g * mrows + mrow + gw0 * kSteps * a_step : n_frag;
  const int crow0 = (lane >> 4) * 4;  // accumulator rows of this lane (within a row block)
  // A_RING fragment addresses per row block (rows >= M read the zero entry)
  int r_base[MR], r_step[MR], r_slot[MR];
#pragma unroll
  for (int rb = 0; rb < MR; ++rb) {
    const bool live = 16 * rb + mrow < mrows;
    r_base[rb] = live ? g * mrows + 16 * rb + mrow : ring_zero;
    r_step[rb] = live ? 4 * mrows : 0;
    r_slot[rb] = live ? ring_slot : 0;
  }

  f32x4 acc[MR][4];
#pragma unroll
  for (int rb = 0; rb < MR; ++rb)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[rb][j] = (f32x4){0.f, 0.f, 0.f, 0.f};

  // One batch = one scale group.  The weights are the reference's fp16
  // fp16(q - 8) * s (marlin_cuda_kernel.cu:131-159: exact q - 8 from one
  // v_and_or_b32 and one packed add or fma, then one packed multiply by the
  // group's scale), so every product with an fp16 activation is exact in the
  // fp32 MFMA accumulation, as in the reference's MMA.  Per-column scales: the
  // exact q - 8, scaled after the fp16 rounding of the sum.
  auto consume = [&](int slot, int batch) __attribute__((always_inline)) {
    const u32x4 scl = bs[slot];
    f16x2 sc2[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {  // column 16j + 8h + c
      const f16 s = __builtin_bit_cast(f16, (uint16_t)(scl[j] >> (16 * hsel)));
      sc2[j] = (f16x2){s, s};
    }
    if constexpr (kWaveA) wave_store(aw[slot]);
#pragma unroll
    for (int d = 0; d < kSteps; ++d) {
      f16x8 afrag[MR];
      if constexpr (kWaveA) {
#pragma unroll
        for (int rb = 0; rb < MR; ++rb) afrag[rb] = wave_frag(rb, d);
      } else if constexpr (kDirect) {
#pragma unroll
        for (int rb = 0; rb < MR; ++rb) {
          // odd rows of word 0 (gq = 1: halves 8, 9) <-> even rows of word 2
          // (gq = 0: halves 4, 5); the same for words 1 and 3
          const u32x4 l = aw[slot][d][rb];
          const auto w02 = __builtin_amdgcn_permlane16_swap(l[0], l[2], false, false);
          const auto w13 = __builtin_amdgcn_permlane16_swap(l[1], l[3], false, false);
          afrag[rb] = __builtin_bit_cast(f16x8, (u32x4){w02[0], w13[0], w02[1], w13[1]});
        }
      } else if constexpr (kRing) {
#pragma unroll
        for (int rb = 0; rb < MR; ++rb)
          afrag[rb] = __builtin_bit_cast(f16x8, afr[r_base[rb] + (batch & 1) * r_slot[rb] + d * r_step[rb]]);
      } else {
        afrag[0] = __builtin_bit_cast(f16x8, afr[a_base + (batch * kSteps + d) * a_step]);
      }
      const u32x4 own = bw[slot][d];
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const uint32_t partner = (uint32_t)__builtin_amdgcn_mov_dpp((int)own[j], 0x128, 0xf, 0xf, false);  // row_ror:8
        const uint32_t v0 = __builtin_amdgcn_perm(own[j], partner, psel);
        const uint32_t v1 = v0 >> 8;
        f16x2 l0 = nib_lo_to_h2(v0, nk), l1 = nib_lo_to_h2(v1, nk);
        f16x2 h0 = nib_hi_to_h2(v0, nk), h1 = nib_hi_to_h2(v1, nk);
        if (GROUPED) {
          l0 *= sc2[j];
          l1 *= sc2[j];
          h0 *= sc2[j];
          h1 *= sc2[j];
        }
        const f16x8 bfrag = __builtin_bit_cast(f16x8, make_uint4(as_u32(l0), as_u32(l1), as_u32(h0), as_u32(h1)));
#pragma unroll
        for (int rb = 0; rb < MR; ++rb)
          acc[rb][j] = __builtin_amdgcn_mfma_f32_16x16x32_f16(afrag[rb], bfrag, acc[rb][j], 0, 0, 0);
      }
    }
    if constexpr (kWaveA) asm volatile("" ::: "memory");  // the next batch's stores stay behind these reads
  };

  // Full rounds re-issue every slot kDepth batches ahead; the tail (fewer than
  // 2 kDepth batches left) issues only what exists.  Slot i holds batch b + i.
  // The scheduling barriers keep each re-issue right after the consume that
  // frees its slot (the scheduler would otherwise sink all loads to the end of
  // the round and expose a full memory latency per round).
  // A_RING, after consuming batch bb from slot i: A register slot i holds
  // batch bb + 1; store it to LDS slot (bb + 1) & 1 (whose batch bb - 1 every
  // wave finished before the last barrier), reload the register slot with
  // batch bb + 1 + kDepth, and publish.
  auto ring_step = [&](int i, int bb) __attribute__((always_inline)) {
    if constexpr (kRing) {
      ring_store(ar[i], (bb + 1) & 1);
      ring_load(ar[i], min(bb + 1 + kDepth, nb - 1));
      lds_barrier();
    }
  };
  int b = 0;
  for (; b + 2 * kDepth <= nb; b += kDepth) {
#pragma unroll
    for (int i = 0; i < kDepth; ++i) {
      consume(i, b + i);
      __builtin_amdgcn_sched_barrier(0);
      issue(i, b + i + kDepth);
      ring_step(i, b + i);
      __builtin_amdgcn_sched_barrier(0);
    }
  }
#pragma unroll
  for (int i = 0; i < kDepth; ++i) {
    if (b + i < nb) {
      consume(i, b + i);
      if (b + i + kDepth < nb) issue(i, b + i + kDepth);
      if (b + i + 1 < nb) ring_step(i, b + i);
    }
  }
#pragma unroll
  for (int i = 0; i < kDepth - 1; ++i)
    if (b + kDepth + i < nb) {
      consume(i, b + kDepth + i);
      if (b + kDepth + i + 1 < nb) ring_step(i, b + kDepth + i);
    }

  // Wide tiles (each wave its own chunk): the wave hands off on its own.
  if constexpr (EPI == EPI_STORE && CPW == kWaves) return wave_epilogue<GROUPED, MR>(p, acc, chunk, split, 1);

  // ---- epilogue: accumulators -> LDS tile [mrows][256] fp32 ----
  if constexpr (!kDirect) __syncthreads();  // every wave is done with the staged A (or the ring)
  float* tile = reinterpret_cast<float*>(smem);
  {
#pragma unroll
    for (int rb = 0; rb < MR; ++rb)
#pragma unroll
      for (int j = 0; j < 4; ++j)
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 16 * rb + crow0 + i;
          if (r < mrows) tile[r * kCols + wave * 64 + 16 * j + (lane & 15)] = acc[rb][j][i];
        }
  }
  __syncthreads();

  if constexpr (EPI == EPI_STORE) {
    // Every thread takes one column of the tile and every kRG-th row: the sum
    // of the column's k shares (the waves of its chunk), in share order, then
    // the hand-off or the store.  (One wave per column set would issue all
    // M rows' partial stores alone: at M = 32 that wave's 32 stores and their
    // acknowledgements held the arrival up by about a microsecond.)
    constexpr int kTileCols = 64 * cpw;
    constexpr int kRG = kThreads / kTileCols;  // row groups: 4, 2, 1
    constexpr int kPer = (kRows + kRG - 1) / kRG;
    const int c = tid % kTileCols, rg = tid / kTileCols;
    const int n = cg * kTileCols + c;
    float v[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int r = rg + i * kRG;
      float t = 0.f;
      if (r < mrows) {
        t = tile[r * kCols + c];  // share 0
        for (int ws = 1; ws < ksub; ++ws) t += tile[r * kCols + ws * kTileCols + c];
      }
      v[i] = t;
    }
    if (p.splits > 1) {
      float* part = p.partial + (int64_t)split * p.m * p.n + n;
#pragma unroll
      for (int i = 0; i < kPer; ++i)
        if (rg + i * kRG < mrows) publish(part + (int64_t)(rg + i * kRG) * p.n, v[i]);
      wait_published();
      __syncthreads();
      int32_t* ctr = p.counters + 1 + cg;
      if (tid == 0) s_prev = arrive(ctr);
      __syncthreads();
      if (s_prev != p.splits - 1) return false;  // not the last split of this tile
      after_last_arrival();
      if (tid == 0) reset_counter(ctr);
      const int col0 = cg * kTileCols;  // every thread of the workgroup collects
      collect_store<GROUPED, 16 * CPW, kThreads, kRows, 32>(
          p, p.splits, col0, tid, [&](int row, int col, uint16_t v) { p.c[(int64_t)row * p.n + col0 + col] = v; });
      return true;
    }
    // fp16 rounding (per-column scale after it, as the reference does)
    f16 colscale = (f16)1.0f;
    if (!GROUPED) colscale = __builtin_bit_cast(f16, p.s[per_column_scale_index(n)]);
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int r = rg + i * kRG;
      if (r < mrows) {
        f16 h = (f16)v[i];
        if (!GROUPED) h = h * colscale;
        p.c[(int64_t)r * p.n + n] = __builtin_bit_cast(uint16_t, h);
      }
    }
    return true;
  }

  // EPI_ACT, EPI_ARGMAX: thread t < 64 * cpw owns column t of the tile: the
  // sum of its k shares (the waves of chunk t / 64), in share order.
  const bool col_live = tid < 64 * cpw;
  // this thread's output column
  const int n = EPI == EPI_ACT ? (col_live ? tile_chunk<EPI, CPW>(p, cg, tid >> 6) * 64 + (tid & 63) : 0)
                               : cg * 64 * cpw + (col_live ? tid : 0);
  float v[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    float t = 0.f;
    if (r < mrows && col_live) {
      t = tile[r * kCols + tid];  // share 0 (wave tid / 64)
      for (int ws = 1; ws < ksub; ++ws) t += tile[r * kCols + ws * cpw * 64 + tid];
    }
    v[r] = t;
  }

  // EPI_ACT: thread t forms neuron pair t of a row from the tile's fp16
  // outputs [mrows][64 CPW] (gate half, then up half) in LDS, with the same
  // SiLU-gated product as the A_SILU_PACKED staging, and publishes it.
  auto act_pairs = [&](const uint16_t* xch) __attribute__((always_inline)) {
    constexpr int kPairs = 16 * CPW;  // neuron pairs per row
    const uint32_t* xw = reinterpret_cast<const uint32_t*>(xch);
    for (int it = tid; it < mrows * kPairs; it += kThreads) {
      const int r = it / kPairs, t2 = it - r * kPairs;
      const uint32_t gw = xw[r * (32 * CPW) + t2];
      const uint32_t uw = xw[r * (32 * CPW) + kPairs + t2];
      publish(p.act_out + (int64_t)r * (p.n / 4) + (int64_t)cg * kPairs + t2, silu_mul2(gw, uw));
    }
  };

  if (p.splits > 1) {
    float* part = p.partial + (int64_t)split * p.m * p.n + n;
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      if (r < mrows && col_live) publish(part + (int64_t)r * p.n, v[r]);
    wait_published();
    __syncthreads();
    int32_t* ctr = p.counters + 1 + cg;
    if (tid == 0) s_prev = arrive(ctr);
    __syncthreads();
    if (s_prev != p.splits - 1) return false;  // not the last split of this tile
    after_last_arrival();
    if (tid == 0) reset_counter(ctr);
    if constexpr (EPI == EPI_ACT) {
      // every thread collects, the gate half and then the up half of the tile
      // (each a contiguous run of 32 CPW columns), into the LDS exchange
      constexpr int h = CPW / 2;
      uint16_t* xch = reinterpret_cast<uint16_t*>(smem);
#pragma unroll
      for (int half = 0; half < 2; ++half)
        collect_store<GROUPED, 16 * h, kThreads, kRows, 32>(
            p, p.splits, tile_chunk<EPI, CPW>(p, cg, half * h) * 64, tid,
            [&](int row, int col, uint16_t v) { xch[row * 64 * CPW + half * 64 * h + col] = v; });
      __syncthreads();
      act_pairs(xch);
      return true;
    }
    // Sum the partials in split order; 4 rows x 8 splits of reads in flight.
    const float* src = p.partial + n;
    const int64_t split_stride = (int64_t)p.m * p.n;
#pragma unroll
    for (int r0 = 0; r0 < kRows; r0 += 4) {
      if (r0 < mrows && col_live) {
        float sum[4] = {0.f, 0.f, 0.f, 0.f};
        for (int s0 = 0; s0 < p.splits; s0 += 8) {
          float t[4][8];
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u)
              t[i][u] = collect(src + (int64_t)min(s0 + u, p.splits - 1) * split_stride +
                                (int64_t)min(r0 + i, mrows - 1) * p.n);
#pragma unroll
          for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int u = 0; u < 8; ++u) sum[i] += (s0 + u < p.splits) ? t[i][u] : 0.f;
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) v[r0 + i] = sum[i];
      }
    }
  }

  // fp16 rounding (per-column scale after it, as the reference does)
  f16 colscale = (f16)1.0f;
  if (!GROUPED && col_live) colscale = __builtin_bit_cast(f16, p.s[per_column_scale_index(n)]);
  uint16_t outh[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    f16 h = (f16)v[r];
    if (!GROUPED) h = h * colscale;
    outh[r] = __builtin_bit_cast(uint16_t, h);
  }

  if (EPI == EPI_ACT) {
    // the tile's fp16 outputs go through LDS to act_pairs
    constexpr int kTileCols = 64 * CPW;
    uint16_t* xch = reinterpret_cast<uint16_t*>(smem);
    __syncthreads();  // every thread is done with the fp32 tile
#pragma unroll
    for (int r = 0; r < kRows; ++r)
      if (r < mrows && col_live) xch[r * kTileCols + tid] = outh[r];
    __syncthreads();
    act_pairs(xch);
    return true;
  }

  // ---- argmax: per-row max over this tile's 256 columns, then over tiles ----
#pragma unroll
  for (int r = 0; r < kMaxM; ++r) {
    if (r < mrows) {
      const uint64_t best = wave_max_u64(col_live ? argmax_key(h2f(outh[r]), (uint32_t)n) : 0ull);
      if (lane == 0) s_keys[wave][r] = best;
    }
  }
  __syncthreads();
  if (tid < mrows) {
    uint64_t best = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) best = max_u64(best, s_keys[w][tid]);
    publish(p.tile_keys + (int64_t)tid * p.n_cg + cg, best);
  }
  wait_published();
  __syncthreads();
  int32_t* final_counter = p.counters;
  if (tid == 0) s_prev = arrive(final_counter);
  __syncthreads();
  if (s_prev != p.n_cg - 1) return false;
  after_last_arrival();
  if (tid == 0) reset_counter(final_counter);
  for (int r = wave; r < mrows; r += kWaves) {
    uint64_t best = 0;
    for (int t = lane; t < p.n_cg; t += kWave) best = max_u64(best, collect(p.tile_keys + (int64_t)r * p.n_cg + t));
    best = wave_max_u64(best);
    if (lane == 0) {
      p.argmax_state[r] = (int64_t)best;
      p.argmax_out[r] = (int64_t)(0xffffffffu - (uint32_t)(best & 0xffffffffu));
    }
  }
  return true;
}

// The arguments come first that the prologue and the split hand-off need, as
// separate scalars: gfx950 preloads the leading kernel arguments into SGPRs
// at wave launch (14 dwords here: the build asks for 16, the kernarg pointer
// takes two), so neither the first weight loads nor the partial stores wait
// for a kernarg fetch.  a, b, s, the four sizes and the two hand-off pointers
// fill all 14; the output and argmax pointers follow.  The column-tile count
// is n / (64 CPW).  A struct argument is not preloaded.
template <int AM, int EPI, bool GROUPED, int CPW, int MR = 1>
__global__ __launch_bounds__(kThreads) void marlin_skinny_kernel(const uint16_t* a, const uint32_t* b,
                                                                 const uint16_t* s, int m, int n, int k, int splits,
                                                                 float* partial, int32_t* counters, uint16_t* c,
                                                                 uint64_t* tile_keys, int64_t* argmax_state,
                                                                 int64_t* argmax_out) {
  // `splits` carries the mixed plan's whole-tile count in its high 16 bits, so
  // that the mapping below reads only preloaded arguments
  const int whole = (int)((uint32_t)splits >> 16);
  splits &= 0xffff;
  Params p{};
  p.a = a; p.b = b; p.s = s; p.c = c; p.counters = counters; p.partial = partial;
  p.m = m; p.n = n; p.k = k; p.splits = splits; p.kp_total = k >> 5; p.n_cg = n / (64 * CPW);
  p.tile_keys = tile_keys; p.argmax_state = argmax_state; p.argmax_out = argmax_out;
  int cg = blockIdx.x, split = blockIdx.y;
  if (whole > 0) {
    // Mixed grid (one dimension): tiles 0 .. whole - 1 over the whole K (their
    // waves' k shares summed in LDS, no split-K hand-off), the remaining tiles
    // split `splits` ways.
    const int bid = blockIdx.x;
    if (bid < whole) {
      cg = bid;
      split = 0;
      p.splits = 1;
    } else {
      const int u = bid - whole;
      cg = whole + u / splits;
      split = u - (u / splits) * splits;
    }
  }
  skinny_tile<AM, EPI, GROUPED, CPW, MR>(p, cg, split);
}

// SiLU-gated activations for the launches that do not stage A: act[m][k] =
// fp16(silu(g) * u) of mixed [M, 2K] = [g | u], with the staging's own
// function (silu_mul2), so they see the values the staged A_SILU_PACKED variant
// would.  One thread per 8 halves of a row; rows blockIdx.y, + gridDim.y, ...
// Bound by its 6 bytes per activation (M = 2048, K = 17408: 214 MB).
__global__ __launch_bounds__(256) void silu_pack_kernel(const uint16_t* __restrict__ mixed, uint16_t* __restrict__ act,
                                                        int m, int k) {
  const int k8 = 8 * (int)(blockIdx.x * 256 + threadIdx.x);
  if (k8 >= k) return;
  for (int64_t row = blockIdx.y; row < m; row += gridDim.y) {
    const uint4 g = *reinterpret_cast<const uint4*>(mixed + row * 2 * k + k8);
    const uint4 u = *reinterpret_cast<const uint4*>(mixed + row * 2 * k + k + k8);
    *reinterpret_cast<uint4*>(act + row * k + k8) =
        make_uint4(silu_mul2(g.x, u.x), silu_mul2(g.y, u.y), silu_mul2(g.z, u.z), silu_mul2(g.w, u.w));
  }
}

}  // namespace skinny
}  // namespace lb
