// Launches the rowwise matrix-core product at one bit width, LB_RW_BITS (a
// compile definition: the build compiles this file once per width).

#include <algorithm>

#include "rowwise_mm.hpp"

namespace lb {
namespace rwmm {
namespace {

template <int SPS, int MB, int NB, int W, int DEPTH>
int launch_skinny(const Params& p, int mats, hipStream_t st) {
  const dim3 grid((unsigned)((p.rows + 16 * NB - 1) / (16 * NB)), (unsigned)((p.batch + 16 * MB - 1) / (16 * MB)),
                  (unsigned)mats);
  hipLaunchKernelGGL((skinny_kernel<LB_RW_BITS, SPS, MB, NB, W, DEPTH>), grid, dim3(W * kWave), 0, st, p);
  return lbh::launch_status();
}

template <int SPS, int MB, int NB, int DEPTH>
int launch_tile(const Params& p, hipStream_t st) {
  const dim3 grid((unsigned)((p.rows + 64 * NB - 1) / (64 * NB)), (unsigned)((p.batch + 16 * MB - 1) / (16 * MB)));
  hipLaunchKernelGGL((tile_kernel<LB_RW_BITS, SPS, MB, NB, DEPTH, 2>), grid, dim3(kTileThreads), 0, st, p);
  return lbh::launch_status();
}

// Which form, from sweeps at 2, 3, 4 and 8 bits over M = 2..384, K x N = 5120 x
// 17408 and 17408 x 5120 (times below: 4 bits, g128):
//   up to 16 rows: 32 output rows per workgroup (M = 16, N = 5120: 24 us, 16
//     rows 34 us, 64 rows 38 us), 16 where that leaves half the CUs idle.  One
//     stage in flight per wave: with two the registers (130 at first, 128 now) leave
//     little or no room for a second workgroup on a CU (M = 16, N = 17408: 24.7 us
//     against 22.8, 8 bits 32.3 against 29.8).  Two in flight where there is one workgroup per
//     CU at most anyway, few rows and few bits (K = 17408, N = 5120, M = 6: 19.8
//     against 20.2 us; 2 bits 16.8 against 18.7 at M = 4, even at 16).
//     More than two workgroups of 32 rows per CU: 48 rows from M = 9 on, up to
//     4 bits (M = 16: N = 17408 22.5 -> 21.0 us, N = 34816 36.0 -> 31.4; M = 3
//     16.3 against 17.2; 5 bits 26.0 against 26.5).
//     One (ragged) row, 16 output rows a workgroup on half the CUs at most: a
//     wave's chain of stages is the launch, so sixteen waves take it from K = 8192
//     on (2..8 bits, K = 17400: N = 2048 11.2..13.8 -> 8.7..11.7 us, N = 48 8.6..12.4
//     -> 7.6..10.8; K = 8184 0.99 to 1.14 times as fast, K = 4088 0.85 to 0.98; with 4
//     activation rows 0.95 at K = 12280, with 16 0.93 at K = 17400);
//   17 to 32: two blocks of 16, eight waves and 32 rows (M = 32, N = 5120: 31
//     us; 16 rows 46, four waves 45).  It is one workgroup per CU by its LDS, so
//     with more than one for each four waves run (N = 14336 21.5 -> 20.5 us, K =
//     2048, N = 16384 at 2 bits 12.2 -> 9.7), and with more than two 48 rows (N =
//     17408 30.0 -> 25.7, N = 34816 48.4 -> 44.6; at N = 14336 25.1 against 20.5);
//   above, where 64-column tiles of 64 rows do not give every CU one (N = 5120
//     up to M = 192): four blocks of 16, the waves splitting K (M = 128: 72 us
//     against 88 us); eight waves where that is one round of workgroups (M =
//     64: 53 us against 62 us), four otherwise (M = 128: 72 against 89);
//   else the largest tile that gives 1.5 workgroups per CU (N = 17408: M = 384
//     102 us on 64 x 256, M = 256 79 us on 64 x 128 against 99, M = 128 51 us on
//     32 x 128 against 56).
// At 5, 6 and 7 bits (checked afterwards, g128, M = 4..384, the two shapes and N =
// 34816) the same rules give the fastest form or one within 5 % of it, except: K =
// 17408, N = 5120, M = 128, where eight waves (5 bits, 85 us against 122) or 64 x 64
// tiles (6 and 7 bits, 107 and 111 against 120 and 126) are ahead, and N = 34816, where
// 48 rows up to M = 16 (5 bits 38.6 against 42.9), 64 x 64 tiles at M = 64 (72 against
// 81) and 64 x 128 at M = 384 (220 against 246) are.
template <int SPS>
int launch_sps(const Params& p, int mats, hipStream_t st) {
  const int64_t cus = lbh::device_cus();
  auto wgs = [&](int mb, int rows) {
    return (int64_t)((p.batch + 16 * mb - 1) / (16 * mb)) * ((p.rows + rows - 1) / rows) * mats;
  };
  if (p.batch <= 16) {
    if constexpr (LB_RW_BITS <= 4) {
      if (wgs(1, 32) > 2 * cus && p.batch > 8) return launch_skinny<SPS, 1, 3, 8, 1>(p, mats, st);
      if constexpr (LB_RW_BITS == 2 || SPS == 1)
        if (2 * wgs(1, 32) >= cus && wgs(1, 32) <= cus && (LB_RW_BITS == 2 || p.batch <= 8))
          return launch_skinny<SPS, 1, 2, 8, 2>(p, mats, st);
    }
    if (2 * wgs(1, 32) >= cus) return launch_skinny<SPS, 1, 2, 8, 1>(p, mats, st);
    if (p.batch == 1 && 2 * wgs(1, 16) <= cus && p.cols >= 8192) return launch_skinny<SPS, 1, 1, 16, 2>(p, mats, st);
    return launch_skinny<SPS, 1, 1, 8, 2>(p, mats, st);
  }
  const bool narrow = wgs(4, 64) < cus;
  if (p.batch <= 32 || narrow) {
    if (p.batch > 32 && 2 * wgs(4, 32) >= cus) {
      if (LB_RW_BITS <= 5 && wgs(4, 32) <= cus) return launch_skinny<SPS, 4, 2, LB_RW_BITS <= 5 ? 8 : 4, 1>(p, mats, st);
      return launch_skinny<SPS, 4, 2, 4, 1>(p, mats, st);
    }
    if (wgs(2, 32) > 2 * cus) return launch_skinny<SPS, 2, 3, 4, 1>(p, mats, st);
    if (wgs(2, 32) > cus) return launch_skinny<SPS, 2, 2, 4, 1>(p, mats, st);
    if (2 * wgs(2, 32) >= cus) return launch_skinny<SPS, 2, 2, 8, 1>(p, mats, st);
    if (2 * wgs(2, 16) >= cus) return launch_skinny<SPS, 2, 1, 8, 1>(p, mats, st);
    return launch_skinny<SPS, 1, 1, 8, 2>(p, mats, st);
  }
  if (2 * wgs(4, 256) >= 3 * cus) return launch_tile<SPS, 4, 4, 1>(p, st);
  if (2 * wgs(4, 128) >= 3 * cus) return launch_tile<SPS, 4, 2, 1>(p, st);
  if (p.batch <= 128) return launch_tile<SPS, 2, 2, 2>(p, st);
  return launch_tile<SPS, 4, 1, 2>(p, st);
}

}  // namespace

template <>
int launch<LB_RW_BITS>(const Params& p, int sps, int mats, hipStream_t st) {
  return sps == 1 ? launch_sps<1>(p, mats, st) : sps == 2 ? launch_sps<2>(p, mats, st) : launch_sps<4>(p, mats, st);
}

}  // namespace rwmm
}  // namespace lb
