// Rules that choose between two kernels by sizes alone: plain C++, so that they can be tested without a GPU.
#pragma once

#include <cstdint>

namespace cuasr_amd {

// The staged family's full-size tile with its k shared by two groups of threads, against the quarter-size tile (area_ratio
// of which make a full one).  192 .. 256 full-size workgroups are one per compute unit for most of the chip, whatever their
// number; the quarter-size tiles' time goes by the most that one compute unit gets.  So the full-size tile wins where
// that is as many as make a full one: fp32 min-plus 1984^3, 256 full or 961 quarter-size tiles (four per unit), 223 against 250
// us; 1824^3, 225 or 841, 202 against 223; but 1700^3, 196 or 729 (three per unit), 193 against 169.
inline bool two_group_full_tile(long long full, long long quarter, int area_ratio) {
  return full >= 192 && full <= 256 && quarter > 256LL * (area_ratio - 1);
}

// fwgemm: one thread per element, or tiles of 128 x 128.  The first takes time by outputs, the second by the tiles on the
// fullest compute unit (one, here) and, without a k-contiguous image of A at hand, by lookups that gather 16 cache lines per
// improved element.  us on square problems, one thread per element / tiles.  Without the image: float 1000^3 165 / 310, 1152^3
// 241 / 472, 1408^3 428 / 555, 1536^3 544 / 453; double 800^3 247 / 328, 900^3 360 / 377, 1000^3 449 / 333.  With it
// (three squarings): float 1000 526 / 638, 1100 699 / 716, 1152 758 / 701; double 700 516 / 632, 768 634 / 650, 800 776 / 669.
inline bool fwgemm_one_thread_each(bool f64, bool k_contiguous_image, int m, int n) {
  const int64_t tiles_worth = f64 ? (k_contiguous_image ? 37 : 50) : (k_contiguous_image ? 76 : 128);
  return int64_t(m) * n < tiles_worth * 128 * 128;
}

// ... and the double-precision tile: 64 x 128 by 256 threads while every one of them has a compute unit to itself, and
// without the image (its lookups take the time) at any size; 128 x 128 by 512 threads otherwise.  Three squarings of n = 1024 / 1280 / 1408 /
// 1536 / 1792: 797 / 963 / 1052 / 1718 / 1988 us on 64 x 128, 1174 / 1430 / 1558 / 1675 / 1940 on 128 x 128; one product
// without the image 331 / 414 / 557 / 694 / 945 and 523 / 779 / 865 / 825 / 1153.
inline bool fwgemm_f64_half_tile(bool k_contiguous_image, int64_t half_tiles) { return !k_contiguous_image || half_tiles <= 256; }

}  // namespace cuasr_amd
