// Rules that choose between two kernels by sizes alone, and how work is shared out: plain C++, so that they can be tested
// without a GPU.
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

// fwgemm: one thread per element, or tiles of 128 x 128.  The first takes time by columns of 64 outputs, and more than its share
// once A's columns leave the L2 (long k); the second by the tiles on the fullest compute unit (one, here) and, without a
// k-contiguous image of A at hand, by lookups that gather 16 cache lines per improved element, whatever k.  us on square problems, one thread per element / tiles.  Without the image: float 1000^3 165 / 310, 1152^3
// 241 / 472, 1408^3 428 / 555, 1536^3 544 / 453; double 800^3 247 / 328, 900^3 360 / 377, 1000^3 449 / 333.  With it
// (three squarings): float 1000 526 / 638, 1100 699 / 716, 1152 758 / 701; double 700 516 / 632, 768 634 / 650, 800 776 / 669.
// Long and short k without it: float 1100 x 1100 x 4000 1215 / 966; double 200 x 3000 x 2500 1816 / 1076, 1100 x 1100 x 64 48 / 106.  One row: 1 x 100000 x 300
// float 294 / 258, double 1396 / 257.
inline bool fwgemm_one_thread_each(bool f64, bool k_contiguous_image, int m, int n, int k) {
  const double tiles_worth = double((int64_t(m) + 63) / 64 * 64) * n / (128 * 128);
  if (k_contiguous_image) return tiles_worth < (f64 ? 37 : 79);
  if (f64) return tiles_worth < (k < 2048 ? 53 : 40) || (tiles_worth < 150 && tiles_worth * k < 20000);
  return tiles_worth < (k < 2048 ? 128 : 64);
}

// ... and the double-precision tile: 64 x 128 by 256 threads while every one of them has a compute unit to itself, and
// without the image (its lookups take the time) at any size; 128 x 128 by 512 threads otherwise.  Three squarings of n = 1024 / 1280 / 1408 /
// 1536 / 1792: 797 / 963 / 1052 / 1718 / 1988 us on 64 x 128, 1174 / 1430 / 1558 / 1675 / 1940 on 128 x 128; one product
// without the image 331 / 414 / 557 / 694 / 945 and 523 / 779 / 865 / 825 / 1153.
// (Fewer than 64 rows, 30 x 30000 x 200: 160 and 143.)
inline bool fwgemm_f64_half_tile(bool k_contiguous_image, int m, int64_t half_tiles) {
  return m >= 64 && (!k_contiguous_image || half_tiles <= 256);
}

// The binary16 tile (half_tile.h), by its rows: 128 x 256, 64 x 128, 32 x 128 and, for adds that do not care about order,
// 16 x 128.  ordered: plus.  bits: or-and on masks and the bitwise pairs.  zeros: min- and max-times on binary16.
// A compute unit holds at most two of these workgroups (two waves per SIMD) and works two off faster than one, but not
// twice as fast (a packed instruction occupies the vector ALU for four cycles: one wave per SIMD keeps it busy most of the
// time); smaller tiles do less work per LDS read and per barrier.  `alone` / `paired`: the chip's rate in TOPS with one / two
// workgroups of that tile on every compute unit (min-plus, measured from 512^3 to 4096^3).  The time is about that of the
// rounds of 512 workgroups at the paired rate plus a last round at whichever rate its size gives; the tile with the
// smallest wins.
// 64 x 128 of the order-free adds is the exception: it reaches 60 alone and 74 paired, but a last round of 257 to 340
// workgroups takes it as long as one of 512, so at those rates it would be taken too often (1216 x 2048 x 2048, 304 workgroups,
// 247 us where 32 x 128 takes 227; 1500 x 1500 x 4000 508 and 468).  50 and 72 choose the faster one, or one within 2 %, at 13 sizes of
// 190 to 800 workgroups, binary16 min-plus and max-min, k = 512 and 2048 (1792^2, 392: 232 and 266; 2048 x 2176, 544: 338 and 327;
// 2304^2, 648: 341 and 389; 2560^2, 800: 440 and 448); on int8 32 x 128 is kept at 1500 x 1500 x 2048, 321 us where this takes 307.
// 72 instead of 68, what whole k-tiles per thread reach, moves a quarter of this tile's sizes to it: of 1131 drawn ones
// (64 .. 4096 each way, binary16 and int8) none was slower by more than 0.4 %, on average they were 1.17 (binary16) and 1.23
// times as fast.  Products of binary16 keep 68: their lookups of zeros, not the loop, set the time.
inline int half_tile_rows(bool ordered, bool bits, bool zeros, int m, int n, long long products) {
  auto cost = [&](int bm, int bn, long long alone, long long paired) {
    const long long groups = (m + bm - 1LL) / bm * ((n + bn - 1LL) / bn) * products;
    const long long rest = groups % 512, area = (long long)bm * bn;
    return groups / 512 * (512 * area / paired) + (rest > 256 ? 512 * area / paired : rest > 0 ? 256 * area / alone : 0);
  };
  // (or-and: the full tile's term is half an instruction; the smaller tiles are bound by what surrounds the terms)
  const long long full = bits ? cost(128, 256, 95, 128) : cost(128, 256, 63, 83);
  const long long mid = cost(64, 128, 50, bits ? 76 : ordered || zeros ? 68 : 72);
  if (ordered) {
    const long long small = cost(32, 128, 36, 55);
    return full <= mid && full <= small ? 128 : mid <= small ? 64 : 32;
  }
  // the small tiles share every k-tile out between the four waves (1024^3 min-plus: 47 - 49 TOPS against 33 - 37 with whole
  // k-tiles per thread; 512^3: 13 - 14 against 8)
  const long long sliced = cost(32, 128, 43, 62), narrow = cost(16, 128, 35, 48);
  if (full <= mid && full <= sliced && full <= narrow) return 128;
  return mid <= sliced && mid <= narrow ? 64 : sliced <= narrow ? 32 : 16;
}

// Where part `part` of `parts` begins in a k-tile that holds `rest` k-values only; part + 1's beginning is its end.
constexpr int ragged_share(int rest, int parts, int part) {
  const int begin = part * ((rest + parts - 1) / parts);
  return begin < rest ? begin : rest;
}

}  // namespace cuasr_amd
