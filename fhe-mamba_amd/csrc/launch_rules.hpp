// Launch shapes chosen by size.  Plain host code, so that its rules can be
// checked without a GPU.
//
// A column is M = 2^s1 rows, s1 = ceil(log_n / 2); a tile is one column of one
// poly, 2^s2 of them a poly, s2 = floor(log_n / 2).
#pragma once

#include <algorithm>
#include <cstdint>

namespace fhe {

constexpr uint32_t COMPUTE_UNITS = 256, SIMDS = 4;

// LDS words between the column lines of kernels that keep whole columns in
// LDS, the lanes of a wavefront on one line, and the lines of a wavefront.
constexpr uint32_t column_pitch(uint32_t s1) { return (1u << s1) + (1u << s1) / 16 + 1; }
constexpr uint32_t column_lanes(uint32_t s1) { return s1 >= 8 ? 64 : (1u << s1) / 4; }
constexpr uint32_t column_lines(uint32_t s1) { return 64 / column_lanes(s1); }

// ---- The conversion's middle kernel (k_convert_mid) ----
// Waves a SIMD its registers are limited to, the largest workgroup, and the
// LDS of a workgroup of nw waves: target constants (16 bytes each, in groups
// of four), source lines, lines in flight.
constexpr uint32_t mid_waves_per_simd(uint32_t s1) { return s1 == 9 ? 4 : s1 == 8 ? 7 : 6; }
constexpr uint32_t mid_max_waves(uint32_t s1) { return s1 == 9 ? 16 : 8; }
constexpr uint32_t mid_lds_bytes(uint32_t s1, uint32_t nsrc, uint32_t ndst, uint32_t nw) {
  return (ndst + 3) / 4 * 4 * 16 + (nsrc + nw * column_lines(s1)) * column_pitch(s1) * 8;
}
constexpr uint32_t mid_resident_groups(uint32_t s1, uint32_t nsrc, uint32_t ndst, uint32_t nw,
                                       uint32_t lds) {
  return std::min(lds / mid_lds_bytes(s1, nsrc, ndst, nw), SIMDS * mid_waves_per_simd(s1) / nw);
}

// Waves of a workgroup (4, 8, or 16 at s1 = 9) for a launch of `tiles` tiles
// with up to nsrc sources and ndst targets, on CUs of `lds` bytes of LDS.
//  - No more than the lines fill: a wave without a line idles at every
//    barrier and holds its slot.  32 rotations of one limb and one digit, us,
//    4 / 8 / 16 waves: N=2^14 71 / 104, N=2^16 141 / 196, N=2^17 286 / 400 / 642.
//  - A launch of at most one round of 8-wave workgroups is bound by one tile's
//    chain: 8 (one rotation at N=2^16, 8-limb digits, 24 limbs: 113 / 108).
//  - Else the form with the most waves resident on a CU.  s1 = 9, middle of
//    four ModUps, 15 limbs of 5 sources 132 / 141 / 170, 16 limbs of 8 sources
//    108 / 106 / 128, 30 limbs of 15 sources 346 / 260 / 236; s1 = 8, 16
//    limbs of 4 sources 77 / 81, 30 limbs of 15 sources 110 / 96.  Where two
//    forms are equal, the smaller (s1 = 7, 32 ModDowns of 24 limbs, 8 sources:
//    126 / 138), except at s1 = 8 and 7 or 8 sources: 30 rotations of 24 limbs
//    off one ModUp took 1573 / 1533.
inline uint32_t mid_waves(uint32_t s1, uint32_t tiles, uint32_t nsrc, uint32_t ndst,
                          uint32_t lds) {
  if (std::max(nsrc, ndst) <= 4 * column_lines(s1)) return 4;
  auto groups = [&](uint32_t nw) { return mid_resident_groups(s1, nsrc, ndst, nw, lds); };
  uint32_t best = tiles <= COMPUTE_UNITS * groups(8) ? 8 : 4;
  for (uint32_t nw = 2 * best; nw <= mid_max_waves(s1); nw *= 2) {
    const uint32_t have = best * groups(best), with = nw * groups(nw);
    if (with > have || (with == have && s1 == 8)) best = nw;
  }
  return best;
}

// ---- Digits that one key switch uses ----
// Whether their last block stages run inside ModDown's passes (modup_raw), for
// `count` key switches of nd digits of `limbs` limbs in one launch set.  That
// saves a pass over the digits, and makes them in turn, two at a time, in
// ModDown's workgroups: with three digits or more that chain costs more than
// the pass while the digits are small.  One rotation, us, in a pass of their
// own / inside: 4 digits of 5 limbs at N=2^13 35.0 / 38.5 (1.2 MiB), at N=2^14
// 38.1 / 42.1 (2.5), at N=2^15 44.5 / 46.8 (5); 4 digits of 20 limbs at N=2^13
// 45.5 / 44.5 (5), 3 of 32 47.9 / 46.0 (6), at N=2^15 3 of 20 61.7 / 57.0 (15).
// With two digits this is at most 2.5% behind and up to 15% ahead, with one 3
// to 12% ahead, at any size.
constexpr bool finish_digits_in_moddown(uint32_t nd, uint32_t limbs, uint32_t n, uint32_t count) {
  return nd <= 2 || (uint64_t)count * nd * limbs * n * 8 > (5u << 20);
}

// ---- Rescale, N = 2^13 .. 2^17 ----
// `tiles` columns of the last limb lifted into l other limbs.  Whether one
// kernel per column does it (k_rescale_mid, three launches) and not two column
// passes (four).  The column kernel is ahead except in batches of rings with 128
// rows a column, where its waves, of two lines each, wait for the one that has
// the last limb; the line lies where the intermediate (tiles l KiB) outgrows the
// L2s (32 MiB).  s1 = 7, us, as three launches of 4-wave workgroups / as four:
// 1536 tiles of 19 limbs 44.1 / 46.5 (29 MiB), 4096 of 8 48.7 / 47.0 (32), 2048
// of 19 53.1 / 52.9 (38), of 39 101 / 90, 4096 of 23 122 / 116.  s1 = 8: 8192 of
// 29 limbs 521 / 606; s1 = 9: 8192 of 44 limbs 1685 / 2278.
constexpr bool rescale_by_columns(uint32_t s1, uint32_t tiles, uint32_t l) {
  return s1 > 7 || tiles <= 1024 || (uint64_t)tiles * l <= 32768;
}
// Waves of the column kernel's workgroup.  us at 4 / 8 / 16 waves:
//  - no more than the lines fill: 4 limbs, 32 polys, N=2^16 86 / 91 / 109, and
//    one limb, 2 / 4 / 8 waves: N=2^14 22.0 / 23.6 / 27.0, N=2^17 78 / 84 / 118;
//  - 16 where a launch leaves half the chip's wave slots free at 8, one
//    ciphertext at N=2^16: 12 limbs 25.4 / 24.6 / 24.5, 29 limbs 43.2 / 42.6 /
//    41.5; N=2^15: 44 limbs 40.1 / 35.8 / 34.6; N=2^13 44 limbs 26.9 / 23.4 /
//    22.5.  Not with 512 rows a column, whose lines hold 8 rows a lane: N=2^17
//    16 limbs 52.1 / 51.2 / 54.1, 44 limbs 121.8 / 119.4 / 120.7; nor above 512
//    tiles: 3 polys at N=2^16, 29 limbs 54.6 / 53.7 / 53.8, 8 polys at N=2^14,
//    44 limbs 57.5 / 57.8 / 63.3;
//  - 4 in batches with 128 rows a column (two lines a wave): 20 polys at
//    N=2^13, 19 limbs 38.1 / 41.9 / 43.5; 8 else (32 polys, 44 limbs, N=2^16 795
//    / 792 / 814).
constexpr uint32_t rescale_waves(uint32_t s1, uint32_t tiles, uint32_t l) {
  const uint32_t rounds = (l + column_lines(s1) - 1) / column_lines(s1);  // of one wave
  if (rounds <= 2) return 2;
  if (rounds <= 4 || (s1 == 7 && tiles > 1024)) return 4;
  return rounds > 8 && tiles <= 512 && s1 < 9 ? 16 : 8;
}
// LDS: the last limb's line and one for each in flight, in the 64 KB that any
// device gives a workgroup for every form above.
constexpr uint32_t rescale_lds_bytes(uint32_t s1, uint32_t nw) {
  return (1 + nw * column_lines(s1)) * column_pitch(s1) * 8;
}
static_assert(rescale_lds_bytes(7, 16) <= 65536 && rescale_lds_bytes(8, 16) <= 65536 &&
                  rescale_lds_bytes(9, 8) <= 65536,
              "rescale workgroups");

}  // namespace fhe
