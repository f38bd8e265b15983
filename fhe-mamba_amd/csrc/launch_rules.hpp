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

}  // namespace fhe
