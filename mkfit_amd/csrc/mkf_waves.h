// mkf_waves.h -- how many seeds (or candidates) a one-wavefront workgroup carries.  Host code without HIP.
#pragma once

#include <algorithm>
#include <cstddef>

namespace mkf_find {

// Best-hit finding and the per-layer steps, one lane per track: halved from 64 until there is a wavefront per SIMD of
// the device's `cus` compute units.  Below, SIMDs idle; above, wavefronts of half-used lanes take turns (256 CUs,
// best-hit step at 512 / 1024 / 2048 / 4096 wavefronts: one 10k-seed event 357 / 342 / 432 / 432 us, 4 events - / 858 /
// 933 / 1020 us, 12 events - / 1950 / 2077 / 2311 us; at 500 seeds 1, 2, 4, 8, 16 seeds per wavefront: 286, 292, 298,
// 313, 345 us).  The steps by 8, 16, 32 and 64 lanes, where this takes 8, 16 and 64: k_select of 10k tracks 8.5 / 9.4 /
// 12.3 / 17.7 us, 30k 14.6 / 11.9 / 14.7 / 21.4, 100k 37.9 / 31.8 / 31.9 / 31.6; k_find_candidates 11.0 / 11.2 / 12.9 /
// 19.2, 20.9 / 16.4 / 18.0 / 26.4, 66.7 / 51.5 / 52.2 / 51.6; k_add_best_hit 10.6 / 10.7 / 10.7 / 10.7, 15.9 / 11.1 /
// 11.0 / 11.8, 42.9 / 32.0 / 28.7 / 24.7.
inline int lanes_per_wave(size_t n, int cus) {
  const size_t simds = 4 * (size_t)cus;
  int lanes = 64;
  while (lanes > 1 && n < lanes * simds) lanes /= 2;
  return lanes;
}

// Combinatorial finding, up to `most` seeds: as few as put every wavefront on the device at once, `per_cu` on a CU.  A
// lone wavefront leaves its SIMD waiting for its own results half of the time and its phases grow with its seeds'
// windows and pairs, but one more than fit wait for a whole launch (clone engine, one 10k-seed event, 10 / 9 / 6 / 5 / 4
// / 2 seeds per wavefront: 704 / 692 / 627 / 612 / 889 / 1093 us; standard finding of 5003 seeds, 10 / 4 / 3 / 2: 660 /
// 594 / 886 / 842 us; 500 seeds, 10 / 1: 607 / 432 us).
inline int seeds_per_wave(size_t n, int most, int cus, int per_cu) {
  const size_t resident = (size_t)cus * per_cu;
  return (int)std::min<size_t>(most, std::max<size_t>(1, (n + resident - 1) / resident));
}

}  // namespace mkf_find
