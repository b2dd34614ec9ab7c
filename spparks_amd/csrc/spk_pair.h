// spk_pair.h -- launch of the two-sweep bit-plane kernel (spk_pair.hip).
#pragma once

#include "spk_bits.h"

namespace spk {

constexpr int kPairCus = 256;   // compute units a launch has to fill

// Rows per workgroup: the fewest that leave every band a compute unit of its
// own (a workgroup fills one), since a band of B rows costs 4B + 12 row
// passes: a lattice of 2006 rows in bands of 16 used 126 units, and a launch
// took as long as one of 4096 rows.  us a sweep, in bands of 16 (or one colour
// a launch, marked c) and now: 3000 x 2006 ising/single 15.1, 10.3; 3000^2
// Ising 21.2, 15.8; 2000^2 12.4 c, 7.8; 1500^2 11.2 c, 7.0 (boxes: 7.7); 1000^2
// 10.8 c, 4.2 (boxes: 4.8); 1000 x 4000 12.4 c, 7.4.
inline int pair_band(const Geom &g) {
  for (int band : {4, 8, 12})
    if ((g.hy + band - 1) / band <= kPairCus) return band;
  return kPairBand;
}

// Threads per row group for rows of pw words: the fewest that hold a row.
inline int pair_stage(int pw) { return pw <= 16 ? 64 : pw <= 32 ? 128 : 256; }

// Two sweeps from (bits_in, seed_in) to (bits_out, seed_out).
void launch_pair_kernel(hipStream_t stream, const uint32_t *bits_in, const int32_t *seed_in, uint32_t *bits_out,
                        int32_t *seed_out, const Geom &g, const BitGeom &bg, const Rule &r, bool single,
                        unsigned long long *acc);

}  // namespace spk
