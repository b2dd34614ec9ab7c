// spk_pair.hip -- the two-sweep bit-plane kernel of two-state sq/4n lattices
// (spk_bits.h) and its launch.
#include <hip/hip_runtime.h>

#include "spk_pair.h"

using namespace spk;

// Two sweeps of a lattice that pair_fits, one band of BAND rows per
// workgroup (spk_bits.h): planes and seeds from (bits_in, seed_in) to
// (bits_out, seed_out); sweep 1's counts to the row at acc, sweep 2's to
// the next row.  The grid is the bands rounded up to a multiple of 8.
// Every thread issues the loads of its band's planes first, then the loads
// of its seed slots in the order it uses them, two slots ahead of their use:
// each is waited for just before that use while the later ones are in
// flight.  The seed loads are unconditional (a slot outside every pass, or
// an idle lane, loads a row that exists and is not used) so that the count
// of loads in flight is the same on every path and those waits stay exact.  FULL: rows of kPairMaxPw
// whole words (sub-grid rows of 2048 sites: nx = 4096) and an even number
// of them, so every lane works and the row arithmetic is simpler
// (pair_side, pair_thread).
template <bool SINGLE, bool FULL, int BAND, int STAGE>
__global__ __launch_bounds__(kPairThreads) void k_sweep_bits_pair(const uint32_t *__restrict__ bits_in,
                                                                 const int32_t *__restrict__ seed_in,
                                                                 uint32_t *__restrict__ bits_out,
                                                                 int32_t *__restrict__ seed_out, Geom g, BitGeom bg,
                                                                 Rule r, unsigned long long *__restrict__ acc) {
  using Shape = PairShape<BAND, STAGE>;
  static_assert(!FULL || STAGE == 4 * kPairMaxPw, "full rows fill the widest stage");
  __shared__ PairLdsOf<BAND> L;
  const int y0 = xcd_tile(blockIdx.x, gridDim.x) * BAND;
  if (y0 >= g.hy) return;   // a padding workgroup: all its threads leave together
  // the group is the same on all lanes of a wavefront (STAGE is a
  // multiple of 64); saying so keeps it and the rows in scalar registers
  const int grp = __builtin_amdgcn_readfirstlane((int)(threadIdx.x / STAGE));
  const uint32_t tau = threadIdx.x % STAGE;
  const bool lane_on = FULL || tau < 4u * (uint32_t)bg.pw;
  const uint32_t ta = lane_on ? tau : 0u;
  // the planes: at most 3 words per thread (2 * 24 rows * 64 <= 3 * 1024)
  constexpr int kPlaneLoads = (2 * Shape::rows * (STAGE / 4) + kPairThreads - 1) / kPairThreads;
  const int nplane = 2 * Shape::rows * bg.pw;
  uint32_t pv[kPlaneLoads];
#pragma unroll
  for (int k = 0; k < kPlaneLoads; k++) {
    int c, lr, w;
    pv[k] = bits_in[pair_plane_src<Shape>(g, bg, y0, min((int)threadIdx.x + k * kPairThreads, nplane - 1), c, lr, w)];
  }
  // (a thread past the last word writes that word again, with its value:
  // no condition, so the compiler keeps the loads where they were issued)
#pragma unroll
  for (int k = 0; k < kPlaneLoads; k++) {
    int c, lr, w;
    (void)pair_plane_src<Shape>(g, bg, y0, min((int)threadIdx.x + k * kPairThreads, nplane - 1), c, lr, w);
    L.planes[c][lr][w] = pv[k];
  }
  // The seeds of the thread's rows, colour 0 (passes 0, 2) and colour 1
  // (passes 1, 3), go out a few at a time, two slots ahead of their use:
  // colour 0's first two slots now, the others during pass 0 (below).
  // Issuing all of them at the start had every workgroup's plane loads wait
  // behind every other's seed loads (7 us of a 48 us launch).
  Words<4> s0[Shape::slots0][2], s1[Shape::slots1][2];
  auto load = [&](int c, int j, Words<4>(&dst)[2]) {
    const int rho = min(pair_slot_row<Shape>(y0, c, grp, j), y0 + BAND + 2 - c);   // within pass c's rows
    const int prow = pair_row(rho, g.hy);
#pragma unroll
    for (int h = 0; h < 2; h++)
      dst[h] = *pair_seeds<FULL>(seed_in, bg, c, prow, ta, h);
  };
  constexpr int kAhead = Shape::slots0 >= 4 ? 2 : 1;
  static_assert(Shape::slots1 >= kAhead, "colour 1 has its first slots");
#pragma unroll
  for (int j = 0; j < kAhead; j++) load(0, j, s0[j]);
  __syncthreads();
  PairCounts a1, a2;   // sweep 1 (passes 0, 1) and sweep 2
  // the thread's LDS offsets are the same on every row; opaque, so the
  // compiler keeps them rather than recomputing them a row at a time
  PairLane lane = pair_lane<FULL>(g, bg, pair_slot_row<Shape>(y0, 0, grp, 0), 0, grp, lane_on ? tau : 0u);
  asm volatile("" : "+v"(lane.w4), "+v"(lane.wn4), "+v"(lane.b));
  // a pass over the thread's slots; before(j) runs before slot j
  auto pass = [&](int p, auto &seeds, int slots, auto &&before) {
#pragma unroll
    for (int j = 0; j < slots; j++) {
      before(j);
      const int rho = pair_slot_row<Shape>(y0, p & 1, grp, j);
      if (lane_on && pair_pass_row<Shape>(y0, p, rho)) {
        const PairWords pwd = pair_words(L, y0, p, rho, grp, lane);
        pair_thread<SINGLE, FULL>(L, g, bg, r, y0, p, rho, grp, tau, lane, pwd, seeds[j], seed_out, p < 2 ? a1 : a2);
      }
    }
    __syncthreads();
  };
  // colour 1's first kAhead slots go out during pass 0's last slots and the
  // rest during pass 1, two slots ahead of use, so that each pass reads
  // about one colour's seeds rather than pass 0 reading both
  auto loads_ahead0 = [&](int j) {
    if (j + kAhead < Shape::slots0) load(0, j + kAhead, s0[j + kAhead]);
    if (j >= Shape::slots0 - kAhead) load(1, j - (Shape::slots0 - kAhead), s1[j - (Shape::slots0 - kAhead)]);
  };
  auto loads_ahead1 = [&](int j) {
    if (j + kAhead < Shape::slots1) load(1, j + kAhead, s1[j + kAhead]);
  };
  auto nothing = [](int) {};
  pass(0, s0, Shape::slots0, loads_ahead0);
  // colour 0's last slot that pass 2 uses waits in LDS through pass 1, when
  // both colours' seeds are held (its registers go to pass 1's work), and
  // comes back one slot before pass 2 needs it; the single-flip events need
  // fewer registers and keep it, and so do the smaller bands
  constexpr bool kPark = !SINGLE && Shape::slots0 >= 6;
  constexpr int kParked = kPark ? Shape::slots0 - 2 : 0;
  if constexpr (kPark) {
#pragma unroll
    for (int h = 0; h < 2; h++) L.parked[h][threadIdx.x] = s0[kParked][h];
  }
  pass(1, s1, Shape::slots1, loads_ahead1);
  auto unpark = [&](int j) {
    if (kPark && j == kParked - 1) {
#pragma unroll
      for (int h = 0; h < 2; h++) s0[kParked][h] = L.parked[h][threadIdx.x];
    }
  };
  pass(2, s0, Shape::slots2, unpark);
  pass(3, s1, Shape::slots1, nothing);
  for (int i = threadIdx.x; i < 2 * BAND * bg.pw; i += kPairThreads) pair_store_plane(L, bits_out, g, bg, y0, i);
  const Counts c1 = pair_counts(a1), c2 = pair_counts(a2);
  block_accumulate2(c1.nacc, c1.de, c2.nacc, c2.de, acc, acc + kAccRow, blockIdx.x & (kAccSlots - 1));
}

namespace spk {

void launch_pair_kernel(hipStream_t stream, const uint32_t *bits_in, const int32_t *seed_in, uint32_t *bits_out,
                        int32_t *seed_out, const Geom &g, const BitGeom &bg, const Rule &r, bool single,
                        unsigned long long *acc) {
  const int band = pair_band(g), stage = pair_stage(bg.pw);
  const int bands = (g.hy + band - 1) / band;
  const unsigned grid = (unsigned)((bands + kNumXcd - 1) / kNumXcd * kNumXcd);   // xcd_tile: a multiple of 8
  // 64 words, the last one whole, and an even number of rows
  const bool full = bg.pw == kPairMaxPw && bg.r == 31 && g.hy % 2 == 0;
  auto go = [&]<int BAND, int STAGE>() {
    auto with = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(kPairThreads), 0, stream, bits_in, seed_in, bits_out, seed_out, g, bg, r,
                         acc);
    };
    if constexpr (STAGE == 4 * kPairMaxPw) {
      if (full) return single ? with(k_sweep_bits_pair<true, true, BAND, STAGE>) : with(k_sweep_bits_pair<false, true, BAND, STAGE>);
    }
    single ? with(k_sweep_bits_pair<true, false, BAND, STAGE>) : with(k_sweep_bits_pair<false, false, BAND, STAGE>);
  };
  auto with_stage = [&]<int BAND>() {
    if (stage == 64) go.template operator()<BAND, 64>();
    else if (stage == 128) go.template operator()<BAND, 128>();
    else go.template operator()<BAND, 256>();
  };
  if (band == 4) with_stage.template operator()<4>();
  else if (band == 8) with_stage.template operator()<8>();
  else if (band == 12) with_stage.template operator()<12>();
  else with_stage.template operator()<kPairBand>();
}

}  // namespace spk
