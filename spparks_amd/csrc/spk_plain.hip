// spk_plain.hip -- libspk_hip.so, single-lattice path: the per-colour strict
// sweep kernels, the fused energy / Naccept reductions, device-side initial
// state (set site range, tagreset seeds via Park-Miller jump-ahead), layout
// conversion, and the C ABI declared in include/spk_hip.h.
#include <hip/hip_runtime.h>

#include <cmath>
#include <cstdio>
#include <cstring>
#include <mutex>
#include <new>
#include <string>
#include <algorithm>
#include <utility>
#include <vector>

#include "spk_bits.h"
#include "spk_device.h"
#include "spk_host.h"
#include "spk_kernels.h"
#include "spk_pair.h"
#include "spk_neigh.h"
#include "spk_slice.h"
#include "spk_tile.h"

using namespace spk;

// ==================================================================== kernels

// One colour pass of a two-state sq/4n lattice on bit planes: thread t owns
// SPT sites of one plane word (see spk_bits.h).
template <int SPT, bool SINGLE>
__global__ __launch_bounds__(1024) void k_sweep_bits(uint32_t *__restrict__ bits, int32_t *__restrict__ sseed, Geom g,
                                                    BitGeom bg, Rule r, int color,
                                                    unsigned long long *__restrict__ acc) {
  const uint32_t t = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * blockDim.x + threadIdx.x;
  Counts cnt{0, 0};
  if ((int64_t)t < bg.threads) cnt = bits_thread<SPT, SINGLE>(bits, sseed, g, bg, r, color, t);
  block_accumulate_pack(cnt.nacc, cnt.de, acc, blockIdx.x & (kAccSlots - 1));
}

// u8 state -> planes, one thread per plane word of both colours
__global__ void k_bits_pack(const uint8_t *__restrict__ spin, Geom g, BitGeom bg, uint32_t *__restrict__ bits) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t words = (int64_t)g.hy * bg.pw;
  if (q >= 2 * words) return;
  const int c = q >= words;
  const int64_t t = q - (c ? words : 0);
  const int b = (int)(t / bg.pw), w = (int)(t % bg.pw);
  bits[q] = bits_pack_word(spin, g, c, b, w);
}

__global__ void k_bits_unpack(const uint32_t *__restrict__ bits, Geom g, BitGeom bg, uint8_t *__restrict__ spin) {
  const int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t words = (int64_t)g.hy * bg.pw;
  if (q >= 2 * words) return;
  const int c = q >= words;
  const int64_t t = q - (c ? words : 0);
  const int b = (int)(t / bg.pw), w = (int)(t % bg.pw);
  bits_unpack_word(spin, g, c, b, w, bits[q]);
}

// seeds <-> shadow seeds, one thread per 16-byte group (bits_seed_group_in
// / _out): each wavefront reads or writes 1 KiB of consecutive canonical
// bytes and 128-byte runs of the shadow
__global__ void k_seeds_to_shadow(const int32_t *__restrict__ seed, Geom g, BitGeom bg, int32_t *__restrict__ sseed) {
  const int64_t X = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (X < bg.seedc / 2) bits_seed_group_in(seed, g, bg, X, sseed);
}

__global__ void k_seeds_from_shadow(const int32_t *__restrict__ sseed, Geom g, BitGeom bg, int32_t *__restrict__ seed) {
  const int64_t X = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (X < bg.seedc / 2) bits_seed_group_out(sseed, g, bg, X, seed);
}

// One colour pass: every site of colour `color` performs one strict event.
// A pack is 4 consecutive sites of one sub-grid row (x fastest), so its own
// spins/seeds are one aligned load and a wavefront's accesses are
// unit-stride.  Each workgroup covers one TileMap tile (rows of its own
// waves supply most of the y/z neighbour rows); tiles are remapped so that
// neighbouring tiles share an XCD.
template <int LAT, typename T, int V, bool TWO, typename I, int XDIR>
__global__ __launch_bounds__(1024) void k_sweep_color(T *__restrict__ spin, int32_t *__restrict__ seed,
                                                      Geom g, Rule r, TileMap m, int color,
                                                      unsigned long long *__restrict__ acc) {
  static_assert(V == 4, "tiles map 4 sites per thread");
  __shared__ int s_thr[32];
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  int a0, b, e;
  const bool live = tile < m.nxc * m.nyg * m.nzg && tile_site(g, m, (uint32_t)tile, threadIdx.x, a0, b, e);
  // the thresholds are staged in LDS between counting and deciding, so the
  // pack's loads are not held behind a barrier
  const int thr_v = threadIdx.x < 28 ? r.thr[threadIdx.x] : 0;
  PackWork<T, TWO, I> w;
  if (live) w = pack_count<LAT, T, TWO, I, XDIR>(spin, seed, g, r, color, a0, b, e);
  if (threadIdx.x < 28) s_thr[threadIdx.x] = thr_v;
  __syncthreads();
  Counts cnt{0, 0};
  if (live) cnt = pack_decide<LAT, T, TWO, I>(w, spin, seed, g, r, s_thr, color);
  __syncthreads();   // block_accumulate reuses LDS after the decide step's reads
  block_accumulate_pack(cnt.nacc, cnt.de, acc, blockIdx.x & (kAccSlots - 1));
}

// Every sweep of a lattice small enough to live in one workgroup's LDS
// (the reference's CPU-sized cases): spins and seeds are read once, all
// colour passes run on the LDS copy with a barrier between passes, and the
// state is written back once.  The same per-pack events as k_sweep_color,
// on LDS addresses; sweep s's (Naccept, dE) go to rows[2s], rows[2s+1] (host
// memory).
template <int LAT, typename T, bool TWO>
__global__ __launch_bounds__(1024) void k_sweep_resident(T *__restrict__ spin, int32_t *__restrict__ seed, Geom g,
                                                         Rule r, int nsweeps, unsigned long long *__restrict__ rows) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_thr[32];
  const uint32_t slots = (uint32_t)g.K * (uint32_t)g.Mp;
  const uint32_t spin_words = slots * (uint32_t)sizeof(T) / 4;   // Mp is a multiple of 4
  T *ls = reinterpret_cast<T *>(lds);
  int32_t *lk = reinterpret_cast<int32_t *>(lds + (spin_words * 4 + 15) / 16 * 16);
  for (uint32_t i = threadIdx.x; i < spin_words; i += blockDim.x)
    reinterpret_cast<uint32_t *>(ls)[i] = reinterpret_cast<const uint32_t *>(spin)[i];
  for (uint32_t i = threadIdx.x; i < slots; i += blockDim.x) lk[i] = seed[i];
  if (threadIdx.x < 28) s_thr[threadIdx.x] = r.thr[threadIdx.x];
  __syncthreads();
  const uint32_t npack = (uint32_t)g.Mp / 4;
  for (int sw = 0; sw < nsweeps; sw++) {
    int na = 0, de = 0;
    for (int c = 0; c < g.K; c++) {
      for (uint32_t p = threadIdx.x; p < npack; p += blockDim.x) {
        int a0, b, e;
        pack_site(g, p, a0, b, e);
        const Counts cnt = sweep_sites<LAT, T, 4, TWO, uint32_t>(ls, lk, g, r, s_thr, c, a0, b, e);
        na += cnt.nacc;
        de += cnt.de;
      }
      __syncthreads();   // the next colour reads this colour's new spins
    }
    block_store(na, de, rows + 2 * (size_t)sw);
    __syncthreads();
  }
  for (uint32_t i = threadIdx.x; i < spin_words; i += blockDim.x)
    reinterpret_cast<uint32_t *>(spin)[i] = reinterpret_cast<const uint32_t *>(ls)[i];
  for (uint32_t i = threadIdx.x; i < slots; i += blockDim.x) seed[i] = lk[i];
}

// The two colours of row pair m on bit planes of the spins (spk_slice.h): a
// wavefront works on s.rw whole rows, four lanes on a word of each colour.
// What bounds it at 256^3 (Q = 10^4, 14 planes, 4096 wavefronts, all resident
// at once): VALU 55% busy (1400 instructions a wavefront, 88 a site against 131
// of the packed kernel), 70 MB a launch at 4.2 TB/s, the seeds of all
// wavefronts asked for at once at the start and written at the end.  us a
// sweep, the packed per-colour kernel and this one:
//   Q = 3000: 64^3 34.0, 25.1; 128^3 35.5, 25.4; 160^3 45.2, 36.4; 224^3 79.1, 55.0;
//   256^3 96.6, 59.0; 320^3 162, 121; Q = 5 at 256^3 80.4, 41.4; Q = 10^6 137, 78.4
constexpr int kSliceThreads = 256;

template <bool FULL, int PG>
__global__ __launch_bounds__(kSliceThreads) void k_sweep_slice(uint32_t *__restrict__ planes,
                                                               int32_t *__restrict__ sseed, Geom g, SliceGeom s, Rule r,
                                                               int m, unsigned long long *__restrict__ acc) {
  __shared__ SliceLds L[kSliceThreads / 64];
  const uint32_t wid = (uint32_t)__builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
  const uint32_t v = (uint32_t)xcd_tile(blockIdx.x, gridDim.x) * (kSliceThreads / 64) + wid;
  SliceCounts n;
  if (v < (uint32_t)s.waves) slice_wave<FULL, PG>(planes, sseed, g, s, r, L[wid], m, v, threadIdx.x & 63, n);
  const Counts cnt = slice_counts(n);
  block_accumulate(cnt.nacc, cnt.de, acc, blockIdx.x & (kAccSlots - 1));
}

// Several colour passes in one launch (spk_tile.h): workgroup t loads box t
// with its halo into LDS, runs the plan's passes on it with a barrier after
// each, and writes the box it owns to the other state buffer.  The counts of
// each sweep the passes touch go to consecutive rows at acc.
// What bounds it: small boxes, one thread's chain per pass (LDS reads, draw,
// compare, decide, barrier: 0.8-1 us for 32 passes of 128^2 sq/8n, VALU busy
// 38%); large ones, the VALU (54% busy on 1500 x 1002 sq/8n, with 14% of the
// events in the halo).  us a sweep, before and now:
//   sq/4n Ising 256^2 10.2, 2.3 (1000^2 10.8, 4.8, but 4.1 in k_sweep_bits_pair)
//   sq/8n Potts 128^2 Q=100 9.2, 3.8 (one workgroup before)
//   sq/8n Potts 1500 x 1002 Q=100 15.1, 8.8
//   sc/26n Potts 32^3 Q=1000 33.6, 12.1; 64^3 Q=10^5 37.6, 15.1
// One site a thread (VEC 1) against packs of 4: 16.2 against 24.1 on 64^3
// sc/26n, 4.4 against 5.6 on 128^2 sq/8n, but 11.2 against 9.5 on 1500 x 1002,
// where the VALU counts.
template <int LAT, typename T, bool TWO, int VEC, int APP>
__global__ __launch_bounds__(1024) void k_sweep_tile(const T *__restrict__ spin_in, const int32_t *__restrict__ seed_in,
                                                     T *__restrict__ spin_out, int32_t *__restrict__ seed_out, Geom g,
                                                     Rule r, TilePlan tp, unsigned long long *__restrict__ acc) {
  extern __shared__ __align__(16) unsigned char lds[];
  __shared__ int s_thr[32];
  __shared__ int s_cnt[kTileMaxSweeps][2];
  __shared__ TilePass s_pass[kTileMaxPass];
  int nt = (int)blockDim.x;
  asm("" : "+s"(nt));   // held, not read again from the dispatch in every pass
  T *ls = reinterpret_cast<T *>(lds);
  int32_t *lk = reinterpret_cast<int32_t *>(lds + tp.spin_bytes);
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  if (tile >= tp.cx * tp.cy * tp.cz) return;   // a padding workgroup: all its threads leave together
  const TileBox bx = tile_box(tp, tile);
  const uint32_t packs = (uint32_t)tp.gl.K * (uint32_t)(tp.gl.Mp / 4);
  for (uint32_t i = threadIdx.x; i < packs; i += nt) tile_load<LAT, T>(spin_in, seed_in, g, tp, bx, i, ls, lk);
  if (threadIdx.x < 28) s_thr[threadIdx.x] = r.thr[threadIdx.x];
  if (threadIdx.x < 2 * kTileMaxSweeps) (&s_cnt[0][0])[threadIdx.x] = 0;
  // the pass table to LDS: read from the kernel's arguments, each pass began
  // with two scalar loads that missed, one after the other
  constexpr int kPassWords = kTileMaxPass * (int)sizeof(TilePass) / 4;
  for (int i = threadIdx.x; i < kPassWords; i += nt)
    reinterpret_cast<uint32_t *>(s_pass)[i] = reinterpret_cast<const uint32_t *>(tp.pass)[i];
  __syncthreads();
  int c = tp.c0, row = 0, na = 0, de = 0;
  for (int k = 0; k < tp.npass; k++) {
    TilePass ps;
#pragma unroll
    for (int i = 0; i < (int)sizeof(TilePass) / 4; i++)
      reinterpret_cast<int *>(&ps)[i] = __builtin_amdgcn_readfirstlane(reinterpret_cast<const int *>(&s_pass[k])[i]);
    auto pass = [&]<int XD>() {
      for (uint32_t i = threadIdx.x; i < ps.items; i += nt) {
        Counts cnt;
        if constexpr (VEC == 1) cnt = tile_event<LAT, T, TWO, APP>(ls, lk, g, r, s_thr, tp, bx, ps, c, i);
        else cnt = tile_events<LAT, T, TWO, XD>(ls, lk, g, r, s_thr, tp, bx, ps, c, i);
        na += cnt.nacc;
        de += cnt.de;
      }
    };
    // packs: the x-shift side is the colour's x parity on a Moore lattice
    if constexpr (VEC > 1 && (LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N)) {
      if (c & 1) pass.template operator()<1>();
      else pass.template operator()<0>();
    } else {
      pass.template operator()<-1>();
    }
    if (++c == tp.gl.K) c = 0;
    if (c == 0 || k == tp.npass - 1) {   // the end of a sweep, or of the launch
      na = wave_sum(na);
      de = wave_sum(de);
      if ((threadIdx.x & 63) == 0) {
        atomicAdd(&s_cnt[row][0], na);
        atomicAdd(&s_cnt[row][1], de);
      }
      na = de = 0;
      row++;
    }
    __syncthreads();   // the next pass reads this one's spins
  }
  const uint32_t own = tile_store_items<LAT>(tp);
  for (uint32_t i = threadIdx.x; i < own; i += nt) tile_store<LAT, T>(spin_out, seed_out, g, tp, bx, i, ls, lk);
  if (threadIdx.x < 2u * (unsigned)row) {
    const int v = (&s_cnt[0][0])[threadIdx.x];
    unsigned long long *a = acc + (size_t)(threadIdx.x >> 1) * kAccRow +
                            (size_t)(blockIdx.x & (kAccSlots - 1)) * kSlotStride + (threadIdx.x & 1);
    if (v) atomicAdd(a, (unsigned long long)(long long)v);
  }
}

// One colour pass of a proposal variant (potts/neigh, potts/neighonly,
// ising/single): one slot per thread (4 consecutive slots per pack, so a
// wavefront's own-site accesses stay unit-stride), neighbours read in the
// reference's order.  The lattices that k_sweep_neigh does not take.
template <int LAT, typename T, int APP>
__global__ __launch_bounds__(1024) void k_sweep_variant(T *__restrict__ spin, int32_t *__restrict__ seed, Geom g,
                                                        Rule r, int color, unsigned long long *__restrict__ acc) {
  __shared__ int s_thr[32];
  if (threadIdx.x < 28) s_thr[threadIdx.x] = r.thr[threadIdx.x];
  __syncthreads();
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t t = (int64_t)tile * blockDim.x + threadIdx.x;
  Counts cnt{0, 0};
  if (t < (int64_t)g.Mp) cnt = variant_site<LAT, T, APP>(spin, seed, g, r, s_thr, color, (uint32_t)t);
  block_accumulate_pack(cnt.nacc, cnt.de, acc, blockIdx.x & (kAccSlots - 1));
}

// The same for potts/neigh and potts/neighonly in halfwords (spk_neigh.h),
// four sites a thread.  VALU bound: 1970 instructions a wavefront of 256 sites
// at sc/26n against 854 for 64, 8 wavefronts a SIMD at 256^3.  us a sweep there,
// Q = 10^4 and 100: k_sweep_variant 390, 390, this kernel 247, 245; sq/8n at
// 2048^2 37.6, 28.0.
template <int LAT, typename T, int APP, typename I, int XD>
__global__ __launch_bounds__(1024) void k_sweep_neigh(T *__restrict__ spin, int32_t *__restrict__ seed, Geom g, Rule r,
                                                      TileMap m, int color, unsigned long long *__restrict__ acc) {
  __shared__ int s_thr[32];
  if (threadIdx.x < 28) s_thr[threadIdx.x] = r.thr[threadIdx.x];
  __syncthreads();
  const int tile = xcd_tile(blockIdx.x, gridDim.x);
  int a0, b, e;
  Counts cnt{0, 0};
  if (tile < m.nxc * m.nyg * m.nzg && tile_site(g, m, (uint32_t)tile, threadIdx.x, a0, b, e))
    cnt = neigh_pack<LAT, T, APP, I, XD>(spin, seed, g, r, s_thr, color, a0, b, e);
  block_accumulate_pack(cnt.nacc, cnt.de, acc, blockIdx.x & (kAccSlots - 1));
}

// ===================================================================== host

constexpr int kBitSites = 32;   // default sites per thread on bit planes

// Boxes of the tile kernel: extents of the owned box (lattice sites), sweeps
// per launch, sites per thread, threads per workgroup.
struct TileShape {
  int w[3];
  int sweeps;
  int vec;
  int block;
};

// How a sweeps call runs (route()).
enum Route { kRouteColour, kRouteBits, kRouteTile, kRouteSlice };

struct spk_hip_lattice {
  spk_hip_desc d;
  Geom g;
  Rule rule;
  int64_t N = 0;
  int device = 0;
  int stype = kI32;                    // storage type of spins on the device
  int64_t slots = 0;                   // K*Mp stored values (sites + row pads)
  hipStream_t stream = nullptr;
  void *spin = nullptr;                // slots spins, colour-blocked, stype
  int32_t *seed = nullptr;             // slots seeds, colour-blocked
  // bit planes of a two-state sq/4n lattice (spk_bits.h).  Once a sweeps
  // call has packed them they hold the state (bits_active) until a call
  // that needs the byte layout unpacks them (bits_leave).
  // bitplanes: 0 planes off; 1 the default (two sweeps per launch where
  // that pays, else kBitSites sites per thread); 8, 16, 32 sites per thread
  // of the per-colour kernel
  int bitplanes = 1;
  bool bits_active = false;
  bool pairs = false;                  // planes in the spt-8 layout, sweeps two per launch
  bool pairs_ok = true;                // false once the second planes did not fit the device's memory
  // the same for bit-sliced lattices (spk_slice.h), which use bits and sseed
  // for their planes and seeds
  bool slice_active = false;
  bool slice_ok = true;                // false once the planes did not fit the device's memory
  SliceGeom sg{};
  BitGeom bg{};
  uint32_t *bits = nullptr;
  int32_t *sseed = nullptr;
  int64_t sseed_cap = 0;               // shadow seed slots allocated
  uint32_t *bits2 = nullptr;           // the second planes and seeds of two-sweep launches
  int32_t *sseed2 = nullptr;
  int64_t sseed2_cap = 0;
  // lattices that fit one workgroup's LDS run every sweep in one launch
  int resident = 1;
  bool resident_set = false;           // set_resident asked for it
  // lattices whose colour passes are short run several per launch
  // (spk_tile.h), from spin/seed to spin2/seed2 and back
  TileShape tile{};                    // boxes of the tile kernel (sweeps 0: not used)
  bool tile_known = false;             // tile is up to date with the settings
  bool block_set = false;              // set_launch asked for the per-colour kernel
  void *spin2 = nullptr;
  int32_t *seed2 = nullptr;
  size_t max_lds = 0;                  // LDS bytes a workgroup may use
  int32_t *stage = nullptr;            // N int32, natural order (transfers)
  unsigned long long *acc = nullptr;   // [cap][kAccRow]: per-sweep slots
  int acc_cap = 0;
  int block = 256;
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  double last_ms = 0.0;
  int64_t last_nlaunch = 0;
  bool energy_valid = false;
  int64_t energy = 0;                  // total energy, exact integer
  // graph replay: a call of n sweeps replays n / chunk graphs of `chunk`
  // sweeps, then one graph of the remainder
  int chunk = 32;                      // sweeps per full graph (0: eager launches only)
  struct Piece {
    int sweeps;                        // sweeps the graph runs
    int route;                         // Route it was captured on
    hipGraphExec_t exec;
  };
  std::vector<Piece> graphs;
  // per-sweep rows of a call, (Naccept, dE), in pinned host memory: the fold
  // (or the one-workgroup kernel) writes them there itself, so a call takes no
  // copy back
  unsigned long long *pinned = nullptr;
  int pinned_rows = 0;
  int32_t *pinned_state = nullptr;     // spins and seeds of a small lattice, natural order (download)
};

namespace {

constexpr int kInitialAccRows = 1024;
constexpr int64_t kHostStateSites = 1 << 16;   // lattices whose downloads go through pinned_state
constexpr int kMaxChunk = 1024;   // sweeps per captured graph
constexpr int kVec = 4;   // sites per thread in the sweep kernel

// Lets a kernel take `lds` bytes of dynamic LDS (64 KiB need no leave).
template <typename K>
void allow_lds(K kern, size_t lds) {
  if (lds > (64u << 10))
    (void)hipFuncSetAttribute(reinterpret_cast<const void *>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
}

unsigned grid_for(int64_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

// Lattices that k_sweep_neigh takes: row segments of one x side, and values of
// at most 15 bits.  On sq/8n, whose 28 pairs are soon compared, a quarter of the
// wavefronts pays from more than 2^18 sites a colour on; us a sweep, one
// site a thread and this way: 512^2 13.4, 15.1; 1024^2 16.4, 15.4 (18.1 in workgroups of
// 512); 1280^2 22.6, 18.9; 1600^2 25.9, 22.4; 2048^2 35.2, 26.3.  On sc/26n at
// every size: 32^3 59.7, 54.9; 64^3 56.1, 55.0; 96^3 59.5, 57.3; 128^3 73.3, 56.6.
bool neigh_packed(const spk_hip_lattice *h) {
  return (h->d.app == SPK_HIP_POTTS_NEIGH || h->d.app == SPK_HIP_POTTS_NEIGHONLY) &&
         (h->g.lat == SPK_HIP_SC_26N || (h->g.lat == SPK_HIP_SQ_8N && h->g.Mp > (1 << 18))) && h->stype != kI32 &&
         h->rule.nspins <= kNeighMaxQ;
}

// (workgroups of 256 unless the caller chose: 22.4 us a sweep of sq/8n at 1600^2
// against 25.0 with the other kernels' 512)
int launch_neigh(spk_hip_lattice *h, int color, unsigned long long *acc) {
  const int bs = h->block_set ? h->block : 256;
  const TileMap m = make_tile_map(h->g, bs);
  unsigned grid = (unsigned)m.nxc * m.nyg * m.nzg;
  grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
  const bool off32 = offsets_fit_32(h->g);
  with_lattice(h->g.lat, [&]<int LAT>() {
    with_type(h->stype, [&]<typename T>() {
      if constexpr ((LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N) && sizeof(T) <= 2) {
        auto go = [&](auto kern) {
          hipLaunchKernelGGL(kern, dim3(grid), dim3(bs), 0, h->stream, static_cast<T *>(h->spin), h->seed, h->g,
                             h->rule, m, color, acc);
        };
        auto with_x = [&]<int APP, typename I>() {
          color & 1 ? go(k_sweep_neigh<LAT, T, APP, I, 1>) : go(k_sweep_neigh<LAT, T, APP, I, 0>);
        };
        auto with_app = [&]<int APP>() {
          off32 ? with_x.template operator()<APP, uint32_t>() : with_x.template operator()<APP, int64_t>();
        };
        if (h->d.app == SPK_HIP_POTTS_NEIGH) with_app.template operator()<SPK_HIP_POTTS_NEIGH>();
        else with_app.template operator()<SPK_HIP_POTTS_NEIGHONLY>();
      }
    });
  });
  return check_hip(hipGetLastError(), "sweep kernel launch");
}

int launch_variant(spk_hip_lattice *h, int color, unsigned long long *acc) {
  if (neigh_packed(h)) return launch_neigh(h, color, acc);
  const int bs = h->block;
  unsigned grid = grid_for(h->g.Mp, bs);
  grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
  const int app = h->d.app;
  with_lattice(h->g.lat, [&]<int LAT>() {
    with_type(h->stype, [&]<typename T>() {
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(bs), 0, h->stream, static_cast<T *>(h->spin), h->seed, h->g,
                           h->rule, color, acc);
      };
      if (app == SPK_HIP_POTTS_NEIGH) go(k_sweep_variant<LAT, T, SPK_HIP_POTTS_NEIGH>);
      else if (app == SPK_HIP_POTTS_NEIGHONLY) go(k_sweep_variant<LAT, T, SPK_HIP_POTTS_NEIGHONLY>);
      else if constexpr (sizeof(T) == 1) go(k_sweep_variant<LAT, T, SPK_HIP_ISING_SINGLE>);   // two states: u8
    });
  });
  return check_hip(hipGetLastError(), "sweep kernel launch");
}

int launch_sweep(spk_hip_lattice *h, int color, unsigned long long *acc) {
  if (h->bits_active) {
    const int bs = h->block;
    unsigned grid = grid_for(h->bg.threads, bs);
    grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
    auto go = [&](auto kern) {
      hipLaunchKernelGGL(kern, dim3(grid), dim3(bs), 0, h->stream, h->bits, h->sseed, h->g, h->bg, h->rule, color,
                         acc);
    };
    const bool single = h->d.app == SPK_HIP_ISING_SINGLE;
    if (h->bg.spt == 8) single ? go(k_sweep_bits<8, true>) : go(k_sweep_bits<8, false>);
    else if (h->bg.spt == 16) single ? go(k_sweep_bits<16, true>) : go(k_sweep_bits<16, false>);
    else single ? go(k_sweep_bits<32, true>) : go(k_sweep_bits<32, false>);
    return check_hip(hipGetLastError(), "bit-plane sweep launch");
  }
  if (variant_app(h->d.app)) return launch_variant(h, color, acc);
  const int bs = h->block;
  const TileMap m = make_tile_map(h->g, bs);
  unsigned grid = (unsigned)m.nxc * m.nyg * m.nzg;
  grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
  const bool two = h->rule.nspins == 2;   // two states are always stored as u8
  const bool off32 = offsets_fit_32(h->g);
  with_lattice(h->g.lat, [&]<int LAT>() {
    with_type(h->stype, [&]<typename T>() {
      auto go = [&](auto kern) {
        hipLaunchKernelGGL(kern, dim3(grid), dim3(bs), 0, h->stream, static_cast<T *>(h->spin), h->seed, h->g,
                           h->rule, m, color, acc);
      };
      // sq/8n and sc/26n: the x-shift side is the colour's x parity, a
      // constant of the launch, so it is a template argument
      auto with_x = [&]<bool TWO, typename I>() {
        if constexpr (LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N) {
          if (color & 1) go(k_sweep_color<LAT, T, kVec, TWO, I, 1>);
          else go(k_sweep_color<LAT, T, kVec, TWO, I, 0>);
        } else {
          go(k_sweep_color<LAT, T, kVec, TWO, I, -1>);
        }
      };
      if constexpr (sizeof(T) == 1) {
        if (two) {
          if (off32) with_x.template operator()<true, uint32_t>();
          else with_x.template operator()<true, int64_t>();
          return;
        }
      }
      if (off32) with_x.template operator()<false, uint32_t>();
      else with_x.template operator()<false, int64_t>();
    });
  });
  return check_hip(hipGetLastError(), "sweep kernel launch");
}

void drop_graphs(spk_hip_lattice *h) {
  for (auto &c : h->graphs) (void)hipGraphExecDestroy(c.exec);
  h->graphs.clear();
}

// Two-state sq/4n lattices on the per-colour path sweep on bit planes.
// (bits_events takes the proposal from bit 30 of the first draw, so half
// must be 2^30, which RandomPark's AM*s >= 0.5 gives)
bool bits_eligible(const spk_hip_lattice *h) {
  return h->bitplanes && h->g.lat == SPK_HIP_SQ_4N && h->rule.nspins == 2 && h->stype == kU8 &&
         h->rule.half == (1 << 30) &&
         (!variant_app(h->d.app) || h->d.app == SPK_HIP_ISING_SINGLE);
}

// LDS bytes of the resident kernel's copy of the state (spins, then seeds
// at a 16-byte boundary), or 0 when the lattice does not fit one workgroup.
size_t resident_bytes(const spk_hip_lattice *h) {
  if (variant_app(h->d.app) || !h->resident) return 0;
  const size_t slots = (size_t)h->g.K * h->g.Mp;
  const size_t bytes = (slots * spin_bytes(h->stype) + 15) / 16 * 16 + slots * sizeof(int32_t);
  return bytes <= h->max_lds ? bytes : 0;
}

// VALU instructions of a site event in the packed kernels, roughly: a part
// per site (draws, proposal, decision) and one per neighbour.  From the
// counters: 54 a site for two states on sq/4n, 71 for u8 on sq/8n, 131 for
// u16 on sc/26n.
double site_valu(const spk_hip_lattice *h) {
  const int nn = maxneigh_of(h->g.lat);
  if (h->rule.nspins == 2) return 40 + 3.5 * nn;
  return h->stype == kU8 ? 45 + 3.3 * nn : h->stype == kU16 ? 66 + 2.5 * nn : 60 + 4.5 * nn;
}

// potts/neigh and potts/neighonly
bool first_appearance(const spk_hip_lattice *h) { return variant_app(h->d.app) && h->d.app != SPK_HIP_ISING_SINGLE; }

// The same for the tile kernel's one-site events.
double tile_site_valu(const spk_hip_lattice *h) {
  const int nn = maxneigh_of(h->g.lat);
  // the first-appearance rules compare every pair of neighbours, each
  // compare's mask through the scalar unit (counted as their time, not only
  // their instructions: 5.2 us a pass of sc/26n with one wavefront a SIMD)
  if (first_appearance(h)) return 75 + 8.0 * nn + 1.9 * nn * nn;
  return h->rule.nspins == 2 ? 70 + 2.0 * nn : 75 + 5.0 * nn;
}

constexpr double kUsPerValu = 4.0 / 2400.0;   // a wavefront's instruction on its SIMD: 4 cycles at 2.4 GHz
constexpr int kSimds = 4, kCus = 256;

// Whether a pass on bit planes (two colours) is faster than two of the packed
// kernel.  Rows of an awkward width leave bits of their plane words empty, as work
// and as seed memory (hx 8: three quarters of them).  Both sides' times fitted
// to 487 lattices from 16 x 100^2 to 256^3 and 40 x 1000^2, Q of 5 to 10^6,
// mostly within 5%: two of them are on the slower side, by 1 and 4%.  us a sweep,
// packed and on planes:
//   16 x 400^2 Q=5 38.3, 33.2; Q=3000 42.3, 45.8; 16 x 700^2 Q=5 55.5, 64.3
//   16 x 1000^2 Q=100 82.1, 134; Q=10^4 97, 190; 32 x 512^2 Q=100 55.7, 49.7; Q=60000 62.8, 66.6
//   40 x 400^2 Q=5 52.0, 34.6; Q=10^6 76.6, 57.9; 256^3 Q=5 80.2, 42.9; Q=10^6 142, 74.9
bool slice_pays(const spk_hip_lattice *h) {
  const SliceGeom sg = slice_geom(h->g, h->rule.nspins);
  const double waves = sg.waves / 1024.0, planes = 4.1 + 0.33 * sg.PG + waves * (1.28 + 0.469 * sg.PG);
  const double pw = (double)h->g.Mp / 4 / 64 / 1024;   // the packed kernel's wavefronts
  const double packed = h->stype == kU8    ? std::max(4.0, 3.7 + 0.855 * pw)
                        : h->stype == kU16 ? std::max(4.3, 4.05 + 1.038 * pw)
                                           : std::max(4.8, 3.8 + 1.83 * pw);
  return planes < 0.98 * 2 * packed;
}

// Lattices that sweep on bit planes of the spins (spk_slice.h).
bool slice_eligible(const spk_hip_lattice *h) {
  return h->slice_ok && !variant_app(h->d.app) && !h->block_set && slice_fits(h->g, h->rule.nspins) &&
         h->rule.half == (1 << 30) && slice_pays(h);
}

// Microseconds a sweep is expected to take on bit planes, one colour a launch
// and two sweeps a launch.
double colour_bits_us(const spk_hip_lattice *h) { return 2 * std::max(4.7 + 0.38e-6 * h->N, 2.5 + h->N / 1520e3); }
double pair_sweep_us(const spk_hip_lattice *h) {
  const int band = pair_band(h->g), rounds = ((h->g.hy + band - 1) / band + kCus - 1) / kCus;
  // band rows of the four passes, wavefronts a row, their time a row
  const double rows = 4 * band + 12, waves = pair_stage((h->g.hx + 31) / 32) / 64;
  double us = h->d.app == SPK_HIP_ISING_SINGLE ? 0.085 : 0.105;
  // bands that wait for a compute unit, of rows that fill one wavefront a group:
  // 1.0 to 1.3 of that time
  if (rounds > 1 && waves == 1) us *= 1.3;
  return (5.0 + rounds * rows * waves * us) / 2;
}

// Two sweeps a launch on bit planes where that is faster (of 160 lattices two are on
// the slower side, by 3 and 6%).  us a sweep, one colour a launch and two sweeps a launch:
// ising/single 44 x 4748 8.6, 9.7; 834 x 8680 13.6, 14.7; 558 x 9782 12.6, 14.9;
// 1580 x 5552 17.8, 15.7; Ising 1404 x 7722 23.5, 20.8
bool pair_pays(const spk_hip_lattice *h) { return pair_fits(h->g) && pair_sweep_us(h) < colour_bits_us(h); }

// Microseconds a sweep is expected to take through the kernels that pass
// over the lattice one colour at a time (bit planes where they apply) or in
// one workgroup.  Short passes are latency: 3 us and a thread's own chain
// (measured 3.5 us on sc/6n at 40^3, 4.2 on sc/26n at 32^3 to 100^3, 5.1-6.2
// on bit planes at 256^2 to 2000^2).
double plain_sweep_us(const spk_hip_lattice *h) {
  if (resident_bytes(h)) {
    const double waves = std::ceil((double)h->g.Mp / 4 / 64);
    return h->g.K * (0.25 + std::max(1.0, waves / kSimds) * 4 * site_valu(h) * kUsPerValu * 1.2);
  }
  if (bits_eligible(h))
    return h->bitplanes == 1 && pair_pays(h) ? pair_sweep_us(h) : colour_bits_us(h);
  if (slice_eligible(h)) {
    // a wavefront's own time, and what a launch adds as its wavefronts fill
    // the SIMDs (22 to 31 us a sweep for 1 to 5 plane groups up to 128^3, 41
    // to 78 at 256^3)
    const SliceGeom sg = slice_geom(h->g, h->rule.nspins);
    return h->g.K / 2 * (4.6 + 0.55 * sg.PG + sg.waves / 4096.0 * (3.4 + 1.75 * sg.PG));
  }
  if (neigh_packed(h)) {   // 6.9-7.1 us a pass of sc/26n up to 128^3, 10.9 at 160^3, 31 at 256^3
    const int nn = maxneigh_of(h->g.lat);
    const double us = (260 + 30 * nn + 1.5 * nn * (nn - 1)) * kUsPerValu, waves = (double)h->g.Mp / 4 / 64;
    return h->g.K * std::max(3.0 + 1.2 * us, 2.6 + 1.06 * waves / (kCus * kSimds) * us);
  }
  if (variant_app(h->d.app)) {
    const double us = tile_site_valu(h) * kUsPerValu, waves = (double)h->g.Mp / 64;
    return h->g.K * std::max(3.0 + 1.6 * us, 2.6 + 0.8 * waves / (kCus * kSimds) * us);
  }
  const double us = 4 * site_valu(h) * kUsPerValu, waves = (double)h->g.Mp / 4 / 64;
  return h->g.K * std::max(3.0 + 1.2 * us, 2.6 + 1.5 * waves / (kCus * kSimds) * us);
}

// a wavefront's time for one item (vec sites a thread) of a tile pass
double tile_item_us(const spk_hip_lattice *h, int vec) {
  return (vec == 1 ? tile_site_valu(h) : 4 * site_valu(h) + 40) * kUsPerValu;
}

// Microseconds a sweep is expected to take in boxes of w sites, S sweeps a
// launch, vec sites a thread: the launch with its loads and stores, then each
// pass bound by the wavefronts a SIMD has of it or by one wavefront's own time.
// us a sweep no better than `best` come back as 1e30.
double tile_sweep_us(const spk_hip_lattice *h, const int (&w)[3], int S, int vec, const TileRegion &r, double best,
                     TileShape *shape) {
  const int size = (int)spin_bytes(h->stype), K = h->g.K;
  Geom gl;
  geom_init(gl, h->g.lat, r.ext[0], r.ext[1], r.ext[2]);
  const int64_t slots = (int64_t)K * gl.Mp;
  const size_t lds = (size_t)((slots * size + 15) / 16 * 16 + slots * 4);   // tile_lds of the plan
  if (lds > h->max_lds) return 1e30;
  uint32_t items[kTileMaxPass], most = 0;
  for (int k = 0, c = 0; k < S * K; k++, c = c + 1 == K ? 0 : c + 1) {
    const TileSpan t = tile_span(h->g.lat, r, k, c);
    items[k] = tile_packs(t, vec) * (uint32_t)(t.b[1] - t.b[0]) * (uint32_t)(t.e[1] - t.e[0]);
    most = std::max(most, items[k]);
  }
  const uint32_t packs = (uint32_t)(slots / 4);   // loaded and stored by every thread
  const int block = (int)std::min<uint32_t>(1024, (std::max(most, packs) + 63) / 64 * 64);
  int64_t tiles = 1;
  const int n[3] = {h->g.nx, h->g.ny, h->g.nz};
  double own = 1;
  for (int d = 0; d < 3; d++) tiles *= r.whole[d] ? 1 : (n[d] + w[d] - 1) / w[d], own *= r.whole[d] ? n[d] : w[d];
  const int per_cu = (int)((tiles + kCus - 1) / kCus);
  const int fit = std::max(1, std::min((int)((160 << 10) / (lds + 1024)), 16 * 64 / block));   // boxes a CU holds at once
  const int together = std::min(per_cu, fit), rounds = (per_cu + together - 1) / together;
  const double item_us = tile_item_us(h, vec);
  const double moved = (double)lds + own * (4 + size);   // bytes a box moves
  double us = together * moved / 20e3;   // a CU's share of the memory rate, about 20 GB/s a us
  const uint32_t threads = (uint32_t)block;
  for (int k = 0; k < S * K; k++) {
    const double waves = (items[k] + 63) / 64, turns = (items[k] + threads - 1) / threads;
    us += 0.3 + std::max(turns * (0.15 + 1.3 * item_us), 1.2 * together * waves / kSimds * item_us);
  }
  // (a site a thread: 1.05 to 1.4 of that in 900 lattices, but for the
  // first-appearance rules' 0.9 to 1.3; packs 0.8 to 1.2)
  if (vec == 1 && !first_appearance(h)) us *= 1.15;
  us = (5.0 + rounds * us) / S;
  if (us >= best) return 1e30;
  *shape = TileShape{{w[0], w[1], w[2]}, S, vec, block};
  return us;
}

// Whether boxes of w sites fit LDS for launches that start at any colour
// (launch_tiles): a launch of fewer passes needs no more halo than S sweeps
// that end at the same colour.
bool tile_fits(const spk_hip_lattice *h, const int (&w)[3], int S, int vec) {
  for (int c = 0; c < h->g.K; c++) {
    TilePlan tp;
    if (!tile_plan_make(h->g, w, c, S * h->g.K, vec, (int)spin_bytes(h->stype), &tp) || tile_lds(tp) > h->max_lds)
      return false;
  }
  return true;
}

// The boxes for this lattice and its settings, or none (sweeps 0) where the
// other kernels are expected to be as fast.
void tile_choose(spk_hip_lattice *h) {
  h->tile_known = true;
  h->tile = TileShape{};
  // settings that name another kernel keep it
  if (h->block_set || (h->resident_set && resident_bytes(h))) return;
  if (h->g.lat == SPK_HIP_SQ_4N && h->rule.nspins == 2 && h->stype == kU8 && h->bitplanes != 1) return;
  if (h->N > (int64_t)8 << 20 || !offsets_fit_32(h->g)) return;
  // the gain the model can be trusted with (within a fifth of the measured
  // time): of 2000 lattices of 2000 to 8 * 10^6 sites four are slower in boxes, by 4 to 9%
  double best = (resident_bytes(h)                    ? 0.86
                 : slice_eligible(h)                  ? 0.93
                 : h->d.app == SPK_HIP_ISING_SINGLE   ? 0.97
                                                      : 0.9) *
                plain_sweep_us(h);
  auto sizes = [](int n, int unit) {   // extents that cut n into near-equal boxes
    std::vector<int> v;
    for (int cuts : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16, 20, 24, 28, 32, 40, 48, 64}) {
      const int e = ((n + cuts - 1) / cuts + unit - 1) / unit * unit;
      if (v.empty() || e < v.back()) v.push_back(cuts == 1 ? n : e);
    }
    return v;
  };
  const std::vector<int> vx = sizes(h->g.nx, 8), vy = sizes(h->g.ny, 2), vz = sizes(h->g.nz, 2);
  const int64_t most = std::min<int64_t>(h->N - 1, (int64_t)h->max_lds / (4 + (int)spin_bytes(h->stype)));
  const int64_t fewest = (h->N + 1023) / 1024;   // sites of a box: at most 1024 boxes, at least two
  const double item_us[2] = {tile_item_us(h, 1), tile_item_us(h, kVec)}, move_us = 2.0 * (4 + spin_bytes(h->stype)) / 20e3;
  const int vecs = variant_app(h->d.app) ? 1 : 2;
  TileRegion region;
  for (int wx : vx)
    for (int wy : vy) {
      if ((int64_t)wx * wy * vz[0] < fewest) break;   // extents fall
      for (int wz : vz) {
        const int64_t own = (int64_t)wx * wy * wz;
        if (own < fewest) break;
        if (own > most) continue;
        const int per_cu = (int)(((h->N + own - 1) / own + kCus - 1) / kCus);
        const int w[3] = {wx, wy, wz};
        double pass_us[2];   // no less than this a pass whatever the halo: most shapes end here
        for (int v = 0; v < vecs; v++)
          pass_us[v] = 0.3 + std::max(0.15 + 1.3 * item_us[v],
                                      1.2 * per_cu * ((double)own / h->g.K / (v ? kVec : 1)) / 64 / kSimds * item_us[v]);
        for (int S : {1, 2, 3, 4, 6, 8}) {
          if (S * h->g.K > kTileMaxPass) break;
          bool known = false;
          for (int v = 0; v < vecs; v++) {
            if ((5.0 + per_cu * own * move_us) / S + h->g.K * pass_us[v] >= best) continue;
            if (!known && !(known = tile_region(h->g, w, 0, S * h->g.K, region))) break;
            const int vec = v ? kVec : 1;
            TileShape t;
            const double us = tile_sweep_us(h, w, S, vec, region, best, &t);
            if (us < best && tile_fits(h, w, S, vec)) best = us, h->tile = t;
          }
        }
      }
    }
}

// Which kernels a sweeps call of a lattice beyond one workgroup's reach takes
// (enter_route: a single sweep may take another).
Route route(spk_hip_lattice *h) {
  if (!h->tile_known) tile_choose(h);
  if (h->tile.sweeps > 0) return kRouteTile;
  if (bits_eligible(h)) return kRouteBits;
  return slice_eligible(h) ? kRouteSlice : kRouteColour;
}

// LDS bytes of the resident kernel where a call of n sweeps runs on it, else
// 0.  A single sweep stays there also where more would take boxes: they need
// two launches, so that the state ends where it began.
size_t resident_call(spk_hip_lattice *h, int n) {
  const size_t lds = resident_bytes(h);
  return lds && (n == 1 || route(h) != kRouteTile) ? lds : 0;
}

// Packs the state into the planes (allocated on first use) and routes the
// colour passes there until bits_leave.
// (Re)allocates a shadow seed array to hold `slots` slots.
int ensure_shadow(spk_hip_lattice *h, int32_t *&p, int64_t &cap, int64_t slots) {
  if (slots <= cap) return SPK_HIP_OK;
  (void)hipStreamSynchronize(h->stream);
  if (p) (void)hipFree(p);
  cap = 0;
  if (hipMalloc(&p, (size_t)slots * sizeof(int32_t)) != hipSuccess) {
    p = nullptr;
    return set_error(SPK_HIP_ENOMEM, "bit-plane shadow seeds not available");
  }
  cap = slots;
  return SPK_HIP_OK;
}

int ensure_planes(uint32_t *&p, const spk_hip_lattice *h) {
  if (p) return SPK_HIP_OK;   // 2*hy*pw words whatever the sites per thread
  if (hipMalloc(&p, 2 * (size_t)h->g.hy * h->bg.pw * sizeof(uint32_t)) != hipSuccess) {
    p = nullptr;
    return set_error(SPK_HIP_ENOMEM, "bit-plane shadow state not available");
  }
  return SPK_HIP_OK;
}

int bits_enter(spk_hip_lattice *h) {
  h->pairs = h->pairs_ok && h->bitplanes == 1 && pair_pays(h);
  h->bg = bit_geom(h->g, h->pairs ? 8 : h->bitplanes == 1 ? kBitSites : h->bitplanes);
  int rc;
  if ((rc = ensure_planes(h->bits, h)) || (rc = ensure_shadow(h, h->sseed, h->sseed_cap, 2 * h->bg.seedc)))
    return rc;
  if (h->pairs &&
      ((rc = ensure_planes(h->bits2, h)) || (rc = ensure_shadow(h, h->sseed2, h->sseed2_cap, 2 * h->bg.seedc)))) {
    if (rc != SPK_HIP_ENOMEM) return rc;
    (void)hipGetLastError();   // no room for the second planes: one colour a launch, which needs none
    (void)hipFree(h->bits2);
    h->bits2 = nullptr;
    h->pairs_ok = false;
    return bits_enter(h);
  }
  const int64_t words = 2 * (int64_t)h->g.hy * h->bg.pw;
  hipLaunchKernelGGL(k_bits_pack, dim3(grid_for(words, 256)), dim3(256), 0, h->stream,
                     static_cast<const uint8_t *>(h->spin), h->g, h->bg, h->bits);
  hipLaunchKernelGGL(k_seeds_to_shadow, dim3(grid_for(h->bg.seedc / 2, 256)), dim3(256), 0, h->stream, h->seed,
                     h->g, h->bg, h->sseed);
  rc = check_hip(hipGetLastError(), "bit-plane pack");
  if (!rc) h->bits_active = true;
  return rc;
}

// The same for a bit-sliced lattice.
int slice_enter(spk_hip_lattice *h) {
  h->sg = slice_geom(h->g, h->rule.nspins);
  const int64_t words = (int64_t)h->g.K * h->sg.nw;
  int rc;
  if (!h->bits && hipMalloc(&h->bits, (size_t)words * h->sg.PG * sizeof(Words<4>)) != hipSuccess) {
    h->bits = nullptr;
    return set_error(SPK_HIP_ENOMEM, "bit planes not available");
  }
  if ((rc = ensure_shadow(h, h->sseed, h->sseed_cap, h->g.K * h->sg.seedc))) {
    (void)hipFree(h->bits);   // of no use without the seeds
    h->bits = nullptr;
    return rc;
  }
  slice_in(h->stream, h->spin, h->stype, h->seed, h->g, h->sg, h->bits, h->sseed);
  rc = check_hip(hipGetLastError(), "bit-plane pack");
  if (!rc) h->slice_active = true;
  return rc;
}

int slice_leave(spk_hip_lattice *h) {
  h->slice_active = false;
  slice_out(h->stream, h->bits, h->sseed, h->g, h->sg, h->spin, h->stype, h->seed);
  return check_hip(hipGetLastError(), "bit-plane unpack");
}

// One launch of the sliced pass: colours 2m and 2m+1.
int launch_slice(spk_hip_lattice *h, int m, unsigned long long *acc) {
  const SliceGeom &s = h->sg;
  const int per = kSliceThreads / 64;
  unsigned grid = (unsigned)((s.waves + per - 1) / per);
  grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
  auto go = [&](auto kern) {
    hipLaunchKernelGGL(kern, dim3(grid), dim3(kSliceThreads), 0, h->stream, h->bits, h->sseed, h->g, s, h->rule, m,
                       acc);
  };
  with_plane_groups(s.PG, [&]<int PG>() {
    s.W == 32 && s.last == 32 ? go(k_sweep_slice<true, PG>) : go(k_sweep_slice<false, PG>);
  });
  return check_hip(hipGetLastError(), "sliced sweep launch");
}

int bits_leave(spk_hip_lattice *h) {
  if (h->slice_active) return slice_leave(h);
  if (!h->bits_active) return SPK_HIP_OK;
  h->bits_active = false;
  const int64_t words = 2 * (int64_t)h->g.hy * h->bg.pw;
  hipLaunchKernelGGL(k_bits_unpack, dim3(grid_for(words, 256)), dim3(256), 0, h->stream, h->bits, h->g, h->bg,
                     static_cast<uint8_t *>(h->spin));
  hipLaunchKernelGGL(k_seeds_from_shadow, dim3(grid_for(h->bg.seedc / 2, 256)), dim3(256), 0, h->stream,
                     h->sseed, h->g, h->bg, h->seed);
  return check_hip(hipGetLastError(), "bit-plane unpack");
}

__global__ void k_zero_u64(unsigned long long *__restrict__ v, int64_t n) {
  const int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) v[t] = 0ull;
}

// The tile kernel's second state buffers; without room for them the
// lattice keeps to the other kernels.
bool ensure_tile_buffers(spk_hip_lattice *h) {
  if (!h->spin2) {
    const size_t sb = (size_t)h->slots * spin_bytes(h->stype), kb = (size_t)h->slots * sizeof(int32_t);
    if (hipMalloc(&h->spin2, sb) != hipSuccess) h->spin2 = nullptr;
    if (h->spin2 && hipMalloc(&h->seed2, kb) != hipSuccess) {
      (void)hipFree(h->spin2);
      h->spin2 = nullptr;
      h->seed2 = nullptr;
    }
    if (!h->spin2) {
      (void)hipGetLastError();   // not an error of the call
      h->tile = TileShape{};
    }
  }
  return h->spin2 != nullptr;
}

// Lattices of boxes that make a call of one sweep one colour a launch (from
// the host, as boxes are): boxes would take two launches whatever their size,
// each with its halo.  us a call, boxes and colours: sc/6n 16 x 14 x 92 30, 27; sq/4n
// 692 x 580 33, 28, 5126 x 220 41, 31, 234 x 9944 46, 31; sq/8n 1156 x 380 34, 47, 1066 x
// 1402 40, 47, 390 x 6628 56, 49, 1174 x 4090 61, 49.
bool tile_single(const spk_hip_lattice *h) { return h->g.K == 2 || (h->g.K == 4 && h->N > 7 << 18); }

// Brings the state to the layout the next n sweeps run on: the bit planes, or
// the bytes.
int enter_route(spk_hip_lattice *h, int n, Route *out) {
  Route rt = route(h);
  if (rt == kRouteTile && n == 1 && tile_single(h)) rt = kRouteColour;
  if (rt == kRouteTile && !ensure_tile_buffers(h)) rt = route(h);
  *out = rt;
  if (rt == kRouteBits) return h->bits_active ? SPK_HIP_OK : bits_enter(h);
  if (rt == kRouteSlice) {
    const int rc = h->slice_active ? SPK_HIP_OK : slice_enter(h);
    if (rc != SPK_HIP_ENOMEM) return rc;
    (void)hipGetLastError();   // no room for the planes: the per-colour kernels
    h->slice_ok = false;
    *out = kRouteColour;
    return SPK_HIP_OK;
  }
  return bits_leave(h);
}

int64_t sweep_launches(const spk_hip_lattice *h, int n, Route route);
// Whether n sweeps are replayed from graphs.  Two launches are soon made: a
// call of one sweep took 42 us replayed and 33 so on 150 x 130 x 110 sc/6n, 43 and
// 34 on 410 x 7614 sq/4n, 58 and 48 on 4096^2 Ising.  Boxes (and tile_single's colours)
// are launched from the host (launch_tiles), but for long calls of the first-appearance
// rules on sc/26n, whose launches take 45 us and more: 24 sweeps of 92 x 32 x 44 1183 us
// replayed, 1201 launched.
bool replayed(const spk_hip_lattice *h, int n, Route route) {
  if (h->chunk == 0) return false;
  if (route == kRouteTile) return first_appearance(h) && h->g.K == 8 && sweep_launches(h, n, route) >= 8;
  return h->tile.sweeps == 0 && sweep_launches(h, n, route) > 2;
}

int ensure_pinned(spk_hip_lattice *h, int rows) {
  if (rows <= h->pinned_rows) return SPK_HIP_OK;
  int cap = std::max(rows, 2 * h->pinned_rows);
  unsigned long long *p = nullptr;
  if (hipHostMalloc(&p, (size_t)cap * 2 * sizeof(unsigned long long), hipHostMallocDefault) !=
      hipSuccess)
    return set_error(SPK_HIP_ENOMEM, "pinned host allocation failed");
  if (h->pinned) {
    (void)hipStreamSynchronize(h->stream);
    (void)hipHostFree(h->pinned);
  }
  h->pinned = p;
  h->pinned_rows = cap;
  return SPK_HIP_OK;
}

// Pinned memory for the whole state of a small lattice; without it downloads
// go through the staging array.
bool ensure_pinned_state(spk_hip_lattice *h) {
  if (!h->pinned_state && hipHostMalloc(&h->pinned_state, 2 * (size_t)h->N * sizeof(int32_t), hipHostMallocDefault) !=
                              hipSuccess) {
    h->pinned_state = nullptr;
    (void)hipGetLastError();   // not an error of the call
  }
  return h->pinned_state != nullptr;
}

// Two sweeps in one launch (k_sweep_bits_pair), from the planes and seeds
// at `from` (0: bits/sseed, 1: bits2/sseed2) to the others.
int launch_pair(spk_hip_lattice *h, int from, unsigned long long *acc) {
  launch_pair_kernel(h->stream, from ? h->bits2 : h->bits, from ? h->sseed2 : h->sseed, from ? h->bits : h->bits2,
                     from ? h->sseed : h->sseed2, h->g, h->bg, h->rule, h->d.app == SPK_HIP_ISING_SINGLE, acc);
  return check_hip(hipGetLastError(), "two-sweep launch");
}

// Sweep-kernel launches that launch_sweeps makes for n sweeps.
int tile_launches(const spk_hip_lattice *h, int n);
int64_t sweep_launches(const spk_hip_lattice *h, int n, Route route) {
  if (route == kRouteTile) return tile_launches(h, n);
  if (h->slice_active) return (int64_t)h->g.K / 2 * n;
  if (h->bits_active && h->pairs) return 2 * (n / 4) + (int64_t)h->g.K * (n % 4);
  return (int64_t)h->g.K * n;
}

// Launches of n sweeps through the tile kernel: an even number, so that the
// state ends where it began; a single sweep is split between its colours.
int tile_launches(const spk_hip_lattice *h, int n) {
  const int m = (n + h->tile.sweeps - 1) / h->tile.sweeps;
  return n == 1 ? 2 : (m + 1) / 2 * 2;
}

// One launch of the tile kernel: colour passes [q0, q1) of a run of sweeps,
// from buffer `from` (0: spin/seed, 1: spin2/seed2) to the other; acc is the
// row of sweep 0.
int launch_tile(spk_hip_lattice *h, int from, int q0, int q1, unsigned long long *acc) {
  TilePlan tp;
  if (!tile_plan_make(h->g, h->tile.w, q0 % h->g.K, q1 - q0, h->tile.vec, (int)spin_bytes(h->stype), &tp))
    return set_error(SPK_HIP_ESTATE, "no box plan for %d colour passes", q1 - q0);
  const size_t lds = tile_lds(tp);
  unsigned grid = (unsigned)(tp.cx * tp.cy * tp.cz);
  grid = (grid + kNumXcd - 1) / kNumXcd * kNumXcd;   // xcd_tile needs a multiple of 8
  const bool two = h->rule.nspins == 2;
  with_lattice(h->g.lat, [&]<int LAT>() {
    with_type(h->stype, [&]<typename T>() {
      T *s0 = static_cast<T *>(h->spin), *s1 = static_cast<T *>(h->spin2);
      auto go = [&](auto kern) {
        allow_lds(kern, lds);
        hipLaunchKernelGGL(kern, dim3(grid), dim3(h->tile.block), lds, h->stream, from ? s1 : s0,
                           from ? h->seed2 : h->seed, from ? s0 : s1, from ? h->seed : h->seed2, h->g, h->rule, tp,
                           acc + (size_t)(q0 / h->g.K) * kAccRow);
      };
      const int app = h->d.app;
      if (app == SPK_HIP_POTTS_NEIGH) return go(k_sweep_tile<LAT, T, false, 1, SPK_HIP_POTTS_NEIGH>);
      if (app == SPK_HIP_POTTS_NEIGHONLY) return go(k_sweep_tile<LAT, T, false, 1, SPK_HIP_POTTS_NEIGHONLY>);
      const bool one = h->tile.vec == 1;
      if constexpr (sizeof(T) == 1) {   // two states are always stored as u8
        if (app == SPK_HIP_ISING_SINGLE) return go(k_sweep_tile<LAT, T, true, 1, SPK_HIP_ISING_SINGLE>);
        if (two) return one ? go(k_sweep_tile<LAT, T, true, 1, SPK_HIP_POTTS>) : go(k_sweep_tile<LAT, T, true, kVec, SPK_HIP_POTTS>);
      }
      one ? go(k_sweep_tile<LAT, T, false, 1, SPK_HIP_POTTS>) : go(k_sweep_tile<LAT, T, false, kVec, SPK_HIP_POTTS>);
    });
  });
  return check_hip(hipGetLastError(), "tile sweep launch");
}

// n sweeps through the tile kernel, split evenly over its launches: whole
// sweeps each, or (one sweep, or one sweep a launch and an odd number of
// them) at colours inside a sweep.  Launched one by one rather than captured
// (replayed): the device takes longer over a launch than the host, and a graph for
// each number of sweeps and each temperature cost 70 us where one workgroup had
// needed none.  us
// a call of 2, 10 and 200 sweeps: 100^2 Ising replayed 49, 50, 492, launched 32, 43,
// 425; 128^2 sq/8n 45, 66, 857 and 35, 59, 786; 64^3 sc/26n 59, 176, 3018 and
// 51, 175, 2980.  After a change of temperature 2 sweeps took 126, 125 and 134.
int launch_tiles(spk_hip_lattice *h, int n, unsigned long long *acc, int64_t *nlaunch) {
  const int m = tile_launches(h, n);
  auto cut = [&](int j) {
    return m > n ? (int)((int64_t)n * h->g.K * j / m) : (int)((int64_t)n * j / m) * h->g.K;
  };
  for (int j = 0; j < m; j++, (*nlaunch)++)
    if (const int rc = launch_tile(h, j & 1, cut(j), cut(j + 1), acc)) return rc;
  return SPK_HIP_OK;
}

// launches of sweeps whose accumulator rows start at acc; returns launches.
// On planes in the pair layout, every four sweeps are two two-sweep
// launches, there and back, so the state ends in bits/sseed; the last n % 4
// sweeps take the per-colour kernel.
int launch_sweeps(spk_hip_lattice *h, int n, unsigned long long *acc, int64_t *nlaunch) {
  int rc;
  int s = 0;
  if (h->bits_active && h->pairs)
    for (; s + 4 <= n; s += 4, *nlaunch += 2)
      if ((rc = launch_pair(h, 0, acc + (size_t)s * kAccRow)) ||
          (rc = launch_pair(h, 1, acc + (size_t)(s + 2) * kAccRow)))
        return rc;
  if (h->slice_active)
    for (; s < n; s++)
      for (int m = 0; m < h->g.K / 2; m++, (*nlaunch)++)
        if ((rc = launch_slice(h, m, acc + (size_t)s * kAccRow))) return rc;
  for (; s < n; s++)
    for (int c = 0; c < h->g.K; c++, (*nlaunch)++)
      if ((rc = launch_sweep(h, c, acc + (size_t)s * kAccRow))) return rc;
  return SPK_HIP_OK;
}

// folds `rows` accumulator rows at acc into compact (Naccept, dE) pairs at out
int launch_fold(spk_hip_lattice *h, const unsigned long long *acc, int rows, unsigned long long *out) {
  hipLaunchKernelGGL(k_fold_rows, dim3(rows), dim3(64), 0, h->stream, acc, kAccSlots, kAccRow,
                     out);
  return check_hip(hipGetLastError(), "fold launch");
}

// nsweeps sweeps through the resident kernel, in pieces of at most
// kInitialAccRows sweeps, each writing pinned rows [done, ..).
int run_resident(spk_hip_lattice *h, int nsweeps, size_t lds, int64_t *nlaunch) {
  int rc;
  if ((rc = check_hip(hipEventRecord(h->ev0, h->stream), "event"))) return rc;
  for (int done = 0; done < nsweeps;) {
    const int n = std::min(nsweeps - done, kInitialAccRows);
    const bool two = h->rule.nspins == 2;
    with_lattice(h->g.lat, [&]<int LAT>() {
      with_type(h->stype, [&]<typename T>() {
        auto go = [&](auto kern) {
          allow_lds(kern, lds);
          hipLaunchKernelGGL(kern, dim3(1), dim3(1024), lds, h->stream, static_cast<T *>(h->spin), h->seed, h->g,
                             h->rule, n, h->pinned + (size_t)done * 2);
        };
        if constexpr (sizeof(T) == 1) {
          if (two) {
            go(k_sweep_resident<LAT, T, true>);
            return;
          }
        }
        go(k_sweep_resident<LAT, T, false>);
      });
    });
    if ((rc = check_hip(hipGetLastError(), "resident sweep launch"))) return rc;
    (*nlaunch)++;
    done += n;
  }
  return check_hip(hipEventRecord(h->ev1, h->stream), "event");
}

void row_sum(const spk_hip_lattice *h, int row, int64_t *x, int64_t *y);

// After the launches of a sweeps call: waits, takes the timing, and turns
// the folded rows in pinned memory into cumulative Naccept and energies.
int finish_sweeps(spk_hip_lattice *h, int nsweeps, int64_t nlaunch, int64_t e0, int64_t *naccept_total,
                  int64_t *naccept_per_sweep, double *energy_per_sweep) {
  int rc;
  if ((rc = check_hip(hipStreamSynchronize(h->stream), "sweeps sync"))) return rc;
  float ms = 0.f;
  if ((rc = check_hip(hipEventElapsedTime(&ms, h->ev0, h->ev1), "event time"))) return rc;
  h->last_ms = ms;
  h->last_nlaunch = nlaunch;
  int64_t nacc = 0, eng = e0;
  const bool track = h->energy_valid || energy_per_sweep;
  if (track && !energy_per_sweep) eng = h->energy;
  for (int s = 0; s < nsweeps; s++) {
    int64_t a, de;
    row_sum(h, s, &a, &de);
    nacc += a;
    eng += 2 * de;   // a flip changes site i's and its neighbours' counts
    if (naccept_per_sweep) naccept_per_sweep[s] = nacc;
    if (energy_per_sweep) energy_per_sweep[s] = (double)eng;
  }
  if (naccept_total) *naccept_total += nacc;
  if (track) h->energy = eng;
  h->energy_valid = track;
  return SPK_HIP_OK;
}


// The graph of `n` sweeps on the current layout (bit planes or bytes):
// a kernel zeroes accumulator rows [0, n) (no memset node), then the n
// sweeps' launches; the fold of those rows follows each replay.  Cached
// per (n, layout) until a settings change drops the cache.
int piece_graph(spk_hip_lattice *h, int n, Route rt, hipGraphExec_t *out) {
  for (auto &p : h->graphs)
    if (p.sweeps == n && p.route == rt) {
      *out = p.exec;
      return SPK_HIP_OK;
    }
  int rc;
  hipGraph_t graph = nullptr;
  if ((rc = check_hip(hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal), "begin capture")))
    return rc;
  const int64_t words = (int64_t)n * kAccRow;
  hipLaunchKernelGGL(k_zero_u64, dim3(grid_for(words, 256)), dim3(256), 0, h->stream, h->acc, words);
  int64_t nl = 0;
  rc = check_hip(hipGetLastError(), "zero launch");
  if (!rc) rc = rt == kRouteTile ? launch_tiles(h, n, h->acc, &nl) : launch_sweeps(h, n, h->acc, &nl);
  const hipError_t e = hipStreamEndCapture(h->stream, &graph);
  if (!rc) rc = check_hip(e, "end capture");
  if (rc) {
    if (graph) (void)hipGraphDestroy(graph);
    return rc;
  }
  hipGraphExec_t exec;
  rc = check_hip(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0), "graph instantiate");
  (void)hipGraphDestroy(graph);
  if (rc) return rc;
  h->graphs.push_back({n, rt, exec});
  *out = exec;
  return SPK_HIP_OK;
}

// Sweeps per graph replay of a call of n sweeps: n / chunk full graphs,
// then one of the remainder (so at most chunk + 1 graphs are ever cached,
// and a call shorter than chunk is a single replay).
std::vector<int> graph_pieces(int chunk, int n) {
  std::vector<int> p(chunk > 0 ? n / chunk : 0, chunk);
  if (chunk > 0 && n % chunk) p.push_back(n % chunk);
  return p;
}

int launch_energy(spk_hip_lattice *h, unsigned long long *acc) {
  with_lattice(h->g.lat, [&]<int LAT>() {
    with_type(h->stype, [&]<typename T>() {
      hipLaunchKernelGGL((k_energy<LAT, T>), dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream,
                         static_cast<const T *>(h->spin), h->g, acc);
    });
  });
  return check_hip(hipGetLastError(), "energy kernel launch");
}

int launch_fill_spins(spk_hip_lattice *h, int32_t value) {
  with_type(h->stype, [&]<typename T>() {
    hipLaunchKernelGGL((k_fill<T>), dim3(grid_for(h->slots, 256)), dim3(256), 0, h->stream,
                       static_cast<T *>(h->spin), h->slots, value);
  });
  return check_hip(hipGetLastError(), "fill kernel launch");
}

int ensure_acc(spk_hip_lattice *h, int nsweeps) {
  if (nsweeps <= h->acc_cap) return SPK_HIP_OK;
  int cap = h->acc_cap ? h->acc_cap : kInitialAccRows;
  while (cap < nsweeps) cap *= 2;
  unsigned long long *p = nullptr;
  if (hipMalloc(&p, (size_t)cap * kAccRow * sizeof(unsigned long long)) != hipSuccess)
    return set_error(SPK_HIP_ENOMEM, "device allocation of %d accumulator rows failed", cap);
  if (h->acc) {
    (void)hipStreamSynchronize(h->stream);
    (void)hipFree(h->acc);
  }
  drop_graphs(h);   // the accumulator addresses are baked into captured launches
  h->acc = p;
  h->acc_cap = cap;
  return SPK_HIP_OK;
}

// (Naccept, dE) of accumulator row `row`, already folded into h->pinned
void row_sum(const spk_hip_lattice *h, int row, int64_t *x, int64_t *y) {
  *x = (int64_t)h->pinned[2 * (size_t)row];
  *y = (int64_t)h->pinned[2 * (size_t)row + 1];
}

int compute_energy(spk_hip_lattice *h, int64_t *e) {
  int rc;
  if ((rc = bits_leave(h)) || (rc = ensure_acc(h, 1))) return rc;
  if ((rc = check_hip(hipMemsetAsync(h->acc, 0, kAccRow * sizeof(unsigned long long), h->stream), "memset")))
    return rc;
  if ((rc = launch_energy(h, h->acc)) || (rc = launch_fold(h, h->acc, 1, h->pinned))) return rc;
  if ((rc = check_hip(hipStreamSynchronize(h->stream), "energy sync"))) return rc;
  int64_t y;
  row_sum(h, 0, e, &y);
  h->energy = *e;
  h->energy_valid = true;
  return SPK_HIP_OK;
}

// ---------------------------------------------- sweeps without allocation
// Accumulator rows of spk_hip_sweeps_noalloc live in a file-scope device
// array, one copy per GPU, held until the process ends.  Host code uses the
// address hipGetSymbolAddress gives on each device (looked up once per
// device, when the first handle is created there), never the array's name,
// which in host code is only a stand-in.
constexpr int kNoAllocSweeps = 256;   // sweeps per call (8 KiB of rows each: 2 MiB)
constexpr int kMaxDevices = 64;
static __device__ __align__(256) unsigned long long scratch[(size_t)kNoAllocSweeps * kAccRow];
std::mutex g_scratch_mu;
unsigned long long *g_scratch[kMaxDevices] = {};

// Looks up the scratch array's address on the current device `device`.
int scratch_lookup(int device) {
  if (device < 0 || device >= kMaxDevices)
    return set_error(SPK_HIP_EDEVICE, "device %d beyond the %d this library serves", device, kMaxDevices);
  std::lock_guard<std::mutex> lock(g_scratch_mu);
  if (g_scratch[device]) return SPK_HIP_OK;
  void *p = nullptr;
  const int rc = check_hip(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)), "scratch symbol address");
  if (rc) return rc;
  g_scratch[device] = static_cast<unsigned long long *>(p);
  return SPK_HIP_OK;
}

int validate_on_device(spk_hip_lattice *h, const int32_t *buf, int lo, int hi, int64_t *nbad) {
  int rc = ensure_acc(h, 1);
  if (rc) return rc;
  if ((rc = check_hip(hipMemsetAsync(h->acc, 0, sizeof(unsigned long long), h->stream), "memset")))
    return rc;
  hipLaunchKernelGGL(k_count_outside, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, buf, h->N, lo,
                     hi, h->acc);
  if ((rc = check_hip(hipGetLastError(), "validate launch"))) return rc;
  if ((rc = check_hip(hipMemcpyAsync(h->pinned, h->acc, sizeof(*h->pinned), hipMemcpyDeviceToHost, h->stream),
                      "readback")) ||
      (rc = check_hip(hipStreamSynchronize(h->stream), "validate sync")))
    return rc;
  *nbad = (int64_t)h->pinned[0];
  return SPK_HIP_OK;
}

}  // namespace

// ====================================================================== ABI

extern "C" {

int spk_hip_ncolors(const spk_hip_desc *d) {
  Geom g;
  return make_geom(d, &g) ? SPK_HIP_EINVAL : g.K;
}

int spk_hip_create(const spk_hip_desc *d, spk_hip_lattice **out) {
  if (!d || !out) return set_error(SPK_HIP_EINVAL, "null argument");
  *out = nullptr;
  Geom g;
  int rc = make_geom(d, &g);
  if (rc) return rc;
  Rule r;
  if ((rc = make_rule(d->app, d->nspins, d->lattice, d->temperature, &r))) return rc;
  spk_hip_lattice *h = new (std::nothrow) spk_hip_lattice();
  if (!h) return set_error(SPK_HIP_ENOMEM, "host allocation failed");
  h->d = *d;
  h->g = g;
  h->rule = r;
  h->N = (int64_t)g.M * g.K;
  h->slots = (int64_t)g.Mp * g.K;
  h->stype = spin_type_for(d->app, d->nspins);
  // measured best on MI355X: 512 for 4096^2 sq/4n, 256 for 256^3 sc/26n
  h->block = (g.lat == SPK_HIP_SQ_4N || g.lat == SPK_HIP_SQ_8N) ? 512 : 256;
  if ((rc = check_hip(hipGetDevice(&h->device), "hipGetDevice")) || (rc = scratch_lookup(h->device)) ||
      (rc = check_hip(hipStreamCreate(&h->stream), "hipStreamCreate")) ||
      (rc = check_hip(hipEventCreate(&h->ev0), "hipEventCreate")) ||
      (rc = check_hip(hipEventCreate(&h->ev1), "hipEventCreate"))) {
    spk_hip_destroy(h);
    return rc;
  }
  {
    // LDS a workgroup may take, less room for the static arrays of the resident
    // and the tile kernel
    int lds = 0, optin = 0;
    (void)hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, h->device);
    (void)hipDeviceGetAttribute(&optin, hipDeviceAttributeSharedMemPerBlockOptin, h->device);
    const int most = std::max(lds, optin);
    h->max_lds = most > 2048 ? (size_t)most - 2048 : 0;
  }
  if (hipMalloc(&h->spin, (size_t)h->slots * spin_bytes(h->stype)) != hipSuccess ||
      hipMalloc(&h->seed, (size_t)h->slots * sizeof(int32_t)) != hipSuccess ||
      hipMalloc(&h->stage, (size_t)h->N * sizeof(int32_t)) != hipSuccess) {
    spk_hip_destroy(h);
    return set_error(SPK_HIP_ENOMEM, "device allocation of %lld sites failed", (long long)h->N);
  }
  // accumulator rows and their pinned host copy for calls of up to 1024
  // sweeps, so that such calls allocate nothing
  if ((rc = ensure_acc(h, kInitialAccRows)) || (rc = ensure_pinned(h, kInitialAccRows)) ||
      (rc = launch_fill_spins(h, 1))) {
    spk_hip_destroy(h);
    return rc;
  }
  hipLaunchKernelGGL(k_fill<int32_t>, dim3(grid_for(h->slots, 256)), dim3(256), 0, h->stream, h->seed, h->slots,
                     1);
  if ((rc = check_hip(hipStreamSynchronize(h->stream), "create sync"))) {
    spk_hip_destroy(h);
    return rc;
  }
  *out = h;
  return SPK_HIP_OK;
}

void spk_hip_destroy(spk_hip_lattice *h) {
  if (!h) return;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  drop_graphs(h);
  if (h->pinned) (void)hipHostFree(h->pinned);
  if (h->spin) (void)hipFree(h->spin);
  if (h->seed) (void)hipFree(h->seed);
  if (h->stage) (void)hipFree(h->stage);
  if (h->bits) (void)hipFree(h->bits);
  if (h->sseed) (void)hipFree(h->sseed);
  if (h->bits2) (void)hipFree(h->bits2);
  if (h->sseed2) (void)hipFree(h->sseed2);
  if (h->spin2) (void)hipFree(h->spin2);
  if (h->seed2) (void)hipFree(h->seed2);
  if (h->acc) (void)hipFree(h->acc);
  if (h->pinned_state) (void)hipHostFree(h->pinned_state);
  if (h->ev0) (void)hipEventDestroy(h->ev0);
  if (h->ev1) (void)hipEventDestroy(h->ev1);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

int spk_hip_set_temperature(spk_hip_lattice *h, double temperature) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  Rule r;
  int rc = make_rule(h->d.app, h->d.nspins, h->d.lattice, temperature, &r);
  if (rc) return rc;
  h->rule = r;
  h->d.temperature = temperature;
  drop_graphs(h);   // thresholds are kernel arguments of the captured launches
  return SPK_HIP_OK;
}

int spk_hip_upload(spk_hip_lattice *h, const int32_t *spin, const int32_t *seed) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  const size_t bytes = (size_t)h->N * sizeof(int32_t);
  int rc;
  if ((rc = bits_leave(h))) return rc;   // the planes hold the state: back to bytes first
  const int qmax = app_qmax(h->d.app, h->d.nspins);
  if (spin) {
    if ((rc = check_hip(hipMemcpyAsync(h->stage, spin, bytes, hipMemcpyHostToDevice, h->stream), "upload")))
      return rc;
    int64_t nbad = 0;
    if ((rc = validate_on_device(h, h->stage, 1, qmax, &nbad))) return rc;
    if (nbad) return set_error(SPK_HIP_EVALUE, "One or more sites have invalid values (%lld)", (long long)nbad);
    with_type(h->stype, [&]<typename T>() {
      hipLaunchKernelGGL((k_to_blocked<T>), dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->stage,
                         static_cast<T *>(h->spin), h->g);
    });
    if ((rc = check_hip(hipGetLastError(), "layout kernel"))) return rc;
    h->energy_valid = false;
  }
  if (seed) {
    if ((rc = check_hip(hipMemcpyAsync(h->stage, seed, bytes, hipMemcpyHostToDevice, h->stream), "upload")))
      return rc;
    int64_t nbad = 0;
    if ((rc = validate_on_device(h, h->stage, 1, kIM - 1, &nbad))) return rc;
    if (nbad) return set_error(SPK_HIP_EVALUE, "%lld seeds outside [1, 2^31-2]", (long long)nbad);
    hipLaunchKernelGGL(k_to_blocked<int32_t>, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->stage,
                       h->seed, h->g);
    if ((rc = check_hip(hipGetLastError(), "layout kernel"))) return rc;
  }
  return check_hip(hipStreamSynchronize(h->stream), "upload sync");
}

int spk_hip_download(spk_hip_lattice *h, int32_t *spin, int32_t *seed) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  const size_t bytes = (size_t)h->N * sizeof(int32_t);
  int rc;
  if ((rc = bits_leave(h))) return rc;
  if (!spin && !seed) return SPK_HIP_OK;
  // small lattices: one kernel writes the arrays to host memory, and one wait
  // ends it.  As two kernels, two copies and two waits, and so: 64^2 30.8 and
  // 13.9 us, 128^2 45.5 and 17.4, 40^3 52.5 and 32.0; from 50^3 on the copy out
  // of that memory takes what is saved.
  if (h->N <= kHostStateSites && ensure_pinned_state(h)) {
    with_type(h->stype, [&]<typename T>() {
      hipLaunchKernelGGL((k_state_natural<T>), dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream,
                         spin ? static_cast<const T *>(h->spin) : nullptr, seed ? h->seed : nullptr, h->pinned_state,
                         h->g);
    });
    if ((rc = check_hip(hipGetLastError(), "layout kernel")) ||
        (rc = check_hip(hipStreamSynchronize(h->stream), "download sync")))
      return rc;
    if (spin) std::memcpy(spin, h->pinned_state, bytes);
    if (seed) std::memcpy(seed, h->pinned_state + h->N, bytes);
    return SPK_HIP_OK;
  }
  // the second kernel writes the staging array after the first copy has read
  // it (stream order)
  if (spin) {
    with_type(h->stype, [&]<typename T>() {
      hipLaunchKernelGGL((k_to_natural<T>), dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream,
                         static_cast<const T *>(h->spin), h->stage, h->g);
    });
    if ((rc = check_hip(hipGetLastError(), "layout kernel")) ||
        (rc = check_hip(hipMemcpyAsync(spin, h->stage, bytes, hipMemcpyDeviceToHost, h->stream), "download")))
      return rc;
  }
  if (seed) {
    hipLaunchKernelGGL(k_to_natural<int32_t>, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->seed,
                       h->stage, h->g);
    if ((rc = check_hip(hipGetLastError(), "layout kernel")) ||
        (rc = check_hip(hipMemcpyAsync(seed, h->stage, bytes, hipMemcpyDeviceToHost, h->stream), "download")))
      return rc;
  }
  return check_hip(hipStreamSynchronize(h->stream), "download sync");
}

int spk_hip_set_range(spk_hip_lattice *h, int seed0, int lo, int hi) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (hi < lo) return set_error(SPK_HIP_EINVAL, "set range: hi < lo");
  if (seed0 < 1 || seed0 >= kIM) return set_error(SPK_HIP_EINVAL, "set range: seed0 outside [1, 2^31-2]");
  const int qmax = app_qmax(h->d.app, h->d.nspins);
  if (lo < 1 || hi > qmax)
    return set_error(SPK_HIP_EVALUE, "One or more sites have invalid values (set range %d %d, Q = %d)", lo, hi,
                     qmax);
  int rc = bits_leave(h);   // the seeds may live on the planes
  if (rc) return rc;
  const PowTable pw = park_powers();
  with_type(h->stype, [&]<typename T>() {
    hipLaunchKernelGGL((k_set_range<T>), dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream,
                       static_cast<T *>(h->spin), h->g, seed0, lo, hi - lo + 1, pw);
  });
  rc = check_hip(hipGetLastError(), "set_range launch");
  if (rc) return rc;
  h->energy_valid = false;
  return check_hip(hipStreamSynchronize(h->stream), "set_range sync");
}

int spk_hip_set_value(spk_hip_lattice *h, int value) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  const int qmax = app_qmax(h->d.app, h->d.nspins);
  if (value < 1 || value > qmax)
    return set_error(SPK_HIP_EVALUE, "One or more sites have invalid values (set value %d, Q = %d)", value, qmax);
  int rc;
  if ((rc = bits_leave(h)) || (rc = launch_fill_spins(h, value))) return rc;
  h->energy_valid = false;
  return check_hip(hipStreamSynchronize(h->stream), "set_value sync");
}

int spk_hip_init_seeds(spk_hip_lattice *h, double rseed) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (!(rseed >= 0.0 && rseed < 1.0)) return set_error(SPK_HIP_EINVAL, "init_seeds: rseed outside [0,1)");
  int rc = bits_leave(h);   // the spins may live on the planes
  if (rc) return rc;
  const double xbase = rseed * (double)kIM;
  const uint32_t a100 = park_warmup100();
  hipLaunchKernelGGL(k_init_seeds, dim3(grid_for(h->N, 256)), dim3(256), 0, h->stream, h->seed, h->g, xbase,
                     a100);
  rc = check_hip(hipGetLastError(), "init_seeds launch");
  if (rc) return rc;
  return check_hip(hipStreamSynchronize(h->stream), "init_seeds sync");
}

int spk_hip_sweeps(spk_hip_lattice *h, int nsweeps, int64_t *naccept_total, int64_t *naccept_per_sweep,
                   double *energy_per_sweep) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (nsweeps < 0) return set_error(SPK_HIP_EINVAL, "nsweeps < 0");
  if (nsweeps == 0) return SPK_HIP_OK;
  int rc;
  int64_t e0 = 0;
  if (energy_per_sweep) {
    if (h->energy_valid) e0 = h->energy;
    else if ((rc = compute_energy(h, &e0))) return rc;
  }
  int64_t nlaunch = 0;
  if (const size_t lds = resident_call(h, nsweeps)) {
    if ((rc = bits_leave(h)) || (rc = ensure_pinned(h, nsweeps)) || (rc = run_resident(h, nsweeps, lds, &nlaunch)))
      return rc;
    return finish_sweeps(h, nsweeps, nlaunch, e0, naccept_total, naccept_per_sweep, energy_per_sweep);
  }
  // (on the bit planes the state stays there)
  Route rt;
  if ((rc = enter_route(h, nsweeps, &rt)) || (rc = ensure_pinned(h, nsweeps))) return rc;
  // rows [0, n) cleared
  auto clear = [&](int n) {
    const int64_t words = (int64_t)n * kAccRow;
    hipLaunchKernelGGL(k_zero_u64, dim3(grid_for(words, 256)), dim3(256), 0, h->stream, h->acc, words);
    return check_hip(hipGetLastError(), "zero launch");
  };
  if (replayed(h, nsweeps, rt)) {
    // graph replays (graph_pieces); each piece's rows are folded into the
    // pinned rows [done, done + n) before the next piece clears them
    const std::vector<int> pieces = graph_pieces(h->chunk, nsweeps);
    if ((rc = ensure_acc(h, pieces[0]))) return rc;
    std::vector<hipGraphExec_t> execs(pieces.size());
    for (size_t k = 0; k < pieces.size(); k++)
      if ((rc = piece_graph(h, pieces[k], rt, &execs[k]))) return rc;
    if ((rc = check_hip(hipEventRecord(h->ev0, h->stream), "event"))) return rc;
    int done = 0;
    for (size_t k = 0; k < pieces.size(); k++) {
      if ((rc = check_hip(hipGraphLaunch(execs[k], h->stream), "graph launch")) ||
          (rc = launch_fold(h, h->acc, pieces[k], h->pinned + (size_t)done * 2)))
        return rc;
      done += pieces[k];
    }
    for (int n : pieces) nlaunch += sweep_launches(h, n, rt);
  } else if (rt == kRouteTile) {
    // boxes: from the host (launch_tiles), in pieces of kInitialAccRows sweeps
    if ((rc = ensure_acc(h, std::min(nsweeps, kInitialAccRows))) ||
        (rc = check_hip(hipEventRecord(h->ev0, h->stream), "event")))
      return rc;
    for (int done = 0; done < nsweeps;) {
      const int n = std::min(nsweeps - done, kInitialAccRows);
      if ((rc = clear(n)) || (rc = launch_tiles(h, n, h->acc, &nlaunch)) ||
          (rc = launch_fold(h, h->acc, n, h->pinned + (size_t)done * 2)))
        return rc;
      done += n;
    }
  } else {
    // every launch from the host: rows [0, nsweeps)
    if ((rc = ensure_acc(h, nsweeps)) || (rc = check_hip(hipEventRecord(h->ev0, h->stream), "event")) ||
        (rc = clear(nsweeps)) || (rc = launch_sweeps(h, nsweeps, h->acc, &nlaunch)) ||
        (rc = launch_fold(h, h->acc, nsweeps, h->pinned)))
      return rc;
  }
  if ((rc = check_hip(hipEventRecord(h->ev1, h->stream), "event"))) return rc;
  return finish_sweeps(h, nsweeps, nlaunch, e0, naccept_total, naccept_per_sweep, energy_per_sweep);
}

int spk_hip_sweeps_noalloc(spk_hip_lattice *h, int nsweeps, unsigned long long *rows) {
  if (!h || !rows) return set_error(SPK_HIP_EINVAL, "null argument");
  if (nsweeps < 0 || nsweeps > kNoAllocSweeps)
    return set_error(SPK_HIP_EINVAL, "nsweeps %d outside [0, %d] for sweeps without allocation", nsweeps,
                     kNoAllocSweeps);
  if (nsweeps == 0) return SPK_HIP_OK;
  unsigned long long *acc = g_scratch[h->device];   // looked up when the handle was created
  if (!acc) return set_error(SPK_HIP_ESTATE, "no scratch rows on device %d", h->device);
  // the state in the byte layout (an unpack when the planes hold it: kernels
  // only, into buffers that exist), then per-colour launches on the stream
  int rc = bits_leave(h);
  if (rc) return rc;
  const int64_t words = (int64_t)nsweeps * kAccRow;
  hipLaunchKernelGGL(k_zero_u64, dim3(grid_for(words, 256)), dim3(256), 0, h->stream, acc, words);
  int64_t nlaunch = 0;
  if ((rc = check_hip(hipGetLastError(), "zero launch")) || (rc = launch_sweeps(h, nsweeps, acc, &nlaunch)) ||
      (rc = launch_fold(h, acc, nsweeps, rows)))
    return rc;
  h->energy_valid = false;   // the energy changed on the device only
  return SPK_HIP_OK;
}

int spk_hip_prepare(spk_hip_lattice *h, int nsweeps) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (nsweeps < 0) return set_error(SPK_HIP_EINVAL, "nsweeps < 0");
  if (nsweeps == 0 || resident_call(h, nsweeps)) return SPK_HIP_OK;
  int rc;
  Route rt;
  if ((rc = enter_route(h, nsweeps, &rt)) || (rc = ensure_pinned(h, nsweeps))) return rc;
  if (replayed(h, nsweeps, rt)) {
    const std::vector<int> pieces = graph_pieces(h->chunk, nsweeps);
    if ((rc = ensure_acc(h, pieces[0]))) return rc;
    for (int n : pieces) {
      hipGraphExec_t exec;
      if ((rc = piece_graph(h, n, rt, &exec))) return rc;
    }
  } else if ((rc = ensure_acc(h, rt == kRouteTile ? std::min(nsweeps, kInitialAccRows) : nsweeps))) {
    return rc;
  }
  return check_hip(hipStreamSynchronize(h->stream), "prepare sync");
}

int spk_hip_energy(spk_hip_lattice *h, double *energy) {
  if (!h || !energy) return set_error(SPK_HIP_EINVAL, "null argument");
  int64_t e;
  int rc = compute_energy(h, &e);
  if (rc) return rc;
  *energy = (double)e;
  return SPK_HIP_OK;
}

int spk_hip_checksum(spk_hip_lattice *h, uint64_t *sum) {
  if (!h || !sum) return set_error(SPK_HIP_EINVAL, "null argument");
  int rc;
  if ((rc = bits_leave(h)) || (rc = ensure_acc(h, 1))) return rc;
  if ((rc = check_hip(hipMemsetAsync(h->acc, 0, sizeof(unsigned long long), h->stream), "memset"))) return rc;
  with_type(h->stype, [&]<typename T>() {
    launch_checksum<T>(h->stream, h->spin, h->seed, h->g, h->acc);
  });
  if ((rc = check_hip(hipGetLastError(), "checksum launch"))) return rc;
  if ((rc = check_hip(hipMemcpyAsync(h->pinned, h->acc, sizeof(*h->pinned), hipMemcpyDeviceToHost, h->stream),
                      "readback")) ||
      (rc = check_hip(hipStreamSynchronize(h->stream), "sync")))
    return rc;
  *sum = h->pinned[0];
  return SPK_HIP_OK;
}

int spk_hip_sync(spk_hip_lattice *h) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  return check_hip(hipStreamSynchronize(h->stream), "sync");
}

int spk_hip_set_launch(spk_hip_lattice *h, int block) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (block < 64 || block > 1024 || (block & (block - 1)))
    return set_error(SPK_HIP_EINVAL, "block must be a power of two in [64, 1024]");
  h->block = block;
  const int rc = bits_leave(h);
  if (rc) return rc;
  h->block_set = true;   // the per-colour kernel, with this workgroup
  h->tile_known = false;
  drop_graphs(h);
  return SPK_HIP_OK;
}

int spk_hip_set_resident(spk_hip_lattice *h, int enable) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  h->resident = enable ? 1 : 0;
  h->resident_set = enable != 0;
  h->tile_known = false;
  drop_graphs(h);
  return SPK_HIP_OK;
}

int spk_hip_set_bitplanes(spk_hip_lattice *h, int enable) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (enable != 0 && enable != 1 && enable != 8 && enable != 16 && enable != 32)
    return set_error(SPK_HIP_EINVAL, "bit planes: 0 (off), 1 (on), or 8, 16, 32 sites per thread");
  const int rc = bits_leave(h);   // the plane layout depends on the sites per thread
  if (rc) return rc;
  h->bitplanes = enable;
  h->tile_known = false;
  drop_graphs(h);   // captured launches name one kernel or the other
  return SPK_HIP_OK;
}

int spk_hip_set_graph(spk_hip_lattice *h, int chunk_sweeps) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (chunk_sweeps < 0 || chunk_sweeps > kMaxChunk)
    return set_error(SPK_HIP_EINVAL, "chunk_sweeps must be in [0, %d]", kMaxChunk);
  drop_graphs(h);
  h->chunk = chunk_sweeps;
  return SPK_HIP_OK;
}

int spk_hip_last_timing(spk_hip_lattice *h, double *ms, int64_t *nlaunch) {
  if (!h) return set_error(SPK_HIP_EINVAL, "null handle");
  if (ms) *ms = h->last_ms;
  if (nlaunch) *nlaunch = h->last_nlaunch;
  return SPK_HIP_OK;
}

}  // extern "C"
