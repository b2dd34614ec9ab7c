// spk_neigh.h -- potts/neigh and potts/neighonly on sq/8n and sc/26n, four
// sites a thread: the packed form of variant_event (spk_device.h).
//
// The rules compare every pair of a site's neighbours (325 on sc/26n) to find
// its distinct unlike values in order of first appearance.  Here the four
// sites are halfwords of two words, and a value stands as its XOR with the site's
// old spin, D: "unlike" is D != 0, the new spin is old ^ D.  For values of 15
// bits, bit 15 of (D_i ^ D_m) + 0x7fff says that the two differ and nothing
// carries into the other half; that is one instruction for two sites, and a
// three-operand AND joins two of them: 0.75 of an instruction a comparison and
// site, where the one-site form has a compare and a scalar AND each.
#pragma once

#include "spk_bits.h"
#include "spk_device.h"
#include "spk_slice.h"

namespace spk {

constexpr int kNeighMaxQ = 0x7fff;   // D of 15 bits

constexpr uint32_t kHalfMax = 0x7fff7fffu, kHalfTop = 0x80008000u;
constexpr uint32_t kAndNotAnd = truth3([](int x, int y, int z) { return x & (1 - y) & z; });

typedef uint16_t HalfPair __attribute__((ext_vector_type(2)));
__host__ __device__ __forceinline__ uint32_t half_tops(uint32_t x) {   // bit 15 of each half, as 0 or 1
  return __builtin_bit_cast(uint32_t, __builtin_bit_cast(HalfPair, x) >> (uint16_t)15);
}
__host__ __device__ __forceinline__ uint32_t half_mad(uint32_t x, uint32_t y, uint32_t z) {
  return __builtin_bit_cast(uint32_t, (HalfPair)(__builtin_bit_cast(HalfPair, x) * __builtin_bit_cast(HalfPair, y) +
                                                 __builtin_bit_cast(HalfPair, z)));
}
// bit 15 of each half: the halves differ (bits 0..14 of each; bit 15 is 0 in both)
__host__ __device__ __forceinline__ uint32_t half_differ(uint32_t x, uint32_t y) { return (x ^ y) + kHalfMax; }

// four sites as halves
struct Halves {
  uint32_t w[2];
};
template <typename T>
__host__ __device__ __forceinline__ Halves halves_of(const Lanes<T> &l) {
  if constexpr (sizeof(T) == 1) return Halves{{byte_perm(0u, l.w[0], 0x04010400u), byte_perm(0u, l.w[0], 0x04030402u)}};
  else return Halves{{l.w[0], l.w[1]}};
}

// The strict events of sites a0..a0+3 of row (b, e) of colour c.  XD: the
// colour's x parity.
template <int LAT, typename T, int APP, typename I, int XD>
__host__ __device__ __forceinline__ Counts neigh_pack(T *__restrict__ spin, int32_t *__restrict__ seed, const Geom &g,
                                                      const Rule &r, const int *thr, int c, int a0, int b, int e) {
  static_assert((LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N) && sizeof(T) <= 2);
  static_assert(APP == SPK_HIP_POTTS_NEIGH || APP == SPK_HIP_POTTS_NEIGHONLY);
  constexpr int NN = NeighCount<LAT>::value;
  const PackLoad<LAT, T, I> ld = pack_load<LAT, T, I, XD>(spin, seed, g, c, a0, b, e);
  const bool ragged = (g.hx & 3) != 0;
  const Halves old = halves_of<T>(ld.old);

  // D in the reference's order (Shell): the row segment as loaded holds the
  // x-neighbours on one side, shifted those on the other
  uint32_t D[NN][2];
#pragma unroll
  for (int m = 0; m < NN; m++) {
    int dx = 0, dy = 0, dz = 0;
    Shell<LAT>::offset(m, dx, dy, dz);
    const int row = LAT == SPK_HIP_SQ_8N ? dy + 1 : 3 * (dz + 1) + dy + 1;
    const int mid = LAT == SPK_HIP_SQ_8N ? 1 : 4;
    const Lanes<T> x = dx == 0                 ? ld.raw.pk[row < mid ? row : row - 1]
                       : (dx > 0) == (XD == 0) ? ld.raw.seg[row]
                                               : ld.beside(row, XD, ragged);
    const Halves h = halves_of<T>(x);
    D[m][0] = h.w[0] ^ old.w[0];
    D[m][1] = h.w[1] ^ old.w[1];
  }
  // unlike neighbours; then, from the last neighbour down, bit 15 of D_m: it
  // is the first of its value and unlike (those before it are unmarked yet)
  uint32_t ei[2] = {0, 0}, ef[2] = {0, 0}, n[2] = {0, 0};
#pragma unroll
  for (int h = 0; h < 2; h++) {
#pragma unroll
    for (int m = 0; m < NN; m += 2) add_ne_halves2(ei[h], D[m][h], D[m + 1][h]);
#pragma unroll
    for (int m = NN - 1; m >= 0; m--) {
      uint32_t f = D[m][h] + kHalfMax;
#pragma unroll
      for (int i = 0; i + 1 < m; i += 2)
        f = bop3<kAnd3>(f, half_differ(D[i][h], D[m][h]), half_differ(D[i + 1][h], D[m][h]));
      if (m & 1) f &= half_differ(D[m - 1][h], D[m][h]);
      D[m][h] = bop3<kOrAnd>(f, kHalfTop, D[m][h]);
    }
    if constexpr (APP == SPK_HIP_POTTS_NEIGHONLY)
#pragma unroll
      for (int m = 0; m < NN; m++) n[h] += half_tops(D[m][h]);
  }
  // which of them the first draw takes: floor(count * s/M) by integers
  // (slice_propose), as the doubles give it; the first with no event, or past the last, takes none
  int32_t s[4];
  uint32_t rank[4];
#pragma unroll
  for (int v = 0; v < 4; v++) {
    s[v] = (int32_t)ld.sd.w[v];
    uint32_t count = NN;
    if constexpr (APP == SPK_HIP_POTTS_NEIGHONLY) count = (n[v >> 1] >> (16 * (v & 1))) & 0xffffu;
    const int32_t u = pm_step(s[v]);
    s[v] = count ? u : s[v];
    rank[v] = slice_propose(2u * count, (uint32_t)u);
  }
  // P: D of the proposal, 0 if there is none
  uint32_t P[2];
#pragma unroll
  for (int h = 0; h < 2; h++) {
    const uint32_t want = rank[2 * h] | rank[2 * h + 1] << 16;
    uint32_t before = 0, d = 0;
#pragma unroll
    for (int m = 0; m < NN; m++) {
      const uint32_t sel = bop3<kAndNotAnd>(D[m][h], half_differ(before, want), kHalfTop);
      d = half_mad(D[m][h], half_tops(sel), d);
      before += half_tops(D[m][h]);
    }
    P[h] = d & kHalfMax;
#pragma unroll
    for (int m = 0; m < NN; m += 2)
      add_ne_halves2(ef[h], bop3<kXorAnd>(D[m][h], P[h], kHalfMax), bop3<kXorAnd>(D[m + 1][h], P[h], kHalfMax));
  }
  Counts out{0, 0};
  Words<4> nsd;
  uint32_t change[2] = {0, 0};
#pragma unroll
  for (int v = 0; v < 4; v++) {
    const int sh = 16 * (v & 1);
    const int i = (int)((ei[v >> 1] >> sh) & 0xffffu), f = (int)((ef[v >> 1] >> sh) & 0xffffu);
    const uint32_t p = (P[v >> 1] >> sh) & 0xffffu;
    // (no proposal: ef == ei, so no second draw)
    const bool accept = metropolis_select(r, thr, i, f, s[v]);
    const bool changed = v < ld.k && accept && p != 0;
    if (changed) change[v >> 1] |= p << sh;
    nsd.w[v] = (uint32_t)s[v];
    out.nacc += changed;
    out.de += changed ? f - i : 0;
  }
  const I Mp = (I)g.Mp;
  *reinterpret_cast<Words<4> *>(elem<I>(elem<I>(seed, (I)c * Mp), ld.self)) = nsd;
  if (change[0] | change[1]) {
    Lanes<T> nsp = ld.old;
    if constexpr (sizeof(T) == 1) {
      nsp.w[0] ^= byte_perm(change[1], change[0], 0x06040200u);
    } else {
      nsp.w[0] ^= change[0];
      nsp.w[1] ^= change[1];
    }
    store_lanes<T, I>(elem<I>(spin, (I)c * Mp), ld.self, nsp);
  }
  return out;
}

}  // namespace spk
