// spk_slice.h -- bit-sliced colour passes of Potts (and two-state) lattices on
// sc/26n: the sweep path of large lattices there.
//
// The packed kernel (pack_count, spk_device.h) spends half its instructions
// comparing 26 neighbours with the old and the proposed spin, 1.25 for each
// comparison of a 16-bit value.  Here spins are held as bit planes: plane p of
// a row holds bit p of (spin - 1) of up to 32 consecutive sites a word, so
// "unlike" for 32 sites is one (x ^ own) | acc per plane, P/32 instructions a
// site and comparison (P = bits of Q-1: 0.44 at Q = 10^4), and carry-save
// adders turn the 52 flags of a site into ef - ei.  The draws and the accept
// test stay one site at a time, on seeds of 4 bytes a site as before.
//
// The two colours of a sub-grid row pair (c = 2m: even x, 2m+1: odd x) see
// the same eight neighbouring rows, none of which either of them changes, so
// one pass runs both: colour 2m first, then colour 2m+1, which takes the row's
// new even sites from the wavefront itself.  Each neighbour word is read once
// for both colours, a sweep is 4 launches instead of 8, and nothing is computed
// twice.
//
// Four lanes share a word: each compares two of the eight neighbouring rows,
// for all 32 sites and both colours, and draws and decides for eight of the
// sites; their partial counts meet by lane swaps.  One lane a word instead
// had 4 times fewer wavefronts (one a SIMD at 256^3), each a chain that
// nothing overlapped: 26.5 us a pass.  The four are 16 lanes apart, so the 16
// lanes that a load serves at once read consecutive words of one row.
//
// Layout (a shadow of the colour-blocked state, as the two-state planes of
// spk_bits.h are).  A row of hx sites is pw words of W = ceil(hx/pw) sites, the
// last word `last` of them (W balances the words: hx = 40 is 2 words of 20,
// not 32 + 8); bits at and above a word's width are zero.
//   plane p of colour c: words[((c*PG + p/4)*nw + row*pw + w)*4 + p%4], row = b +
//   hy*e, PG = ceil(P/4): four planes of a word are one 16-byte load
// A wavefront works on rw = 16/pw whole rows; lane 16q + k on sites 8q..8q+7 of
// word k % pw of its row k / pw.  The seeds of lane l of wavefront v are two
// groups of four,
//   c*seedc + ((v*2 + j)*64 + l)*4 + i: site 8q + 4j + i,
// so each 16-byte seed load of a wavefront covers 1 KiB of consecutive bytes.
#pragma once

#include "spk_bits.h"
#include "spk_device.h"

namespace spk {

constexpr int kSliceMaxPlanes = 20;
constexpr int kSliceMaxPw = 16;
// Proposals come from integers (slice_propose), exact up to this Q.
constexpr int kSliceMaxQ = 1 << kSliceMaxPlanes;

struct SliceGeom {
  int P, PG;         // planes, and groups of four of them
  int pw, W, last;   // words per row, sites per word, sites of the last word
  int rw;            // rows per wavefront
  int rows;          // hy*hz
  int waves;         // wavefronts per colour pair
  int nw;            // words per plane of a colour (rows*pw)
  int64_t seedc;     // seed slots per colour
  FastDiv fpw, fhy;  // division by pw, hy
};

__host__ __device__ inline SliceGeom slice_geom(const Geom &g, int q) {
  SliceGeom s;
  s.P = 1;
  while ((1ll << s.P) < q) s.P++;
  s.PG = (s.P + 3) / 4;
  s.pw = (g.hx + 31) / 32;
  s.W = (g.hx + s.pw - 1) / s.pw;
  s.last = g.hx - (s.pw - 1) * s.W;
  s.rw = s.pw <= kSliceMaxPw ? kSliceMaxPw / s.pw : 0;
  s.rows = g.hy * g.hz;
  s.waves = s.rw ? (s.rows + s.rw - 1) / s.rw : 0;
  s.nw = s.rows * s.pw;
  s.seedc = (int64_t)s.waves * 512;
  s.fpw = fastdiv_make((uint32_t)s.pw);
  s.fhy = fastdiv_make((uint32_t)g.hy);
  return s;
}

// Lattices the sliced pass can run: sc/26n, rows of at most 16 words, the
// planes and a colour's seeds within 31-bit byte offsets.
__host__ __device__ inline bool slice_fits(const Geom &g, int q) {
  if (g.lat != SPK_HIP_SC_26N || q < 2 || q > kSliceMaxQ || (g.hx + 31) / 32 > kSliceMaxPw) return false;
  const SliceGeom s = slice_geom(g, q);
  return s.rows < (1 << 24) && (int64_t)g.K * s.PG * s.rows * s.pw * 16 < (int64_t(1) << 31) &&
         s.seedc * 4 < (int64_t(1) << 31);
}

// f.template operator()<PG>() for a lattice's plane groups
template <typename F>
__host__ __device__ __forceinline__ void with_plane_groups(int pg, F &&f) {
  static_assert(kSliceMaxPlanes == 20, "1..5 groups");
  switch (pg) {
    case 1: f.template operator()<1>(); break;
    case 2: f.template operator()<2>(); break;
    case 3: f.template operator()<3>(); break;
    case 4: f.template operator()<4>(); break;
    default: f.template operator()<5>(); break;
  }
}

// ------------------------------------------------------------- conversions
// sites of word w
__host__ __device__ __forceinline__ int slice_width(const SliceGeom &s, int w) { return w == s.pw - 1 ? s.last : s.W; }

// lane l of wavefront v: its row and word; false past the last row
__host__ __device__ __forceinline__ bool slice_word(const SliceGeom &s, uint32_t v, uint32_t l, uint32_t &row,
                                                    uint32_t &w) {
  uint32_t r;
  fastdiv(s.fpw, l & 15u, r, w);
  row = v * (uint32_t)s.rw + r;
  return r < (uint32_t)s.rw && row < (uint32_t)s.rows;
}

// Word w of row `row` of colour c (t = row*pw + w): the spins into every
// plane, or back.
template <typename T>
__host__ __device__ __forceinline__ void slice_pack_word(const T *__restrict__ spin, const Geom &g, const SliceGeom &s,
                                                         int c, uint32_t t, uint32_t *__restrict__ planes) {
  uint32_t row, w;
  fastdiv(s.fpw, t, row, w);
  const T *src = spin + (int64_t)c * g.Mp + (int64_t)g.px * row + (int64_t)w * s.W;
  uint32_t out[kSliceMaxPlanes] = {};
  const int n = slice_width(s, (int)w);
  for (int i = 0; i < n; i++) {
    const uint32_t v = (uint32_t)src[i] - 1u;
#pragma unroll
    for (int p = 0; p < kSliceMaxPlanes; p++) out[p] |= ((v >> p) & 1u) << i;
  }
#pragma unroll
  for (int p = 0; p < kSliceMaxPlanes; p++)
    if (p < 4 * s.PG) planes[(((int64_t)c * s.PG + p / 4) * s.nw + t) * 4 + p % 4] = out[p];   // planes from P on are 0
}

template <typename T>
__host__ __device__ __forceinline__ void slice_unpack_word(const uint32_t *__restrict__ planes, const Geom &g,
                                                           const SliceGeom &s, int c, uint32_t t, T *__restrict__ spin) {
  uint32_t row, w;
  fastdiv(s.fpw, t, row, w);
  T *dst = spin + (int64_t)c * g.Mp + (int64_t)g.px * row + (int64_t)w * s.W;
  uint32_t in[kSliceMaxPlanes];
#pragma unroll
  for (int p = 0; p < kSliceMaxPlanes; p++) in[p] = p < s.P ? planes[(((int64_t)c * s.PG + p / 4) * s.nw + t) * 4 + p % 4] : 0u;
  const int n = slice_width(s, (int)w);
  for (int i = 0; i < n; i++) {
    uint32_t v = 0;
#pragma unroll
    for (int p = 0; p < kSliceMaxPlanes; p++) v |= ((in[p] >> i) & 1u) << p;
    dst[i] = (T)(v + 1u);
  }
}

// Seed group x (0 .. K*seedc/4 - 1) in the conversions' order: colour,
// wavefront, word, q, j with j fastest, so consecutive groups are consecutive
// 16-byte pieces of a row; unit is its place in the shadow.  Returns its real
// sites (0..4) and the canonical offset of the first.
__host__ __device__ __forceinline__ int slice_seed_group(const Geom &g, const SliceGeom &s, int64_t x, int64_t &unit,
                                                         int64_t &home) {
  const int64_t per = s.seedc / 4;
  const int c = (int)(x / per);
  const uint32_t r = (uint32_t)(x - (int64_t)c * per), j = r & 1u, q = (r >> 1) & 3u, v = r >> 7;
  const uint32_t l = 16u * q + ((r >> 3) & 15u);
  unit = (int64_t)c * per + ((int64_t)v * 2 + j) * 64 + l;
  uint32_t row, w, b, e;
  if (!slice_word(s, v, l, row, w)) return 0;
  const int first = (int)(8u * q + 4u * j);
  fastdiv(s.fhy, row, e, b);
  home = (int64_t)c * g.Mp + (int64_t)w * s.W + first + (int64_t)g.px * (b + (int64_t)g.hy * e);
  return min(4, max(0, slice_width(s, (int)w) - first));
}

// canonical seeds -> shadow group (padding slots hold 1), and back
__host__ __device__ __forceinline__ void slice_seeds_in(const int32_t *__restrict__ seed, const Geom &g,
                                                        const SliceGeom &s, int64_t x, int32_t *__restrict__ sseed) {
  int64_t unit, home = 0;
  const int n = slice_seed_group(g, s, x, unit, home);
  Words<4> o;
  if (n == 4 && (home & 3) == 0) {
    o = *reinterpret_cast<const Words<4> *>(seed + home);
  } else {
#pragma unroll
    for (int k = 0; k < 4; k++) o.w[k] = k < n ? (uint32_t)seed[home + k] : 1u;
  }
  reinterpret_cast<Words<4> *>(sseed)[unit] = o;
}

__host__ __device__ __forceinline__ void slice_seeds_out(const int32_t *__restrict__ sseed, const Geom &g,
                                                         const SliceGeom &s, int64_t x, int32_t *__restrict__ seed) {
  int64_t unit, home = 0;
  const int n = slice_seed_group(g, s, x, unit, home);
  if (n == 0) return;
  const Words<4> o = reinterpret_cast<const Words<4> *>(sseed)[unit];
  if (n == 4 && (home & 3) == 0) {
    *reinterpret_cast<Words<4> *>(seed + home) = o;
    return;
  }
#pragma unroll
  for (int k = 0; k < 4; k++)
    if (k < n) seed[home + k] = (int32_t)o.w[k];
}

// Spin of the site at (i, j, k), and the place of its seed in the shadow.
struct SliceSite {
  int c, i;          // colour, and site within its word
  uint32_t row, w;   // its word
};
__host__ __device__ __forceinline__ SliceSite slice_site(const Geom &g, const SliceGeom &s, int i, int j, int k) {
  const int a = i >> 1, w = a / s.W;
  return SliceSite{(i & 1) | (j & 1) << 1 | (k & 1) << 2, a - w * s.W, (uint32_t)((j >> 1) + g.hy * (k >> 1)),
                   (uint32_t)w};
}
__host__ __device__ __forceinline__ int32_t slice_spin_at(const uint32_t *__restrict__ planes, const SliceGeom &s,
                                                          const SliceSite &x) {
  const Words<4> *p = reinterpret_cast<const Words<4> *>(planes) + (int64_t)x.c * s.PG * s.nw + x.row * s.pw + x.w;
  uint32_t v = 0;
  for (int t = 0; t < s.PG; t++) {
    const Words<4> y = p[(int64_t)t * s.nw];
#pragma unroll
    for (int b = 0; b < 4; b++) v |= ((y.w[b] >> x.i) & 1u) << (4 * t + b);
  }
  return (int32_t)v + 1;
}
__host__ __device__ __forceinline__ int64_t slice_seed_slot(const SliceGeom &s, const SliceSite &x) {
  const uint32_t v = x.row / (uint32_t)s.rw, l = 16u * (uint32_t)(x.i >> 3) + (x.row - v * (uint32_t)s.rw) * s.pw + x.w;
  return (int64_t)x.c * s.seedc + (((int64_t)v * 2 + ((x.i >> 2) & 1)) * 64 + l) * 4 + (x.i & 3);
}

// -------------------------------------------------------------- primitives
// A seed group in and out past the caches (nothing reads it again in the
// pass): 46.4 to 43.7 us a sweep at 192^3, 53.7 to 51.3 at 256^3 with Q = 100.
__host__ __device__ __forceinline__ Words<4> slice_seeds_load(const Words<4> *p) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  const v4 x = __builtin_nontemporal_load(reinterpret_cast<const v4 *>(p));
  return Words<4>{{x[0], x[1], x[2], x[3]}};
#else
  return *p;
#endif
}
__host__ __device__ __forceinline__ void slice_seeds_store(Words<4> *p, const Words<4> &u) {
#ifdef __HIP_DEVICE_COMPILE__
  typedef uint32_t v4 __attribute__((ext_vector_type(4)));
  __builtin_nontemporal_store(v4{u.w[0], u.w[1], u.w[2], u.w[3]}, reinterpret_cast<v4 *>(p));
#else
  *p = u;
#endif
}

// prop - 1 of a Potts draw s: floor(Q * s/M), M = 2^31 - 1.  The reference
// takes (int)(Q * (AM*s)) in doubles (src/app_potts.cpp:119); Q*s is no
// multiple of the prime M, so its quotient is at least 1/M away from an
// integer, and the three roundings move it by less than 3.01 * 2^-53 * Q <
// 1/M for Q up to 2^20: the floors agree, and the clamp to Q never acts.
// With x = Q*s = h*2^31 + l = h*M + (h + l), the floor is h, plus one when h
// + l >= M.  For two states it is the Ising proposal (s >= 2^30) as well.
__host__ __device__ __forceinline__ uint32_t slice_propose(uint32_t q2, uint32_t s) {
  const uint64_t y = (uint64_t)s * q2;   // q2 = 2*Q: y's high word is h, its low word 2*l
  const uint32_t h = (uint32_t)(y >> 32), l = (uint32_t)y >> 1;
  return h + ((h + l + 1u) >> 31);
}

constexpr uint32_t kOrXor = truth3([](int x, int y, int z) { return (x ^ y) | z; });             // (x ^ y) | z
constexpr uint32_t kAndXnor = truth3([](int x, int y, int z) { return (1 - (x ^ y)) & z; });     // ~(x ^ y) & z
constexpr uint32_t kMaj3 = truth3([](int x, int y, int z) { return (x & y) | (x & z) | (y & z); });
constexpr uint32_t kXorAnd = truth3([](int x, int y, int z) { return (x ^ y) & z; });            // (x ^ y) & z

// 8x8 bit transpose of the 8 bytes hi:lo: bit k of byte j becomes bit j of
// byte k.
__host__ __device__ __forceinline__ void slice_transpose8(uint32_t &lo, uint32_t &hi) {
  auto step = [](uint32_t x, int n, uint32_t m) {   // swaps bit pairs n apart
    const uint32_t t = bop3<kXorAnd>(x, x >> n, m);
    return bop3<kXor3>(x, t, t << n);
  };
  lo = step(step(lo, 7, 0x00aa00aau), 14, 0x0000ccccu);
  hi = step(step(hi, 7, 0x00aa00aau), 14, 0x0000ccccu);
  const uint32_t a = lo >> 4, b = hi << 4;
  lo = bop3<kSel>(0x0f0f0f0fu, lo, b);
  hi = bop3<kSel>(0x0f0f0f0fu, a, hi);
}

// byte `s` of 4 values in one word
__host__ __device__ __forceinline__ uint32_t slice_bytes(int s, uint32_t v0, uint32_t v1, uint32_t v2, uint32_t v3) {
  const uint32_t sel = 0x00000400u + 0x0101u * (uint32_t)s;   // byte s of lo, byte s of hi
  const uint32_t a = byte_perm(v1, v0, sel), b = byte_perm(v3, v2, sel);
  return byte_perm(b, a, 0x05040100u);
}

// per site: how many of N words have its bit set, as 5 bit planes (N <= 31)
template <int N>
__host__ __device__ __forceinline__ void slice_count(const uint32_t (&x)[N], uint32_t (&cnt)[5]) {
  uint32_t lv[N];
  int n = N;
#pragma unroll
  for (int i = 0; i < N; i++) lv[i] = x[i];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    uint32_t up[N];
    int m = 0;
#pragma unroll
    for (int guard = 0; guard < N; guard++) {
      if (n <= 2) break;   // full adders until at most two words of this weight are left
      const uint32_t a = lv[n - 1], b = lv[n - 2], c = lv[n - 3];
      lv[n - 3] = bop3<kXor3>(a, b, c);
      up[m++] = bop3<kMaj3>(a, b, c);
      n -= 2;
    }
    if (n == 2) {
      up[m++] = lv[0] & lv[1];
      lv[0] ^= lv[1];
      n = 1;
    }
    cnt[k] = n ? lv[0] : 0u;
#pragma unroll
    for (int i = 0; i < N; i++)
      if (i < m) lv[i] = up[i];
    n = m;
  }
}

// The word of the sites one to the left (site i takes i-1; site 0 the last of
// the previous word) and one to the right.  FULL: words of 32 sites.  Bits at
// and above the width are junk for the right one.
template <bool FULL>
__host__ __device__ __forceinline__ uint32_t slice_left(uint32_t x, uint32_t xprev, int wprev) {
  if constexpr (FULL) return (x << 1) | (xprev >> 31);
  return (x << 1) | (xprev >> (wprev - 1));
}
template <bool FULL>
__host__ __device__ __forceinline__ uint32_t slice_right(uint32_t x, uint32_t xnext, int width) {
  if constexpr (FULL) return (x >> 1) | (xnext << 31);
  return (x >> 1) | (xnext << (width - 1));
}

// ------------------------------------------------------------------ a lane
struct SliceLane {
  uint32_t q;          // which eight sites of its word
  uint32_t own;        // byte offset of its word's first four planes in colour 2m, from those of colour 0
  uint32_t row[2];     // the same of the two neighbouring rows it compares (even-x colour)
  uint32_t prev;       // lane holding the row's previous word (periodic), same q
  uint32_t next;
  int width, wprev;    // sites of the word, and of the previous one
  uint32_t mask;       // its real sites among its eight; 0 on an idle lane
};

// The eight rows around (b, e) of pair m = 2*pk + pj, two a lane: q 0 the two
// in the same z, q 1..3 six of the other z parity.
__host__ __device__ __forceinline__ SliceLane slice_lane(const Geom &g, const SliceGeom &s, int m, uint32_t v,
                                                         uint32_t l) {
  SliceLane t;
  uint32_t row, w, e, b;
  const bool on = slice_word(s, v, l, row, w);
  if (!on) row = (uint32_t)s.rows - 1u;   // a row that exists; nothing is stored
  fastdiv(s.fhy, row, e, b);
  t.q = l >> 4;
  const int pj = m & 1, pk = m >> 1;
  const uint32_t yo = (uint32_t)(pj ? wrap_inc((int)b, g.hy) : wrap_dec((int)b, g.hy));
  const uint32_t zo = (uint32_t)(pk ? wrap_inc((int)e, g.hz) : wrap_dec((int)e, g.hz));
  // (rows and pw are below 2^24: 24-bit products)
  const RowOffset<uint32_t> hy((uint32_t)g.hy), pw((uint32_t)s.pw);
  const uint32_t pair_words = 2u * (uint32_t)s.PG * (uint32_t)s.nw;
  auto at = [&](int pair, uint32_t y, uint32_t z) {
    return ((uint32_t)pair * pair_words + pw * (y + hy * z) + w) * 16u;
  };
  t.own = at(m, b, e);
  // q: 0 (y, z), (yo, z); 1 (own y) at e and zo; 2, 3 (y, yo) at e, at zo
  t.row[0] = t.q == 0 ? at(m ^ 1, b, e) : t.q == 1 ? at(m ^ 2, b, e) : at(m ^ 3, b, t.q == 2 ? e : zo);
  t.row[1] = t.q == 0 ? at(m ^ 1, yo, e) : t.q == 1 ? at(m ^ 2, b, zo) : at(m ^ 3, yo, t.q == 2 ? e : zo);
  // (lanes past the last whole row look at themselves)
  const bool whole = (l & 15u) < (uint32_t)(s.rw * s.pw);
  t.prev = !whole ? l : w == 0 ? l + (uint32_t)s.pw - 1u : l - 1u;
  t.next = !whole ? l : w + 1 == (uint32_t)s.pw ? l - w : l + 1u;
  t.width = slice_width(s, (int)w);
  t.wprev = slice_width(s, w == 0 ? s.pw - 1 : (int)w - 1);
  const int n = t.width - (int)(8u * t.q);
  t.mask = !on || n <= 0 ? 0u : n >= 8 ? 0xffu : (1u << n) - 1u;
  return t;
}

// 16-byte seed group j of lane l of wavefront v
__host__ __device__ __forceinline__ uint32_t slice_seed_at(uint32_t v, int j, uint32_t l) {
  return ((v * 2u + (uint32_t)j) * 64u + l) * 4u;
}

// The eight seeds of a lane, advanced by their first draws, and the
// proposals' plane bytes: byte p % 4 of bytes[p / 4] holds plane p of the
// lane's sites.
template <int PG>
__host__ __device__ __forceinline__ void slice_draws(uint32_t q2, Words<4> (&u)[2], uint32_t (&bytes)[6]) {
  uint32_t v[8];
#pragma unroll
  for (int i = 0; i < 8; i++) {
    uint32_t &x = u[i >> 2].w[i & 3];
    x = (uint32_t)pm_step((int32_t)x);
    v[i] = slice_propose(q2, x);
  }
#pragma unroll
  for (int b = 0; b < 3; b++) {
    if (2 * b >= PG) continue;
    uint32_t lo = slice_bytes(b, v[0], v[1], v[2], v[3]), hi = slice_bytes(b, v[4], v[5], v[6], v[7]);
    slice_transpose8(lo, hi);
    bytes[2 * b] = lo;
    bytes[2 * b + 1] = hi;
  }
}

// Unlike / like words of one colour against one proposal: like (to the spin)
// starts at ~0, differ (from the proposal) at 0.
struct SliceFlags {
  uint32_t like, differ;
};
__host__ __device__ __forceinline__ void slice_compare(SliceFlags &f, uint32_t x, uint32_t own, uint32_t prop) {
  f.like = bop3<kAndXnor>(x, own, f.like);
  f.differ = bop3<kOrXor>(x, prop, f.differ);
}

// What a lane gathers for a colour: three flags words of each of its rows,
// and (after the word's lanes have joined them) two of the own row and the sites
// whose proposal is not their spin.
struct SliceColour {
  SliceFlags row[6], own[2];
  uint32_t moves;
};
__host__ __device__ __forceinline__ void slice_clear(SliceColour &c) {
#pragma unroll
  for (int k = 0; k < 6; k++) c.row[k] = SliceFlags{0xffffffffu, 0u};
  c.own[0] = c.own[1] = SliceFlags{0xffffffffu, 0u};
  c.moves = 0;
}

// One plane of the lane's two rows (even-x words e, odd-x o) against both
// colours of the own row (own0, own1) and their proposals.  prev[r]: the odd-x
// word of row r at lane t.prev; next[r]: the even-x word at t.next.
template <bool FULL>
__host__ __device__ __forceinline__ void slice_rows(const SliceLane &t, const uint32_t (&e)[2], const uint32_t (&o)[2],
                                                    const uint32_t (&prev)[2], const uint32_t (&next)[2],
                                                    uint32_t own0, uint32_t own1, uint32_t pr0, uint32_t pr1,
                                                    SliceColour &c0, SliceColour &c1) {
#pragma unroll
  for (int r = 0; r < 2; r++) {
    slice_compare(c0.row[3 * r], e[r], own0, pr0);
    slice_compare(c0.row[3 * r + 1], o[r], own0, pr0);
    slice_compare(c1.row[3 * r], o[r], own1, pr1);
    slice_compare(c1.row[3 * r + 1], e[r], own1, pr1);
    slice_compare(c0.row[3 * r + 2], slice_left<FULL>(o[r], prev[r], t.wprev), own0, pr0);
    slice_compare(c1.row[3 * r + 2], slice_right<FULL>(e[r], next[r], t.width), own1, pr1);
  }
}

// One plane of the own row for colour 2m: its odd-x neighbours.
template <bool FULL>
__host__ __device__ __forceinline__ void slice_own_first(const SliceLane &t, uint32_t e, uint32_t o, uint32_t oprev,
                                                         uint32_t pr0, SliceColour &c0) {
  slice_compare(c0.own[0], o, e, pr0);
  slice_compare(c0.own[1], slice_left<FULL>(o, oprev, t.wprev), e, pr0);
  c0.moves = bop3<kOrXor>(e, pr0, c0.moves);
}
// And for colour 2m+1, e being the new even-x words.
template <bool FULL>
__host__ __device__ __forceinline__ void slice_own_second(const SliceLane &t, uint32_t e, uint32_t enext, uint32_t o,
                                                          uint32_t pr1, SliceColour &c1) {
  slice_compare(c1.own[0], e, o, pr1);
  slice_compare(c1.own[1], slice_right<FULL>(e, enext, t.width), o, pr1);
  c1.moves = bop3<kOrXor>(o, pr1, c1.moves);
}

// The lane's part of ef - ei + 26 = sum of (differs from the proposal) + (like
// the spin) over the neighbours, as 5 planes; the own row counts on q = 0.
__host__ __device__ __forceinline__ void slice_part(const SliceLane &t, const SliceColour &c, uint32_t (&d)[5]) {
  const uint32_t mine = t.q == 0 ? 0xffffffffu : 0u;
  uint32_t x[16];
#pragma unroll
  for (int k = 0; k < 6; k++) x[2 * k] = c.row[k].like, x[2 * k + 1] = c.row[k].differ;
#pragma unroll
  for (int k = 0; k < 2; k++) x[12 + 2 * k] = c.own[k].like & mine, x[13 + 2 * k] = c.own[k].differ & mine;
  slice_count<16>(x, d);
}

// a + b of two numbers of N planes, into N+1 planes of which M are kept
template <int N, int M>
__host__ __device__ __forceinline__ void slice_add(const uint32_t (&a)[N], const uint32_t (&b)[N], uint32_t (&r)[M]) {
  uint32_t c = a[0] & b[0];
  r[0] = a[0] ^ b[0];
#pragma unroll
  for (int k = 1; k < N; k++) {
    r[k] = bop3<kXor3>(a[k], b[k], c);
    if (k + 1 < M) c = bop3<kMaj3>(a[k], b[k], c);
  }
  if constexpr (M > N) r[N] = c;
}

// Decision thresholds by ef - ei + 26 (0..52), kept in LDS: a move that is
// not uphill always passes; an uphill one passes when its second draw is
// below thr[ef - ei] (never at T = 0).
constexpr int kSliceThr = 53;
__host__ __device__ __forceinline__ int32_t slice_threshold(const Rule &r, int i) {
  return i <= 26 ? 0x7fffffff : r.zero_t ? 0 : r.thr[i - 26];
}

// changes of a lane's sites: n, and per plane of ef - ei + 26 how many have it
struct SliceCounts {
  uint32_t n = 0, bit[6] = {0, 0, 0, 0, 0, 0};
};
__host__ __device__ __forceinline__ Counts slice_counts(const SliceCounts &c) {
  int sum = 0;
#pragma unroll
  for (int k = 5; k >= 0; k--) sum = 2 * sum + (int)c.bit[k];
  return Counts{(int)c.n, sum - 26 * (int)c.n};
}

// The accept test of a lane's eight sites: d = ef - ei + 26 of the word as 6
// planes; u the first draws, replaced by the seeds to keep; thr the table of
// slice_threshold; limit: 4 * (the largest d that takes no second draw).
// Returns the changed sites (bit i: site 8q + i).
__host__ __device__ __forceinline__ uint32_t slice_decide(const SliceLane &t, const uint32_t (&d)[6], uint32_t moves,
                                                          const int32_t *thr, uint32_t limit, Words<4> (&u)[2],
                                                          SliceCounts &cnt) {
  const uint32_t sh = 8u * t.q;
  uint32_t by[6];
#pragma unroll
  for (int k = 0; k < 6; k++) by[k] = (d[k] >> sh) & 0xffu;
  // 4*d as a byte per site: planes 2..7, transposed
  uint32_t lo = (by[0] << 16) | (by[1] << 24), hi = by[2] | (by[3] << 8) | (by[4] << 16) | (by[5] << 24);
  slice_transpose8(lo, hi);
  uint32_t pass = 0;
#pragma unroll
  for (int i = 7; i >= 0; i--) {
    uint32_t &x = u[i >> 2].w[i & 3];
    const uint32_t at = ((i < 4 ? lo : hi) >> (8 * (i & 3))) & 0xffu;   // 4*d
    const int32_t th = *reinterpret_cast<const int32_t *>(reinterpret_cast<const char *>(thr) + at);
    const uint32_t u2 = (uint32_t)pm_step((int32_t)x);
    pass = shift_in_sign(pass, u2 - (uint32_t)th);   // u2 < thr
    x = at > limit ? u2 : x;
  }
  const uint32_t ch = (moves >> sh) & pass & t.mask;
  cnt.n += (uint32_t)__builtin_popcount(ch);
#pragma unroll
  for (int k = 0; k < 6; k++) cnt.bit[k] += (uint32_t)__builtin_popcount(ch & by[k]);
  return ch;
}

#ifdef __HIPCC__
// --------------------------------------------------------- a wavefront's pass
// A word's four lanes are q = 0..3, 16 lanes apart.  swap16 gives both lanes
// of a pair (q, q^1) the even one's x and the odd one's; swap32 those of (q,
// q^2).  (The instruction swaps rows of one register with rows of another.)
struct Pair {
  uint32_t a, b;
};
__device__ __forceinline__ Pair swap16(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane16_swap(x, x, false, false);
  return Pair{r[0], r[1]};
}
__device__ __forceinline__ Pair swap32(uint32_t x) {
  const auto r = __builtin_amdgcn_permlane32_swap(x, x, false, false);
  return Pair{r[0], r[1]};
}
__device__ __forceinline__ uint32_t quad_or(uint32_t x) {
  Pair p = swap16(x);
  p = swap32(p.a | p.b);
  return p.a | p.b;
}
__device__ __forceinline__ uint32_t quad_and(uint32_t x) {
  Pair p = swap16(x);
  p = swap32(p.a & p.b);
  return p.a & p.b;
}
// 4x4 byte transpose over the four lanes: byte j of lane q's result is byte q
// of lane j's word
__device__ __forceinline__ uint32_t quad_bytes(uint32_t x, uint32_t q) {
  Pair p = swap16(x);
  p = swap32(byte_perm(p.b, p.a, q & 1 ? 0x07030501u : 0x06020400u));
  return byte_perm(p.b, p.a, q & 2 ? 0x07060302u : 0x05040100u);
}
// word of lane k
__device__ __forceinline__ uint32_t lane_word(uint32_t x, uint32_t k) {
  return (uint32_t)__builtin_amdgcn_ds_bpermute((int)(k << 2), (int)x);
}
__device__ __forceinline__ void slice_join(SliceColour &c) {
#pragma unroll
  for (int k = 0; k < 2; k++) {
    c.own[k].like = quad_and(c.own[k].like);
    c.own[k].differ = quad_or(c.own[k].differ);
  }
  c.moves = quad_or(c.moves);
}
// the sum of the four lanes' parts of d
__device__ __forceinline__ void slice_sum(const uint32_t (&d)[5], uint32_t (&r)[6]) {
  uint32_t a5[5], b5[5], t[6], a6[6], b6[6];
#pragma unroll
  for (int k = 0; k < 5; k++) {
    const Pair p = swap16(d[k]);
    a5[k] = p.a, b5[k] = p.b;
  }
  slice_add(a5, b5, t);
#pragma unroll
  for (int k = 0; k < 6; k++) {
    const Pair p = swap32(t[k]);
    a6[k] = p.a, b6[k] = p.b;
  }
  slice_add(a6, b6, r);
}

// A wavefront's own LDS: for each of its 16 words the planes of the own row
// (0 even x, 1 odd x) and of the two colours' proposals (2, 3); and its own
// table of slice_threshold, so that no wavefront waits for another.
struct SliceLds {
  Words<4> w[4][16][kSliceMaxPlanes / 4];
  int32_t thr[64];
};

// Colours 2m and 2m+1 of wavefront v's rows; the lane's changes are added to
// cnt.  PG: s.PG.
template <bool FULL, int PG>
__device__ __forceinline__ void slice_wave(uint32_t *__restrict__ planes, int32_t *__restrict__ sseed, const Geom &g,
                                           const SliceGeom &s, const Rule &r, SliceLds &L, int m, uint32_t v,
                                           uint32_t l, SliceCounts &cnt) {
  const uint32_t q2 = 2u * (uint32_t)r.nspins, limit = r.zero_t ? 255u : 104u;
  const int32_t threshold = slice_threshold(r, min((int)l, kSliceThr - 1));
  const SliceLane t = slice_lane(g, s, m, v, l);
  const uint32_t slot = l & 15u;
  int32_t *const seeds = sseed + (int64_t)(2 * m) * s.seedc;
  auto seed_group = [&](int c, int j) {
    return reinterpret_cast<Words<4> *>(elem<uint32_t>(seeds + c * s.seedc, slice_seed_at(v, j, l)));
  };
  Words<4> u[2][2];
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int j = 0; j < 2; j++) u[c][j] = slice_seeds_load(seed_group(c, j));   // (idle lanes have seeds of their own too)
  // plane words through a buffer resource: a group's offset is scalar and the
  // lane's never changes, so a load takes no address arithmetic
  const auto rsrc = __builtin_amdgcn_make_buffer_rsrc(planes, 0, (int)((uint32_t)g.K * PG * s.nw * 16u), 0x00020000);
  const int step = s.nw * 16, odd = PG * step;   // bytes from a group to the next, from a colour to its odd one
  // the own row's words of plane 4i + q, held through the pass
  uint32_t own[2][PG];
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int i = 0; i < PG; i++)
      own[c][i] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rsrc, (int)(t.own + 4u * t.q), i * step + c * odd, 0);
  struct Group {
    Words<4> e[2], o[2];
  };
  auto load = [&](int i, Group &x) {
    i *= step;
#pragma unroll
    for (int r = 0; r < 2; r++) {
      const auto a = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)t.row[r], i, 0);
      const auto b = __builtin_amdgcn_raw_buffer_load_b128(rsrc, (int)t.row[r], i + odd, 0);
#pragma unroll
      for (int k = 0; k < 4; k++) x.e[r].w[k] = (uint32_t)a[k], x.o[r].w[k] = (uint32_t)b[k];
    }
  };
  Group x0, x1;
  load(0, x0);
  // the draws, and the proposals' plane words: a lane has the bytes of its
  // eight sites, four planes a word; after the transpose lane q has plane
  // 4i + q
#pragma unroll
  for (int c = 0; c < 2; c++) {
    uint32_t bytes[6];
    slice_draws<PG>(q2, u[c], bytes);
#pragma unroll
    for (int i = 0; i < PG; i++) L.w[2 + c][slot][i].w[t.q] = quad_bytes(bytes[i], t.q);
  }
  if constexpr (PG > 1) load(1, x1);
#pragma unroll
  for (int c = 0; c < 2; c++)
#pragma unroll
    for (int i = 0; i < PG; i++) L.w[c][slot][i].w[t.q] = own[c][i];
  L.thr[l] = threshold;
  wave_lds_sync();
  SliceColour c0, c1;
  slice_clear(c0);
  slice_clear(c1);
  auto group = [&](int i, const Group &x) {
    const Words<4> own0 = L.w[0][slot][i], own1 = L.w[1][slot][i], pr0 = L.w[2][slot][i], pr1 = L.w[3][slot][i];
    uint32_t prev[4][2], next[4][2];
#pragma unroll
    for (int k = 0; k < 4; k++)
#pragma unroll
      for (int r = 0; r < 2; r++) {
        prev[k][r] = lane_word(x.o[r].w[k], t.prev);
        next[k][r] = lane_word(x.e[r].w[k], t.next);
      }
#pragma unroll
    for (int k = 0; k < 4; k++) {
      if (i == PG - 1 && 4 * i + k >= s.P) break;
      const uint32_t e[2] = {x.e[0].w[k], x.e[1].w[k]}, o[2] = {x.o[0].w[k], x.o[1].w[k]};
      slice_rows<FULL>(t, e, o, prev[k], next[k], own0.w[k], own1.w[k], pr0.w[k], pr1.w[k], c0, c1);
    }
  };
#pragma unroll
  for (int i = 0; i < PG; i += 2) {
    group(i, x0);
    if (i + 2 < PG) load(i + 2, x0);
    if (i + 1 < PG) group(i + 1, x1);
    if (i + 3 < PG) load(i + 3, x1);
  }
  // the own row, plane 4i + q on lane q (planes from P on are 0 throughout)
#pragma unroll
  for (int i = 0; i < PG; i++)
    slice_own_first<FULL>(t, own[0][i], own[1][i], lane_word(own[1][i], t.prev), L.w[2][slot][i].w[t.q], c0);
  auto decide = [&](int c, SliceColour &col) {
    slice_join(col);
    uint32_t d[5], sum[6];
    slice_part(t, col, d);
    slice_sum(d, sum);
    return quad_or(slice_decide(t, sum, col.moves, L.thr, limit, u[c], cnt) << (8u * t.q));
  };
  auto store_own = [&](int c, int i, uint32_t x) {
    __builtin_amdgcn_raw_buffer_store_b32(x, rsrc, (int)(t.own + 4u * t.q), i * step + c * odd, 0);
  };
  uint32_t ch = decide(0, c0);
  // colour 2m's new words, and colour 2m+1's neighbours among them
#pragma unroll
  for (int i = 0; i < PG; i++) {
    own[0][i] = bop3<kSel>(ch, L.w[2][slot][i].w[t.q], own[0][i]);
    slice_own_second<FULL>(t, own[0][i], lane_word(own[0][i], t.next), own[1][i], L.w[3][slot][i].w[t.q], c1);
  }
  if (ch) {
#pragma unroll
    for (int i = 0; i < PG; i++) store_own(0, i, own[0][i]);
  }
  ch = decide(1, c1);
  if (FULL || t.mask) {
#pragma unroll
    for (int c = 0; c < 2; c++)
#pragma unroll
      for (int j = 0; j < 2; j++) slice_seeds_store(seed_group(c, j), u[c][j]);
  }
  if (ch) {
#pragma unroll
    for (int i = 0; i < PG; i++) store_own(1, i, bop3<kSel>(ch, L.w[3][slot][i].w[t.q], own[1][i]));
  }
}
#endif

}  // namespace spk
