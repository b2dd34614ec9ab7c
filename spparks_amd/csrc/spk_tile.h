// spk_tile.h -- several colour passes per launch for lattices whose single
// colour pass is too short for the chip.
//
// A colour pass of a lattice of up to a few million sites takes 4-6 us
// whatever it does: the launch, one dependent chain of loads, the counts and
// the drain are most of it (1000^2 Ising: 5.5 us a pass, of which the events
// are about 1).  Here a workgroup loads a box of the lattice with a halo
// into LDS and runs `npass` consecutive colour passes on it, the passes of
// one or more sweeps; only the box it owns is written back, to the other of
// two state buffers, so no workgroup reads what another writes during a
// launch.
//
// The halo comes from the dependence of the passes themselves.  Let N_k be
// the box (lattice coordinates, relative to the owned box) whose sites must
// be right after pass k; N_last is the owned box.  Pass k updates the sites
// of its colour in N_k, each from its neighbours before the pass, so
// N_(k-1) is N_k grown by one row wherever a site of that colour can lie on
// N_k's face: on a checkerboard always, on sq/8n and sc/26n when the face's
// parity is the colour's.  The growth is uneven: per sweep x grows by 4
// rows a side on sq/8n but y by 2 (the colour changes y parity only half as
// often), and on sc/26n x, y, z by 8, 4, 2.  A dimension the box spans whole is
// periodic inside the box and needs no halo.  Sites outside N_k may be
// computed as well (the packs are 4 sites wide): they are never needed
// again, because every later N is smaller.
//
// The events are pack_count / pack_decide (spk_device.h), as in the
// per-colour kernel, on the LDS copy with the box's own geometry.
#pragma once

#include "spk_device.h"

namespace spk {

constexpr int kTileMaxPass = 32;    // colour passes per launch
constexpr int kTileMaxSweeps = 17;  // accumulator rows those can touch (K >= 2)

// One pass: the x range (in units of the plan's vec sites) and the rows of
// the box it works on, in the box's own sub-grid, and their count.
struct alignas(16) TilePass {
  uint16_t p0, np, b0, nb, e0, ne;
  uint32_t items;
  FastDiv fp, fb;   // division by np, nb
};

struct TilePlan {
  Geom gl;             // the box with its halo, as a lattice of its own
  int ox, oy, oz;      // the owned box within it (lattice coordinates)
  int wx, wy, wz;      // its extents (the whole lattice's where the box spans it)
  int cx, cy, cz;      // boxes along x, y, z
  int c0;              // colour of the first pass
  int npass;
  int vec;             // sites per thread: 4 (packs) or 1
  uint32_t spin_bytes; // LDS bytes of the spins (a multiple of 16); the seeds follow
  TilePass pass[kTileMaxPass];
};

// colour c's parity along dimension d (0 x, 1 y, 2 z), or -1 on a
// checkerboard, where a row holds sites of both colours
__host__ __device__ inline int tile_parity(int lat, int c, int d) {
  if (lat == SPK_HIP_SQ_8N || lat == SPK_HIP_SC_26N) return (c >> d) & 1;
  return -1;
}

// What passes c0 .. c0+npass-1 update of a box of w sites: pass k the sites
// [lo[k], hi[k]) of the box moved by org, and the box with its halo, ext sites
// from org.  False where a plan cannot hold it.
struct TileRegion {
  bool whole[3];
  int org[3], ext[3];
  int lo[kTileMaxPass][3], hi[kTileMaxPass][3];
};
inline bool tile_region(const Geom &g, const int (&w)[3], int c0, int npass, TileRegion &r) {
  if (npass < 1 || npass > kTileMaxPass) return false;
  const int n[3] = {g.nx, g.ny, g.nz};
  int lo[3], hi[3];
  for (int d = 0; d < 3; d++) {
    r.whole[d] = w[d] >= n[d];
    lo[d] = 0;
    hi[d] = r.whole[d] ? n[d] : w[d];
  }
  int c = (c0 + npass - 1) % g.K;
  for (int k = npass - 1; k >= 0; k--, c = c ? c - 1 : g.K - 1) {
    for (int d = 0; d < 3; d++) {
      r.lo[k][d] = lo[d];
      r.hi[k][d] = hi[d];
      if (r.whole[d]) continue;
      const int p = tile_parity(g.lat, c, d);
      if (p < 0 || (lo[d] & 1) == p) lo[d]--;
      if (p < 0 || ((hi[d] - 1) & 1) == p) hi[d]++;
    }
  }
  // the box with its halo: x from a multiple of 8 (packs of 4 sub-grid
  // sites), y and z from an even row, so parities carry over
  for (int d = 0; d < 3; d++) {
    const int unit = d == 0 ? 8 : 2;
    if (r.whole[d]) {
      r.org[d] = 0;
      r.ext[d] = n[d];
    } else {
      r.org[d] = -((-lo[d] + unit - 1) / unit * unit);
      r.ext[d] = (hi[d] - r.org[d] + unit - 1) / unit * unit;
    }
  }
  return r.ext[0] <= 65535 && r.ext[1] <= 65535 && r.ext[2] <= 65535 &&
         (int64_t)r.ext[0] * r.ext[1] * r.ext[2] <= (1 << 20);
}

// The sub-grid of the halo box that pass k (colour c) updates: a along x in
// sites, b and e its rows and planes.
struct TileSpan {
  int a[2], b[2], e[2];
};
inline TileSpan tile_span(int lat, const TileRegion &r, int k, int c) {
  const bool ysub = lat == SPK_HIP_SQ_8N || lat == SPK_HIP_SC_26N, zsub = lat == SPK_HIP_SC_26N;
  auto sub = [&](int d, bool halved, int (&o)[2]) {
    const int l = r.lo[k][d] - r.org[d], h = r.hi[k][d] - r.org[d];
    if (!halved) {
      o[0] = l, o[1] = h;
      return;
    }
    const int p = tile_parity(lat, c, d);
    if (p < 0) o[0] = l / 2, o[1] = (h + 1) / 2;        // x of a checkerboard: both parities
    else o[0] = (l - p + 1) / 2, o[1] = (h - p + 1) / 2;   // sites 2r + p in [l, h)
  };
  TileSpan t;
  sub(0, true, t.a);
  sub(1, ysub, t.b);
  sub(2, zsub, t.e);
  return t;
}
// packs of vec sites along x from t.a
inline uint32_t tile_packs(const TileSpan &t, int vec) {
  return vec == 4 ? (uint32_t)((t.a[1] + 3) / 4 - t.a[0] / 4) : (uint32_t)(t.a[1] - t.a[0]);
}

// Fills the plan for `npass` passes from colour c0 on, for owned boxes of
// w[] lattice sites (w[d] >= the edge: the whole dimension; otherwise even, a
// multiple of 8 in x).  False when a box would not fit the plan's tables.
// vec: sites per thread; spin_size: bytes per stored spin.
inline bool tile_plan_make(const Geom &g, const int (&w)[3], int c0, int npass, int vec, int spin_size, TilePlan *tp) {
  TileRegion r;
  if (!tile_region(g, w, c0, npass, r)) return false;
  const int n[3] = {g.nx, g.ny, g.nz};
  const int (&org)[3] = r.org, (&ext)[3] = r.ext;
  const bool (&whole)[3] = r.whole;
  geom_init(tp->gl, g.lat, ext[0], ext[1], ext[2]);
  tp->ox = -org[0], tp->oy = -org[1], tp->oz = -org[2];
  tp->wx = whole[0] ? n[0] : w[0], tp->wy = whole[1] ? n[1] : w[1], tp->wz = whole[2] ? n[2] : w[2];
  tp->cx = (n[0] + tp->wx - 1) / tp->wx, tp->cy = (n[1] + tp->wy - 1) / tp->wy, tp->cz = (n[2] + tp->wz - 1) / tp->wz;
  tp->c0 = c0;
  tp->npass = npass;
  tp->vec = vec;
  tp->spin_bytes = ((uint32_t)tp->gl.K * (uint32_t)tp->gl.Mp * (uint32_t)spin_size + 15u) / 16u * 16u;
  for (int k = 0; k < npass; k++) {
    const TileSpan sp = tile_span(g.lat, r, k, (c0 + k) % g.K);
    TilePass &t = tp->pass[k];
    t.p0 = (uint16_t)(sp.a[0] / vec);
    t.np = (uint16_t)tile_packs(sp, vec);
    t.b0 = (uint16_t)sp.b[0], t.nb = (uint16_t)(sp.b[1] - sp.b[0]);
    t.e0 = (uint16_t)sp.e[0], t.ne = (uint16_t)(sp.e[1] - sp.e[0]);
    t.items = (uint32_t)t.np * t.nb * t.ne;
    t.fp = fastdiv_make(t.np);
    t.fb = fastdiv_make(t.nb);
  }
  return true;
}

// LDS bytes of a plan's box: spins, then seeds
inline size_t tile_lds(const TilePlan &tp) {
  return tp.spin_bytes + (size_t)tp.gl.K * tp.gl.Mp * sizeof(int32_t);
}

// the box of workgroup `tile`: lattice coordinates of its owned corner
struct TileBox {
  int x, y, z;
};
__host__ __device__ __forceinline__ TileBox tile_box(const TilePlan &tp, int tile) {
  const int r = tile / tp.cx;
  return TileBox{(tile - r * tp.cx) * tp.wx, (r % tp.cy) * tp.wy, (r / tp.cy) * tp.wz};
}

__host__ __device__ __forceinline__ int tile_wrap(int v, int n) {
  if (v >= n) v -= n;
  if (v < 0) v += n;
  if (v >= 0 && v < n) return v;
  v %= n;   // a box wider than the lattice
  return v < 0 ? v + n : v;
}

// rows per lattice row of the sub-grid: y of a Moore lattice and z of sc/26n
// are halved
template <int LAT> struct TileHalf {
  static constexpr int y = LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N ? 2 : 1;
  static constexpr int z = LAT == SPK_HIP_SC_26N ? 2 : 1;
};

// Pack i of the box's K*Mp/4 packs: its offset in the box (elements), and
// where its first site lies in the lattice: offset of the row's start, and
// the sub-grid x of the site.
struct TileSlot {
  uint32_t local;
  int64_t row;   // lattice offset of the row (x = 0)
  int a;         // x of lane 0 in the lattice's sub-grid, 0..hx-1
  int la;        // x of lane 0 in the box
};
template <int LAT>
__host__ __device__ __forceinline__ TileSlot tile_slot(const Geom &g, const TilePlan &tp, const TileBox &bx, uint32_t i) {
  const Geom &gl = tp.gl;
  uint32_t row, a4, rest, b;
  fastdiv(gl.row4, i, row, a4);
  fastdiv(gl.rows, row, rest, b);
  const uint32_t c = rest / (uint32_t)gl.hz, e = rest - c * (uint32_t)gl.hz;
  TileSlot s;
  s.local = i * 4u;
  s.la = (int)a4 * 4;
  s.a = tile_wrap((bx.x - tp.ox) / 2 + s.la, g.hx);
  const int gb = tile_wrap((bx.y - tp.oy) / TileHalf<LAT>::y + (int)b, g.hy);
  const int ge = tile_wrap((bx.z - tp.oz) / TileHalf<LAT>::z + (int)e, g.hz);
  s.row = (int64_t)c * g.Mp + (int64_t)g.px * (gb + (int64_t)g.hy * ge);
  return s;
}

// One pack from the lattice into the box.  Lanes past the end of a row wrap
// to its start (the box's x runs on unwrapped); where the box spans x, the
// lanes past the row's end are pad lanes and hold whatever they wrap to.
template <int LAT, typename T>
__host__ __device__ __forceinline__ void tile_load(const T *__restrict__ spin, const int32_t *__restrict__ seed,
                                                   const Geom &g, const TilePlan &tp, const TileBox &bx, uint32_t i,
                                                   T *ls, int32_t *lk) {
  const TileSlot s = tile_slot<LAT>(g, tp, bx, i);
  if ((s.a & 3) == 0 && s.a + 4 <= g.hx) {
    store_lanes<T, uint32_t>(ls, s.local, load_lanes<T, int64_t>(spin, s.row + s.a));
    *reinterpret_cast<Words<4> *>(lk + s.local) = *reinterpret_cast<const Words<4> *>(seed + s.row + s.a);
    return;
  }
  int a = s.a;
  for (int v = 0; v < 4; v++) {
    ls[s.local + v] = spin[s.row + a];
    lk[s.local + v] = seed[s.row + a];
    a = a + 1 == g.hx ? 0 : a + 1;
  }
}

// One owned pack back to the lattice (other packs of the box are skipped).
template <int LAT, typename T>
__host__ __device__ __forceinline__ void tile_store(T *__restrict__ spin, int32_t *__restrict__ seed, const Geom &g,
                                                    const TilePlan &tp, const TileBox &bx, uint32_t i, const T *ls,
                                                    const int32_t *lk) {
  // the owned packs, colour, plane, row, pack: the owned box starts at a pack
  const uint32_t npo = (uint32_t)(tp.wx / 2 + 3) / 4, nbo = (uint32_t)(tp.wy / TileHalf<LAT>::y),
                 neo = (uint32_t)(tp.wz / TileHalf<LAT>::z);
  const uint32_t r0 = i / npo, p = i - r0 * npo, r1 = r0 / nbo, b = r0 - r1 * nbo, c = r1 / neo, e = r1 - c * neo;
  const int ga = bx.x / 2 + (int)p * 4, gb = bx.y / TileHalf<LAT>::y + (int)b, ge = bx.z / TileHalf<LAT>::z + (int)e;
  if (ga >= g.hx || gb >= g.hy || ge >= g.hz) return;   // past the lattice's end: another box's sites
  const Geom &gl = tp.gl;
  const uint32_t local = c * (uint32_t)gl.Mp + (uint32_t)(tp.ox / 2) + p * 4u +
                         (uint32_t)gl.px * ((uint32_t)(tp.oy / TileHalf<LAT>::y) + b +
                                            (uint32_t)gl.hy * ((uint32_t)(tp.oz / TileHalf<LAT>::z) + e));
  const int64_t at = (int64_t)c * g.Mp + ga + (int64_t)g.px * (gb + (int64_t)g.hy * ge);
  if (ga + 4 <= g.hx) {
    store_lanes<T, int64_t>(spin, at, load_lanes<T, uint32_t>(ls, local));
    *reinterpret_cast<Words<4> *>(seed + at) = *reinterpret_cast<const Words<4> *>(lk + local);
    return;
  }
  for (int v = 0; ga + v < g.hx; v++) {
    spin[at + v] = ls[local + v];
    seed[at + v] = lk[local + v];
  }
}

// owned packs of a plan's box (the range of tile_store's i)
template <int LAT>
__host__ __device__ __forceinline__ uint32_t tile_store_items(const TilePlan &tp) {
  return (uint32_t)tp.gl.K * ((uint32_t)(tp.wx / 2 + 3) / 4) * (uint32_t)(tp.wy / TileHalf<LAT>::y) *
         (uint32_t)(tp.wz / TileHalf<LAT>::z);
}

// Item i of pass ps on a plan of vec 4: the events of a pack.  Counts only
// the sites the box owns (and that the lattice has).
template <int LAT, typename T, bool TWO, int XDIR>
__host__ __device__ __forceinline__ Counts tile_events(T *ls, int32_t *lk, const Geom &g, const Rule &r, const int *thr,
                                                       const TilePlan &tp, const TileBox &bx, const TilePass &ps, int c,
                                                       uint32_t i) {
  const Geom &gl = tp.gl;
  uint32_t row, p, ze, yb;
  fastdiv(ps.fp, i, row, p);
  fastdiv(ps.fb, row, ze, yb);
  const int a0 = (int)(ps.p0 + p) * 4, b = (int)(ps.b0 + yb), e = (int)(ps.e0 + ze);
  PackWork<T, TWO, uint32_t> w = pack_count<LAT, T, TWO, uint32_t, XDIR>(ls, lk, gl, r, c, a0, b, e);
  // owned lanes [v0, v1) of the pack, if its row is owned
  const int ob = b - tp.oy / TileHalf<LAT>::y, oe = e - tp.oz / TileHalf<LAT>::z, oa = a0 - tp.ox / 2;
  const int rows_y = min(tp.wy, g.ny - bx.y) / TileHalf<LAT>::y, rows_z = min(tp.wz, g.nz - bx.z) / TileHalf<LAT>::z;
  const bool owned = (unsigned)ob < (unsigned)rows_y && (unsigned)oe < (unsigned)rows_z;
  const int v0 = -oa, v1 = owned ? min(tp.wx, g.nx - bx.x) / 2 - oa : 0;
  return pack_decide<LAT, T, TWO, uint32_t>(w, ls, lk, gl, r, thr, c, v0, v1);
}

// Item i of pass ps on a plan of vec 1: one site's event.  A pass over a
// small box has few wavefronts, and its time is one thread's own chain: a
// site takes a third to a fifth of a pack's instructions.  APP: potts or
// ising (SPK_HIP_POTTS stands for both; TWO tells them apart as in
// propose_as), or a proposal variant.
template <int LAT, typename T, bool TWO, int APP = SPK_HIP_POTTS>
__host__ __device__ __forceinline__ Counts tile_event(T *ls, int32_t *lk, const Geom &g, const Rule &r, const int *thr,
                                                      const TilePlan &tp, const TileBox &bx, const TilePass &ps, int c,
                                                      uint32_t i) {
  const Geom &gl = tp.gl;
  uint32_t row, p, ze, yb;
  fastdiv(ps.fp, i, row, p);
  fastdiv(ps.fb, row, ze, yb);
  const int a = (int)(ps.p0 + p), b = (int)(ps.b0 + yb), e = (int)(ps.e0 + ze);
  const RowOffset<uint32_t> px((uint32_t)gl.px), pxy((uint32_t)gl.px * (uint32_t)gl.hy);
  const uint32_t Mp = (uint32_t)gl.Mp;
  const uint32_t at = (uint32_t)c * Mp + (uint32_t)a + px * (uint32_t)b + pxy * (uint32_t)e;
  const int32_t old = (int32_t)ls[at], seed = lk[at];
  constexpr int NN = NeighCount<LAT>::value;
  // the neighbours in the reference's order (Shell), dx outermost
  int32_t nb[NN];
  if constexpr (LAT == SPK_HIP_SQ_4N || LAT == SPK_HIP_SC_6N) {
    const uint32_t o = (uint32_t)(1 - c) * Mp;
    const bool side = (LAT == SPK_HIP_SC_6N ? b + e + c : b + c) & 1;
    const uint32_t xl = (uint32_t)(side ? a : wrap_dec(a, gl.hx)), xr = (uint32_t)(side ? wrap_inc(a, gl.hx) : a);
    const uint32_t zr = o + pxy * (uint32_t)e, yz = px * (uint32_t)b + zr;
    nb[0] = ls[yz + xl];
    nb[NN - 1] = ls[yz + xr];
    nb[1] = ls[zr + px * (uint32_t)wrap_dec(b, gl.hy) + (uint32_t)a];
    nb[NN - 2] = ls[zr + px * (uint32_t)wrap_inc(b, gl.hy) + (uint32_t)a];
    if constexpr (LAT == SPK_HIP_SC_6N) {
      const uint32_t yr = o + px * (uint32_t)b + (uint32_t)a;
      nb[2] = ls[yr + pxy * (uint32_t)wrap_dec(e, gl.hz)];
      nb[3] = ls[yr + pxy * (uint32_t)wrap_inc(e, gl.hz)];
    }
  } else {
    constexpr bool three = LAT == SPK_HIP_SC_26N;
    const int pi = c & 1, pj = (c >> 1) & 1, pk = three ? c >> 2 : 0;
    // x-1 and x+1 lie in the other x parity, at a and beside it
    const uint32_t xl = (uint32_t)(pi ? a : wrap_dec(a, gl.hx)), xr = (uint32_t)(pi ? wrap_inc(a, gl.hx) : a);
    const uint32_t yo = px * (uint32_t)(pj ? wrap_inc(b, gl.hy) : wrap_dec(b, gl.hy)), y0 = px * (uint32_t)b;
    const uint32_t ys[3] = {pj ? y0 : yo, y0, pj ? yo : y0};
    const uint32_t zo = three ? pxy * (uint32_t)(pk ? wrap_inc(e, gl.hz) : wrap_dec(e, gl.hz)) : 0u;
    const uint32_t z0 = pxy * (uint32_t)e;
    const uint32_t zs[3] = {pk ? z0 : zo, z0, pk ? zo : z0};
    constexpr int nz = three ? 3 : 1;
#pragma unroll
    for (int j = 0; j < 3; j++)
#pragma unroll
      for (int k = 0; k < nz; k++) {
        const int dz = three ? k : 1, m = j * nz + k;   // m: the row's place among those of one dx
        const uint32_t q = 2u * (uint32_t)(pj ^ (j != 1)) + 4u * (uint32_t)(pk ^ (dz != 1));
        const uint32_t yz = ys[j] + zs[dz], other = ((uint32_t)(1 - pi) + q) * Mp + yz;
        constexpr int R = 3 * nz, mid = R / 2;
        nb[m] = ls[other + xl];
        if (m != mid) nb[R + m - (m > mid)] = ls[((uint32_t)pi + q) * Mp + yz + (uint32_t)a];
        nb[2 * R - 1 + m] = ls[other + xr];
      }
  }
  const int ob = b - tp.oy / TileHalf<LAT>::y, oe = e - tp.oz / TileHalf<LAT>::z, oa = a - tp.ox / 2;
  const int rows_y = min(tp.wy, g.ny - bx.y) / TileHalf<LAT>::y, rows_z = min(tp.wz, g.nz - bx.z) / TileHalf<LAT>::z;
  const bool owned = (unsigned)ob < (unsigned)rows_y && (unsigned)oe < (unsigned)rows_z &&
                     (unsigned)oa < (unsigned)(min(tp.wx, g.nx - bx.x) / 2);
  if constexpr (APP >= SPK_HIP_POTTS_NEIGH) {
    const SiteOutcome v = variant_event<APP, NN>(r, thr, old, seed, nb);
    lk[at] = v.seed;
    if (v.changed) ls[at] = (T)v.spin;
    return Counts{owned && v.changed, owned ? v.dE : 0};
  }
  int32_t s = pm_step(seed);
  const int32_t prop = propose_as<TWO>(r, s);
  int ei, ef;
  if constexpr (TWO) {
    // values 1 and 2: the sum tells how many are 2
    int sum = 0;
#pragma unroll
    for (int m = 0; m < NN; m++) sum += nb[m];
    ei = old == 1 ? sum - NN : 2 * NN - sum;
    ef = prop == old ? ei : NN - ei;
  } else {
    // flags min(x, 1), not compares: a compare's mask costs two wait states
    // before the add that takes it
    uint32_t o = 0, w = 0;
    static_assert(NN % 2 == 0, "neighbours are counted in pairs");
#pragma unroll
    for (int m = 0; m < NN; m += 2) {
      add_ne_words2(o, (uint32_t)(nb[m] ^ old), (uint32_t)(nb[m + 1] ^ old));
      add_ne_words2(w, (uint32_t)(nb[m] ^ prop), (uint32_t)(nb[m + 1] ^ prop));
    }
    ei = (int)o;
    ef = (int)w;
  }
  const bool accept = metropolis_select(r, thr, ei, ef, s);
  const bool changed = accept && prop != old;
  lk[at] = s;
  if (changed) ls[at] = (T)prop;
  const bool counted = changed && owned;
  return Counts{counted, counted ? ef - ei : 0};
}

}  // namespace spk
