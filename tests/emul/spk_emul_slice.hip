// spk_emul_slice.hip -- host-only emulation of the bit-sliced passes
// (spk_slice.h), for CPU tests: conversions and the kernel's own steps, lane
// by lane, under AddressSanitizer.  Test infrastructure; not part of the library.
//
// usage: spk_emul_slice app lat nx ny nz nspins kT nsweeps in.bin out.bin
//   in.bin : int32 spin[N], int32 seed[N] (reference order)
//   out.bin: int32 spin[N], int32 seed[N], then per sweep int64 naccept and
//            sum of ef - ei
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "spk_slice.h"

using namespace spk;

extern "C" int spk_hip_metropolis_table(double, int, double *, int32_t *);

template <bool FULL>
static Counts wave(std::vector<uint32_t> &planes, std::vector<int32_t> &sseed, const Geom &g, const SliceGeom &s,
                   const Rule &r, const int32_t *thr, int m, uint32_t v) {
  struct Lane {
    SliceLane t;
    Words<4> u[2][2];
    SliceColour c[2];
    uint32_t d[5], sum[6];
    SliceCounts cnt;
    uint32_t ch;
  };
  std::vector<Lane> L(64);
  std::vector<uint32_t> pr(2 * (size_t)s.P * 16);   // [colour][plane][word]
  auto word = [&](uint32_t off, int p, bool odd) -> uint32_t & { return planes.at(off / 4 + (size_t)(p / 4 + (odd ? s.PG : 0)) * s.nw * 4 + p % 4); };
  for (uint32_t l = 0; l < 64; l++) {
    Lane &x = L[l];
    x.t = slice_lane(g, s, m, v, l);
    for (int c = 0; c < 2; c++) {
      for (int j = 0; j < 2; j++)
        for (int k = 0; k < 4; k++) x.u[c][j].w[k] = sseed.at((2 * m + c) * s.seedc + slice_seed_at(v, j, l) + k);
      uint32_t bytes[6];
      slice_draws<kSliceMaxPlanes / 4>(2u * (uint32_t)r.nspins, x.u[c], bytes);
      for (int p = 0; p < s.P; p++)
        pr[((size_t)c * s.P + p) * 16 + (l & 15)] |= ((bytes[p / 4] >> (8 * (p % 4))) & 0xffu) << (8 * (l >> 4));
      slice_clear(x.c[c]);
    }
  }
  for (uint32_t l = 0; l < 64; l++) {
    Lane &x = L[l];
    for (int p = 0; p < s.P; p++) {
      const SliceLane &tp = L[x.t.prev].t, &tn = L[x.t.next].t;
      const uint32_t re[2] = {word(x.t.row[0], p, false), word(x.t.row[1], p, false)};
      const uint32_t ro[2] = {word(x.t.row[0], p, true), word(x.t.row[1], p, true)};
      const uint32_t prev[2] = {word(tp.row[0], p, true), word(tp.row[1], p, true)};
      const uint32_t next[2] = {word(tn.row[0], p, false), word(tn.row[1], p, false)};
      const uint32_t pr0 = pr[(size_t)p * 16 + (l & 15)], pr1 = pr[((size_t)s.P + p) * 16 + (l & 15)];
      const uint32_t e = word(x.t.own, p, false), o = word(x.t.own, p, true);
      slice_rows<FULL>(x.t, re, ro, prev, next, e, o, pr0, pr1, x.c[0], x.c[1]);
      slice_own_first<FULL>(x.t, e, o, word(tp.own, p, true), pr0, x.c[0]);
    }
  }
  Counts sum{0, 0};
  for (int c = 0; c < 2; c++) {
    if (c == 1)
      for (uint32_t l = 0; l < 64; l++) {
        Lane &x = L[l];
        for (int p = 0; p < s.P; p++) {
          const uint32_t pr1 = pr[((size_t)s.P + p) * 16 + (l & 15)];
          slice_own_second<FULL>(x.t, word(x.t.own, p, false), word(L[x.t.next].t.own, p, false), word(x.t.own, p, true), pr1, x.c[1]);
        }
      }
    for (uint32_t l = 0; l < 64; l++) slice_part(L[l].t, L[l].c[c], L[l].d);
    for (uint32_t l = 0; l < 16; l++) {
      uint32_t a[6], b[6];
      slice_add(L[l].d, L[l + 16].d, a);
      slice_add(L[l + 32].d, L[l + 48].d, b);
      slice_add(a, b, L[l].sum);
      for (int k = 1; k < 4; k++) std::copy(L[l].sum, L[l].sum + 6, L[l + 16 * k].sum);
    }
    for (uint32_t l = 0; l < 16; l++) {
      uint32_t ch = 0;
      for (int k = 0; k < 4; k++) {
        Lane &x = L[l + 16 * k];
        ch |= slice_decide(x.t, x.sum, x.c[c].moves, thr, r.zero_t ? 255u : 104u, x.u[c], x.cnt) << (8 * k);
        if (x.t.mask)
          for (int j = 0; j < 2; j++)
            for (int i = 0; i < 4; i++) sseed.at((2 * m + c) * s.seedc + slice_seed_at(v, j, l + 16 * k) + i) = x.u[c][j].w[i];
      }
      if (!ch) continue;
      for (int p = 0; p < s.P; p++) {
        uint32_t &o = word(L[l].t.own, p, c == 1);
        o = bop3<kSel>(ch, pr[((size_t)c * s.P + p) * 16 + (l & 15)], o);
      }
    }
  }
  for (auto &x : L) {
    const Counts c = slice_counts(x.cnt);
    sum.nacc += c.nacc, sum.de += c.de;
  }
  return sum;
}

template <int LAT>
static int run(int app, const int *n, int q, double kt, int nsw, const char *in, const char *out) {
  Geom g{};
  geom_init(g, LAT, n[0], n[1], n[2]);
  if (!slice_fits(g, q)) { fprintf(stderr, "does not fit\n"); return 4; }
  const long long N = (long long)n[0] * n[1] * n[2], S = (long long)g.K * g.Mp;
  Rule r{};
  r.app = app, r.nspins = app == SPK_HIP_ISING ? 2 : q, r.zero_t = kt == 0.0;
  int32_t thr[27];
  spk_hip_metropolis_table(kt > 0 ? kt : 1.0, maxneigh_of(LAT), nullptr, thr);
  r.half = thr[0];
  for (int d = 1; d <= maxneigh_of(LAT); d++) r.thr[d] = thr[d];
  // proposals: integers against the rule's doubles
  uint32_t x = 12345;
  for (int i = 0; i < 20000; i++) {
    x = (uint32_t)pm_step((int32_t)x);
    const uint32_t at[3] = {x, (uint32_t)i + 1, (uint32_t)kIM - 1 - (uint32_t)i};
    for (uint32_t sd : at)
      if ((int32_t)slice_propose(2u * (uint32_t)r.nspins, sd) + 1 != propose(r, (int32_t)sd)) {
        fprintf(stderr, "proposal of draw %u differs\n", sd);
        return 7;
      }
  }
  std::vector<int32_t> sn(N), kn(N);
  FILE *f = fopen(in, "rb");
  if (!f || fread(sn.data(), 4, N, f) != (size_t)N || fread(kn.data(), 4, N, f) != (size_t)N) return 2;
  fclose(f);
  std::vector<int32_t> sp(S, 1), sd(S, 1);
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    sp[p] = sn[t], sd[p] = kn[t];
  }
  const SliceGeom s = slice_geom(g, r.nspins);
  std::vector<uint32_t> planes((size_t)g.K * s.PG * s.nw * 4, 0xffffffffu);
  std::vector<int32_t> sseed((size_t)g.K * s.seedc);
  for (int c = 0; c < g.K; c++)
    for (int t = 0; t < s.nw; t++) slice_pack_word<int32_t>(sp.data(), g, s, c, t, planes.data());
  for (int64_t i = 0; i < g.K * s.seedc / 4; i++) slice_seeds_in(sd.data(), g, s, i, sseed.data());
  const bool full = s.W == 32 && s.last == 32;
  int32_t table[kSliceThr];
  for (int i = 0; i < kSliceThr; i++) table[i] = slice_threshold(r, i);
  std::vector<long long> na(nsw), de(nsw);
  for (int sw = 0; sw < nsw; sw++)
    for (int m = 0; m < g.K / 2; m++)
      for (int v = 0; v < s.waves; v++) {
        const Counts c = full ? wave<true>(planes, sseed, g, s, r, table, m, v) : wave<false>(planes, sseed, g, s, r, table, m, v);
        na[sw] += c.nacc, de[sw] += c.de;
      }
  std::fill(sp.begin(), sp.end(), -1);
  std::fill(sd.begin(), sd.end(), -1);
  for (int c = 0; c < g.K; c++)
    for (int t = 0; t < s.nw; t++) slice_unpack_word<int32_t>(planes.data(), g, s, c, t, sp.data());
  for (int64_t i = 0; i < g.K * s.seedc / 4; i++) slice_seeds_out(sseed.data(), g, s, i, sd.data());
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    sn[t] = sp[p], kn[t] = sd[p];
    const SliceSite x = slice_site(g, s, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    if (slice_spin_at(planes.data(), s, x) != sn[t] || sseed.at(slice_seed_slot(s, x)) != kn[t]) {
      fprintf(stderr, "site %lld read in place differs\n", t);
      return 8;
    }
  }
  f = fopen(out, "wb");
  if (!f) return 6;
  fwrite(sn.data(), 4, N, f);
  fwrite(kn.data(), 4, N, f);
  for (int i = 0; i < nsw; i++) {
    fwrite(&na[i], 8, 1, f);
    fwrite(&de[i], 8, 1, f);
  }
  fclose(f);
  return 0;
}

int main(int argc, char **argv) {
  if (argc != 11) { fprintf(stderr, "usage: app lat nx ny nz q kT nsweeps in out\n"); return 1; }
  const int app = atoi(argv[1]), n[3] = {atoi(argv[3]), atoi(argv[4]), atoi(argv[5])};
  return run<SPK_HIP_SC_26N>(app, n, atoi(argv[6]), atof(argv[7]), atoi(argv[8]), argv[9], argv[10]);
}
