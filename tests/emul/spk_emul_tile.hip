// spk_emul_tile.hip -- host-only emulation of the tile kernel (spk_tile.h), for
// CPU tests: the kernel's own load, pass and store steps, one item at a time,
// under AddressSanitizer.  Test infrastructure; not part of the library.
//
// usage: spk_emul_tile app lat nx ny nz nspins kT stype vec wx wy wz cuts in.bin out.bin
//   stype: 0 uint8, 1 uint16, 2 int32; vec: sites per thread (1, 4); wx wy wz: the owned box; cuts: the
//   colour passes of each launch, "8,8,4" (their sum a whole number of sweeps)
//   in.bin : int32 spin[N], int32 seed[N] (reference order)
//   out.bin: int32 spin[N], int32 seed[N], then per sweep int64 naccept and
//            sum of ef - ei
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <string>
#include <vector>

#include "spk_tile.h"

using namespace spk;

extern "C" int spk_hip_metropolis_table(double, int, double *, int32_t *);

template <int LAT, typename T, bool TWO, int APP>
static int run(int vec, int app, const int *n, int q, double kt, const int (&w)[3], const std::vector<int> &cuts,
               const char *in, const char *out) {
  Geom g{};
  geom_init(g, LAT, n[0], n[1], n[2]);
  const long long N = (long long)n[0] * n[1] * n[2], S = (long long)g.K * g.Mp;
  Rule r{};
  r.app = app, r.nspins = app == SPK_HIP_ISING || app == SPK_HIP_ISING_SINGLE ? 2 : q, r.zero_t = kt == 0.0;
  int32_t thr[27];
  spk_hip_metropolis_table(kt > 0 ? kt : 1.0, maxneigh_of(LAT), nullptr, thr);
  r.half = thr[0];
  for (int d = 1; d <= maxneigh_of(LAT); d++) r.thr[d] = thr[d];
  std::vector<int32_t> sn(N), kn(N);
  FILE *f = fopen(in, "rb");
  if (!f || fread(sn.data(), 4, N, f) != (size_t)N || fread(kn.data(), 4, N, f) != (size_t)N) return 2;
  fclose(f);
  std::vector<T> s[2] = {std::vector<T>(S, (T)0), std::vector<T>(S, (T)0)};
  std::vector<int32_t> k[2] = {std::vector<int32_t>(S, 1), std::vector<int32_t>(S, 1)};
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    s[0][p] = (T)sn[t], k[0][p] = kn[t];
  }
  int total = 0, from = 0, q0 = 0;
  for (int c : cuts) total += c;
  std::vector<long long> na(total / g.K), de(total / g.K);
  for (int np : cuts) {
    TilePlan tp;
    if (!tile_plan_make(g, w, q0 % g.K, np, vec, sizeof(T), &tp)) { fprintf(stderr, "no plan\n"); return 4; }
    std::vector<int> written(S, 0);
    for (int tile = 0; tile < tp.cx * tp.cy * tp.cz; tile++) {
      const TileBox bx = tile_box(tp, tile);
      const uint32_t packs = (uint32_t)tp.gl.K * (uint32_t)(tp.gl.Mp / 4);
      // heap copies of the exact LDS size; whole words for the vector steps
      std::vector<Words<4>> lw((size_t)(tile_lds(tp) + 15) / 16);
      T *ls = reinterpret_cast<T *>(lw.data());
      int32_t *lk = reinterpret_cast<int32_t *>(reinterpret_cast<char *>(lw.data()) + tp.spin_bytes);
      for (uint32_t i = 0; i < packs; i++) tile_load<LAT, T>(s[from].data(), k[from].data(), g, tp, bx, i, ls, lk);
      for (int p = 0; p < np; p++) {
        const int c = (tp.c0 + p) % g.K;
        for (uint32_t i = 0; i < tp.pass[p].items; i++) {
          Counts cnt;
          if (vec == 1)
            cnt = tile_event<LAT, T, TWO, APP>(ls, lk, g, r, r.thr, tp, bx, tp.pass[p], c, i);
          else if (LAT == SPK_HIP_SQ_8N || LAT == SPK_HIP_SC_26N)
            cnt = c & 1 ? tile_events<LAT, T, TWO, 1>(ls, lk, g, r, r.thr, tp, bx, tp.pass[p], c, i)
                        : tile_events<LAT, T, TWO, 0>(ls, lk, g, r, r.thr, tp, bx, tp.pass[p], c, i);
          else
            cnt = tile_events<LAT, T, TWO, -1>(ls, lk, g, r, r.thr, tp, bx, tp.pass[p], c, i);
          na[(q0 + p) / g.K] += cnt.nacc;
          de[(q0 + p) / g.K] += cnt.de;
        }
      }
      std::vector<T> before = s[!from];
      std::vector<int32_t> kb = k[!from];
      // every real site is stored by exactly one box
      std::fill(s[!from].begin(), s[!from].end(), (T)~(T)0);
      std::fill(k[!from].begin(), k[!from].end(), -1);
      for (uint32_t i = 0; i < tile_store_items<LAT>(tp); i++)
        tile_store<LAT, T>(s[!from].data(), k[!from].data(), g, tp, bx, i, ls, lk);
      for (long long p = 0; p < S; p++) {
        if (k[!from][p] == -1) s[!from][p] = before[p], k[!from][p] = kb[p];
        else written[p]++;
      }
    }
    long long once = 0;
    for (int v : written) once += v == 1;
    if (once != N) { fprintf(stderr, "boxes store %lld of %lld sites once\n", once, N); return 5; }
    from = !from;
    q0 += np;
  }
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    sn[t] = (int32_t)s[from][p], kn[t] = k[from][p];
  }
  f = fopen(out, "wb");
  if (!f) return 6;
  fwrite(sn.data(), 4, N, f);
  fwrite(kn.data(), 4, N, f);
  for (size_t i = 0; i < na.size(); i++) {
    fwrite(&na[i], 8, 1, f);
    fwrite(&de[i], 8, 1, f);
  }
  fclose(f);
  return 0;
}

template <int LAT>
static int with_type(int vec, int st, int app, const int *n, int q, double kt, const int (&w)[3], const std::vector<int> &cuts,
                     const char *in, const char *out) {
  auto with_app = [&]<typename T>() {
    if (app == SPK_HIP_POTTS_NEIGH) return run<LAT, T, false, SPK_HIP_POTTS_NEIGH>(vec, app, n, q, kt, w, cuts, in, out);
    if (app == SPK_HIP_POTTS_NEIGHONLY)
      return run<LAT, T, false, SPK_HIP_POTTS_NEIGHONLY>(vec, app, n, q, kt, w, cuts, in, out);
    if constexpr (sizeof(T) == 1) {
      if (app == SPK_HIP_ISING_SINGLE) return run<LAT, T, true, SPK_HIP_ISING_SINGLE>(vec, app, n, q, kt, w, cuts, in, out);
      if (app == SPK_HIP_ISING || q == 2) return run<LAT, T, true, SPK_HIP_POTTS>(vec, app, n, q, kt, w, cuts, in, out);
    }
    return run<LAT, T, false, SPK_HIP_POTTS>(vec, app, n, q, kt, w, cuts, in, out);
  };
  if (st == 0) return with_app.template operator()<uint8_t>();
  if (st == 1) return with_app.template operator()<uint16_t>();
  return with_app.template operator()<int32_t>();
}

int main(int argc, char **argv) {
  if (argc != 16) { fprintf(stderr, "usage: app lat nx ny nz q kT stype vec wx wy wz cuts in out\n"); return 1; }
  const int app = atoi(argv[1]), lat = atoi(argv[2]), n[3] = {atoi(argv[3]), atoi(argv[4]), atoi(argv[5])};
  const int q = atoi(argv[6]), st = atoi(argv[8]), vec = atoi(argv[9]), w[3] = {atoi(argv[10]), atoi(argv[11]), atoi(argv[12])};
  const double kt = atof(argv[7]);
  std::vector<int> cuts;
  for (char *p = strtok(argv[13], ","); p; p = strtok(nullptr, ",")) cuts.push_back(atoi(p));
  switch (lat) {
    case SPK_HIP_SQ_4N: return with_type<SPK_HIP_SQ_4N>(vec, st, app, n, q, kt, w, cuts, argv[14], argv[15]);
    case SPK_HIP_SQ_8N: return with_type<SPK_HIP_SQ_8N>(vec, st, app, n, q, kt, w, cuts, argv[14], argv[15]);
    case SPK_HIP_SC_6N: return with_type<SPK_HIP_SC_6N>(vec, st, app, n, q, kt, w, cuts, argv[14], argv[15]);
    default: return with_type<SPK_HIP_SC_26N>(vec, st, app, n, q, kt, w, cuts, argv[14], argv[15]);
  }
}
