// spk_emul_neigh.hip -- host-only emulation of the packed potts/neigh and
// potts/neighonly pass (spk_neigh.h), for CPU tests: the kernel's own code, a
// pack at a time, under AddressSanitizer.  Test infrastructure; not part of the
// library.
//
// usage: spk_emul_neigh app lat nx ny nz nspins kT nsweeps stype in.bin out.bin
//   stype: 0 uint8, 1 uint16 spin storage
//   in.bin : int32 spin[N], int32 seed[N] (reference order)
//   out.bin: int32 spin[N], int32 seed[N], then per sweep int64 naccept and
//            sum of ef - ei
#include <cstdio>
#include <cstdlib>
#include <vector>

#include "spk_neigh.h"

using namespace spk;

extern "C" int spk_hip_metropolis_table(double, int, double *, int32_t *);

template <int LAT, typename T, int APP>
static int run(const int *n, int q, double kt, int nsw, const char *in, const char *out) {
  Geom g{};
  geom_init(g, LAT, n[0], n[1], n[2]);
  const long long N = (long long)n[0] * n[1] * n[2], S = (long long)g.K * g.Mp;
  Rule r{};
  r.app = APP, r.nspins = q, r.zero_t = kt == 0.0;
  int32_t thr[27];
  spk_hip_metropolis_table(kt > 0 ? kt : 1.0, maxneigh_of(LAT), nullptr, thr);
  r.half = thr[0];
  for (int d = 1; d <= maxneigh_of(LAT); d++) r.thr[d] = thr[d];
  std::vector<int32_t> sn(N), kn(N);
  FILE *f = fopen(in, "rb");
  if (!f || fread(sn.data(), 4, N, f) != (size_t)N || fread(kn.data(), 4, N, f) != (size_t)N) return 2;
  fclose(f);
  std::vector<T> s(S, (T)-1);   // pad slots: values that no site holds
  std::vector<int32_t> k(S, 0x7ffffff0);
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    s[p] = (T)sn[t], k[p] = kn[t];
  }
  std::vector<long long> na(nsw), de(nsw);
  for (int sw = 0; sw < nsw; sw++)
    for (int c = 0; c < g.K; c++)
      for (int t = 0; t < g.Mp / 4; t++) {
        int a0, b, e;
        pack_site(g, (uint32_t)t, a0, b, e);
        const Counts x = c & 1 ? neigh_pack<LAT, T, APP, uint32_t, 1>(s.data(), k.data(), g, r, r.thr, c, a0, b, e)
                               : neigh_pack<LAT, T, APP, int64_t, 0>(s.data(), k.data(), g, r, r.thr, c, a0, b, e);
        na[sw] += x.nacc, de[sw] += x.de;
      }
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % n[0], (t / n[0]) % n[1], t / ((long long)n[0] * n[1]));
    sn[t] = (int32_t)s[p], kn[t] = k[p];
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
  if (argc != 12) { fprintf(stderr, "usage: app lat nx ny nz q kT nsweeps stype in out\n"); return 1; }
  const int app = atoi(argv[1]), lat = atoi(argv[2]), n[3] = {atoi(argv[3]), atoi(argv[4]), atoi(argv[5])};
  const int q = atoi(argv[6]);
  if (q > kNeighMaxQ) return 4;
  auto types = [&]<int LAT, int APP>() {
    return atoi(argv[9]) == 0 ? run<LAT, uint8_t, APP>(n, q, atof(argv[7]), atoi(argv[8]), argv[10], argv[11])
                              : run<LAT, uint16_t, APP>(n, q, atof(argv[7]), atoi(argv[8]), argv[10], argv[11]);
  };
  auto apps = [&]<int LAT>() {
    return app == SPK_HIP_POTTS_NEIGH ? types.template operator()<LAT, SPK_HIP_POTTS_NEIGH>()
                                      : types.template operator()<LAT, SPK_HIP_POTTS_NEIGHONLY>();
  };
  return lat == SPK_HIP_SQ_8N ? apps.template operator()<SPK_HIP_SQ_8N>() : apps.template operator()<SPK_HIP_SC_26N>();
}
