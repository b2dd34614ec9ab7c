// spk_emul_pair.hip -- host-only emulation of the two-sweep bit-plane kernel
// (k_sweep_bits_pair, spk_bits.h) in every band and stage it is launched
// with, for CPU tests: the kernel's own steps, thread by thread, under
// AddressSanitizer.  Test infrastructure; not part of the library.
//
// usage: spk_emul_pair app nx ny kT band stage pairs in.bin out.bin
//   app: SPK_HIP_ISING or SPK_HIP_ISING_SINGLE; pairs: two-sweep launches
//   in.bin : int32 spin[N], int32 seed[N] (reference order)
//   out.bin: int32 spin[N], int32 seed[N], then per sweep int64 naccept and
//            sum of ef - ei
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <vector>

#include "spk_bits.h"

using namespace spk;

extern "C" int spk_hip_metropolis_table(double, int, double *, int32_t *);

template <bool SINGLE, bool FULL, int BAND, int STAGE>
static void launch(const std::vector<uint32_t> &bits, const std::vector<int32_t> &sseed, std::vector<uint32_t> &bits2,
                   std::vector<int32_t> &sseed2, const Geom &g, const BitGeom &bg, const Rule &r, long long (&row)[2][2]) {
  using Shape = PairShape<BAND, STAGE>;
  auto L = std::make_unique<PairLdsOf<BAND>>();
  std::vector<Words<4>> regs((size_t)kPairThreads * (Shape::slots0 + Shape::slots1) * 2);
  auto reg = [&](int c, int grp, uint32_t tau, int j) {
    return &regs[((size_t)(grp * STAGE + tau) * (Shape::slots0 + Shape::slots1) + (c ? Shape::slots0 : 0) + j) * 2];
  };
  const uint32_t on = 4u * (uint32_t)bg.pw;
  if (on > (uint32_t)STAGE) { fprintf(stderr, "a row does not fit the stage\n"); exit(30); }
  for (int y0 = 0; y0 < g.hy; y0 += BAND) {
    memset(L.get(), 0xa5, sizeof *L);
    for (int i = 0; i < 2 * Shape::rows * bg.pw; i++) {
      int c, lr, w;
      const int64_t at = pair_plane_src<Shape>(g, bg, y0, i, c, lr, w);
      if (lr >= Shape::rows || w >= bg.pw) { fprintf(stderr, "plane word out of range\n"); exit(31); }
      L->planes[c][lr][w] = bits.at(at);
    }
    for (int grp = 0; grp < Shape::groups; grp++)
      for (uint32_t tau = 0; tau < (uint32_t)STAGE; tau++)
        for (int c = 0; c < 2; c++)
          for (int j = 0; j < (c ? Shape::slots1 : Shape::slots0); j++) {
            const int rho = std::min(pair_slot_row<Shape>(y0, c, grp, j), y0 + BAND + 2 - c);
            for (int h = 0; h < 2; h++) {
              const Words<4> *p = pair_seeds<FULL>(sseed.data(), bg, c, pair_row(rho, g.hy), tau < on ? tau : 0u, h);
              const int64_t at = reinterpret_cast<const int32_t *>(p) - sseed.data();
              if (at < 0 || at + 4 > (int64_t)sseed.size()) { fprintf(stderr, "seeds out of range\n"); exit(32); }
              reg(c, grp, tau, j)[h] = *p;
            }
          }
    for (int p = 0; p < 4; p++) {
      const int c = p & 1, slots = c ? Shape::slots1 : p == 2 ? Shape::slots2 : Shape::slots0;
      // every row of the pass is some group's
      std::vector<int> seen(BAND + 6, 0);
      for (int grp = 0; grp < Shape::groups; grp++)
        for (int j = 0; j < slots; j++) {
          const int rho = pair_slot_row<Shape>(y0, c, grp, j);
          if (pair_pass_row<Shape>(y0, p, rho)) seen.at(rho - (y0 - 3))++;
        }
      for (int k = p; k < BAND + 6 - p; k++)
        if (seen[k] != 1) { fprintf(stderr, "pass %d misses a row\n", p); exit(33); }
      for (int grp = 0; grp < Shape::groups; grp++)
        for (uint32_t tau = 0; tau < on; tau++) {
          const PairLane ln = pair_lane<FULL>(g, bg, pair_slot_row<Shape>(y0, 0, grp, 0), 0, grp, tau);
          for (int j = 0; j < slots; j++) {
            const int rho = pair_slot_row<Shape>(y0, c, grp, j);
            if (!pair_pass_row<Shape>(y0, p, rho)) continue;
            if (pair_side<true>(g, rho, c, grp) != pair_side<false>(g, rho, c, grp)) { fprintf(stderr, "side\n"); exit(34); }
            const PairWords pw = pair_words(*L, y0, p, rho, grp, ln);
            PairCounts a;
            pair_thread<SINGLE, FULL>(*L, g, bg, r, y0, p, rho, grp, tau, ln, pw,
                                      *reinterpret_cast<Words<4>(*)[2]>(reg(c, grp, tau, j)), sseed2.data(), a);
            const Counts n = pair_counts(a);
            row[p >> 1][0] += n.nacc, row[p >> 1][1] += n.de;
          }
        }
    }
    for (int i = 0; i < 2 * BAND * bg.pw; i++) pair_store_plane(*L, bits2.data(), g, bg, y0, i);
  }
}

int main(int argc, char **argv) {
  if (argc != 10) { fprintf(stderr, "usage: app nx ny kT band stage pairs in out\n"); return 1; }
  const int app = atoi(argv[1]), nx = atoi(argv[2]), ny = atoi(argv[3]), band = atoi(argv[5]), stage = atoi(argv[6]),
            pairs = atoi(argv[7]);
  const double kt = atof(argv[4]);
  Geom g{};
  geom_init(g, SPK_HIP_SQ_4N, nx, ny, 1);
  if (!pair_fits(g)) { fprintf(stderr, "does not fit\n"); return 4; }
  Rule r{};
  r.app = app, r.nspins = 2, r.zero_t = kt == 0.0;
  int32_t thr[5];
  spk_hip_metropolis_table(kt > 0 ? kt : 1.0, 4, nullptr, thr);
  r.half = thr[0];
  for (int d = 1; d <= 4; d++) r.thr[d] = thr[d];
  const long long N = (long long)nx * ny, S = (long long)g.K * g.Mp;
  std::vector<int32_t> sn(N), kn(N), k(S, 1);
  std::vector<uint8_t> s(S, 1);
  FILE *f = fopen(argv[8], "rb");
  if (!f || fread(sn.data(), 4, N, f) != (size_t)N || fread(kn.data(), 4, N, f) != (size_t)N) return 2;
  fclose(f);
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % nx, t / nx, 0);
    s[p] = (uint8_t)sn[t], k[p] = kn[t];
  }
  const BitGeom bg = bit_geom(g, 8);
  const int64_t words = (int64_t)g.hy * bg.pw;
  std::vector<uint32_t> bits(2 * words), bits2(2 * words, 0xdeadbeefu);
  std::vector<int32_t> sseed(2 * bg.seedc), sseed2(2 * bg.seedc, 1);
  for (int64_t q = 0; q < 2 * words; q++) bits[q] = bits_pack_word(s.data(), g, (int)(q / words), (int)(q % words / bg.pw), (int)(q % words % bg.pw));
  for (int64_t X = 0; X < bg.seedc / 2; X++) bits_seed_group_in(k.data(), g, bg, X, sseed.data());
  const bool full = bg.pw == kPairMaxPw && bg.r == 31, single = app == SPK_HIP_ISING_SINGLE;
  std::vector<long long> out;
  for (int w = 0; w < pairs; w++) {
    long long row[2][2] = {};
    auto go = [&]<int BAND, int STAGE>() {
      if (STAGE == 4 * kPairMaxPw && full)
        single ? launch<true, STAGE == 256, BAND, STAGE>(bits, sseed, bits2, sseed2, g, bg, r, row)
               : launch<false, STAGE == 256, BAND, STAGE>(bits, sseed, bits2, sseed2, g, bg, r, row);
      else
        single ? launch<true, false, BAND, STAGE>(bits, sseed, bits2, sseed2, g, bg, r, row)
               : launch<false, false, BAND, STAGE>(bits, sseed, bits2, sseed2, g, bg, r, row);
    };
    auto with_stage = [&]<int BAND>() {
      if (stage == 64) go.template operator()<BAND, 64>();
      else if (stage == 128) go.template operator()<BAND, 128>();
      else go.template operator()<BAND, 256>();
    };
    if (band == 4) with_stage.template operator()<4>();
    else if (band == 8) with_stage.template operator()<8>();
    else if (band == 12) with_stage.template operator()<12>();
    else with_stage.template operator()<16>();
    std::swap(bits, bits2);
    std::swap(sseed, sseed2);
    for (auto &x : row) out.push_back(x[0]), out.push_back(x[1]);
  }
  for (int64_t q = 0; q < 2 * words; q++) bits_unpack_word(s.data(), g, (int)(q / words), (int)(q % words / bg.pw), (int)(q % words % bg.pw), bits[q]);
  for (int64_t X = 0; X < bg.seedc / 2; X++) bits_seed_group_out(sseed.data(), g, bg, X, k.data());
  for (long long t = 0; t < N; t++) {
    const long long p = blocked_index(g, t % nx, t / nx, 0);
    sn[t] = s[p], kn[t] = k[p];
  }
  f = fopen(argv[9], "wb");
  if (!f) return 6;
  fwrite(sn.data(), 4, N, f);
  fwrite(kn.data(), 4, N, f);
  fwrite(out.data(), 8, out.size(), f);
  fclose(f);
  return 0;
}
