// Builds the decomposition of a random system on all CPUs and again bound to
// one, and compares every array.
#include <sched.h>

#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <random>
#include <string>
#include <vector>

#include "ba_tiles.h"

template <class V>
static bool same(const char* name, const V& a, const V& b) {
  const bool ok = a.size() == b.size() &&
                  (a.empty() || std::memcmp(a.data(), b.data(), a.size() * sizeof(a[0])) == 0);
  if (!ok) std::printf("%s differs (%zu, %zu entries)\n", name, a.size(), b.size());
  return ok;
}

int main(int argc, char** argv) {
  const int Pvar = std::atoi(argv[1]), L = std::atoi(argv[2]);
  std::mt19937 rng((unsigned)std::atoi(argc > 3 ? argv[3] : "1"));
  std::vector<std::vector<int32_t>> rows(Pvar);
  std::vector<int32_t> obs_lm;
  for (int l = 0; l < L; ++l) {
    const int center = (int)(rng() % Pvar), span = 1 + (int)(rng() % 30), k = (int)(rng() % 12);
    const int anchor = rng() % 4 ? center : -1;
    for (int q = 0; q < k; ++q) {
      const int r = (center + (int)(rng() % span)) % Pvar;
      if (r == anchor) continue;
      rows[r].push_back((int32_t)obs_lm.size());
      obs_lm.push_back(l);
    }
    if (anchor >= 0) rows[anchor].push_back(-1 - l);
  }
  std::vector<int32_t> inc_ptr(Pvar + 1, 0), inc;
  for (int i = 0; i < Pvar; ++i) {
    inc.insert(inc.end(), rows[i].begin(), rows[i].end());
    inc_ptr[i + 1] = (int32_t)inc.size();
  }
  mlba::SchurTiles st[2];
  for (int pass = 0; pass < 2; ++pass) {
    if (pass == 1) {
      cpu_set_t one;
      CPU_ZERO(&one);
      CPU_SET(sched_getcpu(), &one);
      if (sched_setaffinity(0, sizeof(one), &one) != 0) return 2;
    }
    std::string err;
    if (!mlba::build_schur_tiles(Pvar, L, inc_ptr.data(), inc.data(), obs_lm.data(), &st[pass], &err)) {
      std::printf("%s\n", err.c_str());
      return 3;
    }
  }
  const mlba::SchurTiles &a = st[0], &b = st[1];
  bool ok = a.nbands == b.nbands && a.visits == b.visits && a.staged == b.staged;
  ok = same("g_row", a.g_row, b.g_row) && same("g_inc_ptr", a.g_inc_ptr, b.g_inc_ptr) && same("g_inc", a.g_inc, b.g_inc) &&
       same("lm_g_ptr", a.lm_g_ptr, b.lm_g_ptr) && same("slots", a.slots, b.slots) && same("batches", a.batches, b.batches) &&
       same("batch_off", a.batch_off, b.batch_off) && same("pairs", a.pairs, b.pairs) && same("segs", a.segs, b.segs) &&
       same("seg_thread", a.seg_thread, b.seg_thread) && same("seg_block", a.seg_block, b.seg_block) &&
       same("tile_key", a.tile_key, b.tile_key) && same("tile_seg", a.tile_seg, b.tile_seg) && ok;
  std::printf("%d rows, %d landmarks, %zu incidences, %zu batches: %s\n", Pvar, L, inc.size(), a.batches.size() / 4,
              ok ? "same" : "different");
  return ok ? 0 : 1;
}
