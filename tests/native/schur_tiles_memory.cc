// What the host construction of the reduced camera system's structure
// allocates, for a banded system of a given number of rows: bytes in all, and
// the most held at once. With "check" the row structure is compared with a
// plain restatement.
#include <atomic>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <new>
#include <random>
#include <string>
#include <vector>

#include "ba_tiles.h"

static std::atomic<long long> g_total{0}, g_live{0}, g_peak{0};

static void* counted(std::size_t n) {
  char* p = static_cast<char*>(std::malloc(n + 16));
  if (!p) throw std::bad_alloc();
  *reinterpret_cast<std::size_t*>(p) = n;
  g_total += (long long)n;
  const long long live = g_live += (long long)n;
  for (long long peak = g_peak; live > peak && !g_peak.compare_exchange_weak(peak, live);) {
  }
  return p + 16;
}
static void release(void* p) {
  if (!p) return;
  char* q = static_cast<char*>(p) - 16;
  g_live -= (long long)*reinterpret_cast<std::size_t*>(q);
  std::free(q);
}
void* operator new(std::size_t n) { return counted(n); }
void* operator new[](std::size_t n) { return counted(n); }
void operator delete(void* p) noexcept { release(p); }
void operator delete[](void* p) noexcept { release(p); }
void operator delete(void* p, std::size_t) noexcept { release(p); }
void operator delete[](void* p, std::size_t) noexcept { release(p); }

int main(int argc, char** argv) {
  const int Pvar = std::atoi(argv[1]), per = std::atoi(argv[2]);
  const bool check = argc > 3 && !std::strcmp(argv[3], "check");
  const int L = Pvar * per;
  std::mt19937 rng(1);
  std::vector<int32_t> obs_lm, row_of;
  std::vector<int32_t> anchor(L);
  for (int l = 0; l < L; ++l) {
    const int first = l / per;
    anchor[l] = rng() % 4 ? first : -1;
    for (int q = 0; q < 6; ++q) {
      const int r = std::min(Pvar - 1, first + (int)(rng() % 12));
      if (r == anchor[l]) continue;
      row_of.push_back(r);
      obs_lm.push_back(l);
    }
  }
  std::vector<int32_t> inc_ptr(Pvar + 1, 0), inc;
  for (int r : row_of) inc_ptr[r + 1]++;
  for (int l = 0; l < L; ++l)
    if (anchor[l] >= 0) inc_ptr[anchor[l] + 1]++;
  for (int i = 0; i < Pvar; ++i) inc_ptr[i + 1] += inc_ptr[i];
  inc.resize(inc_ptr[Pvar]);
  {
    std::vector<int32_t> fill(inc_ptr.begin(), inc_ptr.end() - 1);
    for (size_t o = 0; o < row_of.size(); ++o) inc[fill[row_of[o]]++] = (int32_t)o;
    for (int l = 0; l < L; ++l)
      if (anchor[l] >= 0) inc[fill[anchor[l]]++] = -1 - l;
  }
  mlba::SchurTiles st;
  mlba::SchurRows rows;
  std::string err;
  const long long live0 = g_live;
  g_total = 0;
  g_peak = live0;
  if (!mlba::build_schur_tiles(Pvar, L, inc_ptr.data(), inc.data(), obs_lm.data(), &st, &err) ||
      !mlba::build_schur_rows(Pvar, L, st, &rows, &err)) {
    std::printf("%s\n", err.c_str());
    return 3;
  }
  std::printf("%lld %lld\n", (long long)g_total, (long long)(g_peak - live0));
  if (!check) return 0;
  // Pairs of incidences of one landmark, by rows.
  std::vector<std::vector<int32_t>> lm_rows(L);
  for (int i = 0; i < Pvar; ++i)
    for (int k = inc_ptr[i]; k < inc_ptr[i + 1]; ++k) lm_rows[inc[k] >= 0 ? obs_lm[inc[k]] : -1 - inc[k]].push_back(i);
  std::map<std::pair<int, int>, long long> pairs;
  for (int i = 0; i < Pvar; ++i) pairs[{i, i}];
  for (const auto& r : lm_rows)
    for (int a : r)
      for (int b : r) pairs[{a, b}]++;
  size_t at = 0, up = 0;
  long long sum = 0;
  for (const auto& e : pairs) {
    const int i = e.first.first, j = e.first.second;
    if (at >= rows.col.size() || rows.col[at] != j || at < (size_t)rows.row_ptr[i] || at >= (size_t)rows.row_ptr[i + 1])
      return 4;
    if (i == j && (size_t)rows.diag_pos[i] != at) return 5;
    if (j >= i) {
      if (up >= rows.upper_pairs.size() || rows.upper_pairs[up] != e.second) return 6;
      ++up;
      sum += e.second;
    }
    ++at;
  }
  if (at != rows.col.size() || up != rows.upper_pairs.size() || sum != rows.pairs) return 7;
  return 0;
}
