// ba_tiles.cc -- host construction of the reduced-camera-system work
// decomposition (factor blocks, tile visits, batches, pair lists, segments).
#include "ba_tiles.h"

#include <algorithm>
#include <atomic>
#include <limits>
#include <thread>

namespace mlba {

namespace {

struct Run {
  int32_t band, g, n;  // band, first factor block, blocks
};

}  // namespace

bool parallel_ranges(int64_t n, int64_t piece, const std::function<void(int64_t, int64_t, int)>& body) {
  if (n <= 0) return true;
  piece = std::max<int64_t>(piece, 1);
  std::atomic<int64_t> next{0};
  std::atomic<bool> ok{true};
  auto work = [&](int thread) {
    for (int64_t b = next.fetch_add(piece); b < n; b = next.fetch_add(piece)) {
      try {
        body(b, std::min(n, b + piece), thread);
      } catch (...) {
        ok = false;
      }
    }
  };
  const int64_t pieces = (n + piece - 1) / piece;
  const int64_t hw = std::max(1u, std::thread::hardware_concurrency());
  std::vector<std::thread> pool;
  try {
    const int64_t extra = std::min<int64_t>({pieces, hw, kMaxHostThreads}) - 1;
    pool.reserve((size_t)std::max<int64_t>(extra, 0));
    for (int64_t t = 0; t < extra; ++t) pool.emplace_back(work, (int)t + 1);
  } catch (...) {
    // Fewer threads than wanted: the ones that run take all pieces.
  }
  work(0);
  for (std::thread& t : pool) t.join();
  return ok;
}

bool build_schur_tiles(int32_t Pvar, int32_t L, const int32_t* inc_ptr, const int32_t* inc,
                       const int32_t* obs_landmark, SchurTiles* out, std::string* err) {
  SchurTiles& T = *out;
  T = SchurTiles();
  const int64_t n_inc = Pvar > 0 ? inc_ptr[Pvar] : 0;
  auto lm_of = [&](int32_t code) { return code >= 0 ? obs_landmark[code] : -1 - code; };
  // Incidences of each landmark in row order (the row lists are row-major).
  std::vector<int32_t> inc_row(n_inc), lm_ptr(L + 1, 0), lm_list(n_inc);
  for (int i = 0; i < Pvar; ++i)
    for (int k = inc_ptr[i]; k < inc_ptr[i + 1]; ++k) inc_row[k] = i;
  for (int64_t k = 0; k < n_inc; ++k) lm_ptr[lm_of(inc[k]) + 1]++;
  for (int l = 0; l < L; ++l) lm_ptr[l + 1] += lm_ptr[l];
  {
    std::vector<int32_t> fill(lm_ptr.begin(), lm_ptr.end() - 1);
    for (int64_t k = 0; k < n_inc; ++k) lm_list[fill[lm_of(inc[k])]++] = (int32_t)k;
  }
  // Factor blocks: the incidences of one landmark in one row. Landmarks are
  // counted first, so that each has its place and pieces of them are filled
  // independently.
  constexpr int64_t kPiece = 4096;  // landmarks
  UnsetVector<int32_t>& lm_g = T.lm_g_ptr;
  lm_g.resize((size_t)L + 1);
  lm_g[0] = 0;
  std::atomic<bool> shared{false};
  bool ok = parallel_ranges(L, kPiece, [&](int64_t l0, int64_t l1, int) {
    for (int64_t l = l0; l < l1; ++l) {
      int n = 0, last = -1;
      for (int m = lm_ptr[l]; m < lm_ptr[l + 1]; ++m) {
        const int row = inc_row[lm_list[m]];
        // An anchor incidence is alone in its row: the anchor vertex's own
        // observations of the landmark do not couple its pose.
        if (row == last && (inc[lm_list[m]] < 0 || inc[lm_list[m - 1]] < 0)) shared = true;
        n += row != last;
        last = row;
      }
      lm_g[l + 1] = n;
    }
  });
  if (shared) {
    *err = "internal: an anchor incidence shares its row with observations";
    return false;
  }
  for (int l = 0; l < L; ++l) lm_g[l + 1] += lm_g[l];
  const int64_t n_g = lm_g[L];
  T.g_row.resize((size_t)n_g);
  T.g_inc_ptr.resize((size_t)n_g + 1);
  T.g_inc.resize((size_t)n_inc);
  T.g_inc_ptr[n_g] = (int32_t)n_inc;
  ok = ok && parallel_ranges(L, kPiece, [&](int64_t l0, int64_t l1, int) {
    for (int64_t l = l0; l < l1; ++l) {
      int g = lm_g[l], last = -1;
      for (int m = lm_ptr[l]; m < lm_ptr[l + 1]; ++m) {
        const int k = lm_list[m];
        if (inc_row[k] != last) {
          last = inc_row[k];
          T.g_row[g] = last;
          T.g_inc_ptr[g++] = m;
        }
        T.g_inc[m] = inc[k];
      }
    }
  });
  const int64_t nb = (Pvar + kTileBand - 1) / kTileBand;
  T.nbands = (int32_t)nb;
  // The runs of a landmark's factor blocks in one band.
  auto landmark_runs = [&](int64_t l, std::vector<Run>& runs) {
    runs.clear();
    for (int g = lm_g[l]; g < lm_g[l + 1]; ++g) {
      const int band = T.g_row[g] / kTileBand;
      if (runs.empty() || runs.back().band != band) runs.push_back(Run{band, g, 0});
      runs.back().n++;
    }
  };
  // Visits (landmark, first block in I, first in J, blocks in I, in J),
  // grouped by tile in (I, J) order, landmarks ascending in a tile (a
  // landmark visits a tile at most once; only visited tiles exist): a stable
  // counting sort over pieces of the landmarks, each with counts of its own. By
  // tile, unless such counts were more than four a landmark: a long map has far
  // more pairs of bands than visited tiles (400000 vertices: 5 GB of counts). Then
  // by I, and by J within each I.
  struct Visit {
    int32_t I, J, l, gi, gj;
    uint8_t ni, nj;  // <= kTileBand
  };
  const int64_t pieces = std::max<int64_t>(1, std::min<int64_t>(16, (L + kPiece - 1) / kPiece));
  const int64_t span = (L + pieces - 1) / pieces;
  const bool by_tile = pieces * nb * nb <= 4 * (int64_t)L;
  const int64_t keys = by_tile ? nb * nb : nb;
  auto key_of = [&](int64_t I, int64_t J) { return by_tile ? I * nb + J : I; };
  std::vector<int64_t> at((size_t)(pieces * keys), 0);  // visits, then the place of the next, by piece and key
  ok = ok && parallel_ranges(pieces, 1, [&](int64_t p0, int64_t p1, int) {
    std::vector<Run> runs;
    for (int64_t q = p0; q < p1; ++q)
      for (int64_t l = q * span; l < std::min<int64_t>(L, (q + 1) * span); ++l) {
        landmark_runs(l, runs);
        for (size_t a = 0; a < runs.size(); ++a)
          for (size_t b = a; b < runs.size(); ++b) at[(size_t)(q * keys + key_of(runs[a].band, runs[b].band))]++;
      }
  });
  std::vector<int64_t> key_end((size_t)keys, 0);
  int64_t n_visits = 0;
  for (int64_t k = 0; k < keys; ++k) {
    for (int64_t q = 0; q < pieces; ++q) {
      const int64_t n = at[(size_t)(q * keys + k)];
      at[(size_t)(q * keys + k)] = n_visits;
      n_visits += n;
    }
    key_end[(size_t)k] = n_visits;
  }
  UnsetVector<Visit> visits;
  visits.resize((size_t)n_visits);
  ok = ok && parallel_ranges(pieces, 1, [&](int64_t p0, int64_t p1, int) {
    std::vector<Run> runs;
    for (int64_t q = p0; q < p1; ++q)
      for (int64_t l = q * span; l < std::min<int64_t>(L, (q + 1) * span); ++l) {
        landmark_runs(l, runs);
        for (size_t a = 0; a < runs.size(); ++a)
          for (size_t b = a; b < runs.size(); ++b)
            visits[(size_t)at[(size_t)(q * keys + key_of(runs[a].band, runs[b].band))]++] =
                Visit{runs[a].band, runs[b].band, (int32_t)l, runs[a].g, runs[b].g, (uint8_t)runs[a].n,
                      (uint8_t)(a == b ? 0 : runs[b].n)};
      }
  });
  if (!by_tile) {
    UnsetVector<Visit> by_band;
    by_band.swap(visits);
    visits.resize((size_t)n_visits);
    std::vector<std::vector<int64_t>> place(kMaxHostThreads);  // by thread: visits of J, then the place of the next
    ok = ok && parallel_ranges(nb, 1, [&](int64_t i0, int64_t i1, int thread) {
      std::vector<int64_t>& p = place[thread];
      if (p.empty()) p.resize((size_t)nb, 0);
      std::vector<int32_t> touched;
      for (int64_t i = i0; i < i1; ++i) {
        const int64_t begin = i ? key_end[i - 1] : 0, end = key_end[i];
        touched.clear();
        for (int64_t k = begin; k < end; ++k)
          if (p[by_band[k].J]++ == 0) touched.push_back(by_band[k].J);
        std::sort(touched.begin(), touched.end());
        int64_t next = begin;
        for (int32_t J : touched) {
          const int64_t n = p[J];
          p[J] = next;
          next += n;
        }
        for (int64_t k = begin; k < end; ++k) visits[(size_t)p[by_band[k].J]++] = by_band[k];
        for (int32_t J : touched) p[J] = 0;
      }
    });
  }
  if (!ok) {
    *err = "host allocation failed";
    return false;
  }
  T.visits = n_visits;
  // A segment runs its batches one after the other, and about kSegmentTarget
  // work-groups run at once (two on each of 256 CUs): the segments are sized
  // for whole rounds of them, kSegmentSlots staged blocks or up to twice that
  // each, and a system too small for one round of those is cut into one round
  // of shorter ones. Build of S (two kernels) with segments of 5120 blocks and
  // cut so: 10 keyframes 130 -> 27 us (2 -> 39 segments), 25 keyframes 203 ->
  // 47, 60 keyframes 206 -> 74; with today's kernel 200 keyframes 234 -> 190,
  // 300 keyframes 344 -> 294, 500 and more unchanged.
  int64_t staged_all = 0;
  for (const Visit& v : visits) staged_all += v.ni + v.nj;
  const int64_t rounds = std::max<int64_t>(1, staged_all / ((int64_t)kSegmentTarget * kSegmentSlots));
  const int64_t segment_slots = staged_all / (kSegmentTarget * rounds);
  auto is_anchor = [&](int g) { return T.g_inc[T.g_inc_ptr[g]] < 0; };
  auto pairs_of = [](const Visit& v) { return v.nj ? v.ni * v.nj : v.ni * (v.ni + 1) / 2; };
  auto same_tile = [&](int64_t v, const Visit& of) { return v < n_visits && visits[v].I == of.I && visits[v].J == of.J; };
  // Batches (LDS-sized groups of visits) and segments (runs of batches of one
  // tile) of every visited tile, counted first: each tile's slots, pairs
  // (batches start on a 32-bit word), batches and segments then have their
  // place, and the tiles are filled independently of one another.
  struct Tile {
    int64_t v0, v1;                   // visits
    int64_t slot, pair, batch, seg;   // first of each
  };
  std::vector<Tile> tiles;
  int64_t n_slots = 0, n_pairs = 0, n_batches = 0, n_segs = 0;
  for (int64_t v = 0; v < n_visits;) {
    const Visit of = visits[v];
    tiles.push_back(Tile{v, v, n_slots, n_pairs, n_batches, n_segs});
    int64_t seg_slots = 0, seg_batches = 0;
    bool open = false;
    while (same_tile(v, of)) {
      int64_t slots = 0, np = 0;
      for (; same_tile(v, of); ++v) {
        const int c = visits[v].ni + visits[v].nj;
        if (slots + c > kBatchSlots) break;
        slots += c;
        np += pairs_of(visits[v]);
      }
      // A visit has at most 16 x 16 pairs over 32 slots (8 per slot), or
      // 16 x 17 / 2 over 16 on a diagonal tile (8.5 per slot).
      if (np > kBatchPairs) {
        *err = "internal: a Schur batch has more pairs than its LDS holds";
        return false;
      }
      n_slots += slots;
      n_pairs += (np + 1) & ~(int64_t)1;
      ++n_batches;
      seg_slots += slots;
      ++seg_batches;
      open = true;
      if (seg_slots >= segment_slots || seg_batches >= kSegmentBatches) {
        ++n_segs;
        seg_slots = seg_batches = 0;
        open = false;
      }
    }
    if (open) ++n_segs;
    tiles.back().v1 = v;
    T.tile_key.push_back(of.I * nb + of.J);
    T.tile_seg.push_back((int32_t)tiles.back().seg);
    T.tile_seg.push_back((int32_t)n_segs);
  }
  const int64_t limit = std::numeric_limits<int32_t>::max();
  if (n_slots > limit) {
    *err = "reduced camera system has too many staged factor blocks";
    return false;
  }
  if (n_pairs > limit) {
    *err = "reduced camera system has too many factor pairs";
    return false;
  }
  T.staged = n_slots;
  T.slots.resize(2 * (size_t)n_slots);
  T.pairs.resize((size_t)n_pairs);
  T.batches.resize(4 * (size_t)n_batches);
  T.batch_off.resize((size_t)n_batches * (kTileBlocks + 1));
  T.segs.resize(4 * (size_t)n_segs);
  T.seg_thread.resize((size_t)n_segs * kTileBlocks);
  T.seg_block.resize((size_t)n_segs * kTileBlocks);
  // Segment sg of tile (I, J): its batches and thread parts.
  auto close_segment = [&](int64_t sg, int64_t b0, int64_t b1, int64_t I, int64_t J) {
    int32_t* out = &T.segs[4 * (size_t)sg];
    out[0] = (int32_t)b0;
    out[1] = (int32_t)b1;
    out[2] = (int32_t)I;
    out[3] = (int32_t)J;
    int64_t seg_cnt[kTileBlocks];
    int parts[kTileBlocks];
    for (int k = 0; k < kTileBlocks; ++k) seg_cnt[k] = 0;
    for (int64_t b = b0; b < b1; ++b) {
      const uint16_t* o = &T.batch_off[(size_t)b * (kTileBlocks + 1)];
      for (int k = 0; k < kTileBlocks; ++k) seg_cnt[k] += o[k + 1] - o[k];
    }
    // One part per block with products, then the remaining threads one at a
    // time to the block with the most products per part (lowest index on
    // ties), at most 255 parts a block.
    int used = 0;
    for (int k = 0; k < kTileBlocks; ++k) {
      parts[k] = seg_cnt[k] > 0 ? 1 : 0;
      used += parts[k];
    }
    auto lower = [&](int a, int b) {  // a ranks below b
      const int64_t x = seg_cnt[a] * parts[b], y = seg_cnt[b] * parts[a];
      return x != y ? x < y : a > b;
    };
    int heap[kTileBlocks], nh = 0;
    for (int k = 0; k < kTileBlocks; ++k)
      if (parts[k]) heap[nh++] = k;
    std::make_heap(heap, heap + nh, lower);
    while (used < kTileBlocks && nh > 0) {
      std::pop_heap(heap, heap + nh, lower);
      const int best = heap[nh - 1];
      if (seg_cnt[best] <= parts[best]) break;
      parts[best]++;
      used++;
      if (parts[best] >= 255) --nh;
      else std::push_heap(heap, heap + nh, lower);
    }
    uint32_t* thread = &T.seg_thread[(size_t)sg * kTileBlocks];
    uint16_t* block = &T.seg_block[(size_t)sg * kTileBlocks];
    for (int k = 0; k < kTileBlocks; ++k) {
      thread[k] = 0u;
      block[k] = 0;
    }
    int t = 0;
    for (int k = 0; k < kTileBlocks; ++k) {
      if (!parts[k]) continue;
      block[k] = (uint16_t)(t | (parts[k] << 8));
      for (int p = 0; p < parts[k]; ++p) thread[t++] = (uint32_t)k | ((uint32_t)p << 8) | ((uint32_t)parts[k] << 16);
    }
  };
  auto fill_tile = [&](const Tile& tile) {
    const int64_t I = visits[tile.v0].I, J = visits[tile.v0].J;
    const bool diag = I == J;
    int64_t slot = tile.slot, pair = tile.pair, batch = tile.batch, seg = tile.seg, seg_first = batch, seg_slots = 0;
    uint16_t block[kBatchPairs], list[kBatchPairs];
    int32_t cnt[kTileBlocks + 1];
    for (int64_t v = tile.v0; v < tile.v1; ++batch) {
      int s = 0, np = 0;
      int32_t* out = &T.slots[2 * (size_t)slot];
      for (; v < tile.v1; ++v) {
        const Visit& vr = visits[v];
        if (s + vr.ni + vr.nj > kBatchSlots) break;
        const int si = s, sj = diag ? s : s + vr.ni;
        for (int a = 0; a < vr.ni + vr.nj; ++a) {
          const int g = a < vr.ni ? vr.gi + a : vr.gj + a - vr.ni;
          *out++ = g;
          *out++ = vr.l | (int32_t)(is_anchor(g) ? kSlotAnchor : 0u);
        }
        const int nj = diag ? vr.ni : vr.nj, gj = diag ? vr.gi : vr.gj;
        for (int a = 0; a < vr.ni; ++a) {
          const int row = (int)(T.g_row[vr.gi + a] - I * kTileBand) * kTileBand;
          for (int b = diag ? a : 0; b < nj; ++b) {
            block[np] = (uint16_t)(row + (int)(T.g_row[gj + b] - J * kTileBand));
            list[np++] = (uint16_t)((si + a) | ((sj + b) << 8));
          }
        }
        s += vr.ni + vr.nj;
      }
      // Stable counting sort of the batch's pairs by block.
      for (int k = 0; k <= kTileBlocks; ++k) cnt[k] = 0;
      for (int k = 0; k < np; ++k) cnt[block[k] + 1]++;
      for (int k = 0; k < kTileBlocks; ++k) cnt[k + 1] += cnt[k];
      uint16_t* off = &T.batch_off[(size_t)batch * (kTileBlocks + 1)];
      for (int k = 0; k <= kTileBlocks; ++k) off[k] = (uint16_t)cnt[k];
      uint16_t* pl = &T.pairs[(size_t)pair];
      for (int k = 0; k < np; ++k) pl[cnt[block[k]]++] = list[k];
      if (np % 2) pl[np] = 0;
      int32_t* bw = &T.batches[4 * (size_t)batch];
      bw[0] = (int32_t)slot;
      bw[1] = s;
      bw[2] = (int32_t)pair;
      bw[3] = np;
      slot += s;
      pair += (np + 1) & ~1;
      seg_slots += s;
      if (v == tile.v1 || seg_slots >= segment_slots || batch + 1 - seg_first >= kSegmentBatches) {
        close_segment(seg++, seg_first, batch + 1, I, J);
        seg_first = batch + 1;
        seg_slots = 0;
      }
    }
  };
  // The whole decomposition of 300 keyframes (1.2M observations, 8.4M pairs):
  // 480 ms on one thread of an eight-core host, 69 ms on its eight.
  if (!parallel_ranges((int64_t)tiles.size(), 1, [&](int64_t b, int64_t e, int) {
        for (int64_t t = b; t < e; ++t) fill_tile(tiles[t]);
      })) {
    *err = "host allocation failed";
    return false;
  }
  return true;
}

bool build_schur_rows(int32_t Pvar, int32_t L, const SchurTiles& T, SchurRows* out, std::string* err) {
  SchurRows& R = *out;
  R = SchurRows();
  R.row_ptr.assign((size_t)Pvar + 1, 0);
  R.diag_pos.assign((size_t)Pvar, 0);
  const int64_t n_g = (int64_t)T.g_row.size();
  std::vector<int32_t> row_g_ptr(Pvar + 1, 0), row_g(n_g), row_l(n_g);  // factor blocks and landmarks of each row
  for (int64_t g = 0; g < n_g; ++g) row_g_ptr[T.g_row[g] + 1]++;
  for (int i = 0; i < Pvar; ++i) row_g_ptr[i + 1] += row_g_ptr[i];
  {
    std::vector<int32_t> fill(row_g_ptr.begin(), row_g_ptr.end() - 1);
    for (int l = 0; l < L; ++l)
      for (int g = T.lm_g_ptr[l]; g < T.lm_g_ptr[l + 1]; ++g) {
        const int k = fill[T.g_row[g]]++;
        row_g[k] = g;
        row_l[k] = l;
      }
  }
  std::vector<std::vector<int32_t>> cols(Pvar), counts(Pvar);  // columns of a row; pairs of those >= the row
  // By thread: the last row that met a column, and the pairs it has with it.
  std::vector<std::vector<int32_t>> marks(kMaxHostThreads), pair_sums(kMaxHostThreads);
  if (!parallel_ranges(Pvar, 4, [&](int64_t i0, int64_t i1, int thread) {
        std::vector<int32_t>&mark = marks[thread], &pairs = pair_sums[thread];
        if (mark.empty()) {
          pairs.resize((size_t)Pvar, 0);
          mark.resize((size_t)Pvar, -1);
        }
        for (int i = (int)i0; i < (int)i1; ++i) {
          std::vector<int32_t>& c = cols[i];
          auto touch = [&](int j) {
            if (mark[j] != i) {
              mark[j] = i;
              pairs[j] = 0;
              c.push_back(j);
            }
          };
          touch(i);
          for (int k = row_g_ptr[i]; k < row_g_ptr[i + 1]; ++k) {
            const int a = row_g[k], l = row_l[k];
            const int ma = T.g_inc_ptr[a + 1] - T.g_inc_ptr[a];
            for (int b = T.lm_g_ptr[l]; b < a; ++b) touch(T.g_row[b]);
            for (int b = a; b < T.lm_g_ptr[l + 1]; ++b) {
              const int j = T.g_row[b];
              touch(j);
              pairs[j] += ma * (T.g_inc_ptr[b + 1] - T.g_inc_ptr[b]);
            }
          }
          std::sort(c.begin(), c.end());
          for (int j : c)
            if (j >= i) counts[i].push_back(pairs[j]);
        }
      })) {
    *err = "host allocation failed";
    return false;
  }
  for (int i = 0; i < Pvar; ++i) {
    R.diag_pos[i] = (int32_t)(R.col.size() + cols[i].size() - counts[i].size());
    R.col.insert(R.col.end(), cols[i].begin(), cols[i].end());
    R.upper_pairs.insert(R.upper_pairs.end(), counts[i].begin(), counts[i].end());
    R.row_ptr[i + 1] = (int32_t)R.col.size();
    R.max_row_blocks = std::max<int32_t>(R.max_row_blocks, (int32_t)cols[i].size());
  }
  for (int32_t n : R.upper_pairs) R.pairs += n;
  return true;
}

}  // namespace mlba
