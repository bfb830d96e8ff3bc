// ba_tiles.h -- work decomposition of the reduced camera system build.
//
// S = sum over landmarks l of the products of l's factor blocks: a factor
// block is the sum of the incidences of one landmark in one row of S
// (normally one observation, or the landmark's anchor). S is cut into tiles
// of kTileBand x kTileBand blocks (block rows I, block columns J >= I); a
// landmark whose factor blocks fall into bands I and J "visits" tile (I, J)
// and contributes the products of its blocks in I with its blocks in J. A
// tile's visits (in landmark order) are cut into batches whose factor blocks
// fit the LDS of one work-group (the batch's slot list names them), and the
// batches into segments (the work items). In a segment, each of the
// kTileBlocks threads owns one part of one block of the tile: blocks with
// more products get more parts (in proportion to their products in the
// segment), and part p of a block with n parts takes the block's products
// p, p + n, ... of every batch. Each part's sum is written to its own slot
// of the segment's partial; a block of S adds its parts in part order and
// its segments in segment order. Nothing here depends on the device, the
// launch or timing, so S repeats bit for bit.
#ifndef MAPLAB_AMD_BA_TILES_H_
#define MAPLAB_AMD_BA_TILES_H_

#include <stdint.h>

#include <functional>
#include <memory>
#include <new>
#include <string>
#include <utility>
#include <vector>

namespace mlba {

constexpr int kTileBand = 16;                        // block rows (and columns) of a tile
constexpr int kTileBlocks = kTileBand * kTileBand;   // blocks of a tile = threads of a work-group
constexpr int kBatchSlots = 256;                     // factor blocks staged in LDS per batch (<= 256)
constexpr int kSegmentSlots = 5120;                  // staged factor blocks per segment of a large system, at least
constexpr int kSegmentTarget = 512;                  // segments that run at once
constexpr int kSegmentBatches = 64;                  // batches per segment, at most
constexpr int kBatchPairs = 2560;                    // pairs per batch, at most
constexpr int kPairWords = kBatchPairs / 2 / kTileBlocks;  // 32-bit pair words a thread stages per batch
constexpr int kPartEntries = 42;                     // a part's block (36) and rhs (6) sums
constexpr int kTilePartial = kTileBlocks * kPartEntries;  // doubles of one segment's partial
constexpr uint32_t kSlotAnchor = 0x80000000u;        // slot word: the block is its landmark's anchor

// Segment thread word: block (bits 0-7), part (8-15), parts of the block
// (16-23); 0 parts: the thread idles. Segment block word: first thread of
// the block (bits 0-7) and its parts (8-15).
constexpr int seg_thread_block(uint32_t w) { return (int)(w & 255u); }
constexpr int seg_thread_part(uint32_t w) { return (int)((w >> 8) & 255u); }
constexpr int seg_thread_parts(uint32_t w) { return (int)((w >> 16) & 255u); }

// A vector whose resize leaves new elements unset: the large arrays are sized
// once and filled by several threads.
template <class T>
struct UnsetAllocator : std::allocator<T> {
  template <class U>
  struct rebind {
    using other = UnsetAllocator<U>;
  };
  template <class U>
  void construct(U* p) noexcept {
    ::new (static_cast<void*>(p)) U;
  }
  template <class U, class... A>
  void construct(U* p, A&&... a) {
    ::new (static_cast<void*>(p)) U(std::forward<A>(a)...);
  }
};
template <class T>
using UnsetVector = std::vector<T, UnsetAllocator<T>>;

constexpr int kMaxHostThreads = 8;  // threads of parallel_ranges, the caller's among them

// Runs body(begin, end, thread) over pieces of [0, n) on up to kMaxHostThreads
// threads (the caller's is thread 0), pieces taken in order; rethrows nothing:
// returns false when a piece threw.
bool parallel_ranges(int64_t n, int64_t piece, const std::function<void(int64_t, int64_t, int)>& body);

struct SchurTiles {
  int32_t nbands = 0;
  UnsetVector<int32_t> g_row;       // row of each factor block (landmark-major, rows ascending)
  UnsetVector<int32_t> g_inc_ptr;   // incidences summed into each factor block
  UnsetVector<int32_t> g_inc;       // their codes (observation >= 0, anchor -1 - landmark)
  UnsetVector<int32_t> lm_g_ptr;    // factor blocks of each landmark (L + 1)
  UnsetVector<int32_t> slots;       // 2 per staged slot: factor block, landmark | kSlotAnchor
  UnsetVector<int32_t> batches;     // 4 per batch: first slot, slots, first pair (even), pairs
  UnsetVector<uint16_t> batch_off;  // kTileBlocks + 1 per batch: pair offsets of each block
  UnsetVector<uint16_t> pairs;      // staged slots x | y << 8, by block, then visit
  UnsetVector<int32_t> segs;        // 4 per segment: first batch, end batch, I, J
  UnsetVector<uint32_t> seg_thread; // kTileBlocks per segment: the thread's part
  UnsetVector<uint16_t> seg_block;  // kTileBlocks per segment: the block's parts
  std::vector<int64_t> tile_key;    // visited tiles, ascending I * nbands + J
  std::vector<int32_t> tile_seg;    // 2 per visited tile: its segment range
  int64_t visits = 0;               // landmark tile visits
  int64_t staged = 0;               // factor blocks staged over all batches
};

// inc_ptr / inc: incidences of each of the Pvar rows of S (codes as above);
// obs_landmark: landmark of each observation. Returns false (and a reason)
// when a count overflows the decomposition's index widths.
bool build_schur_tiles(int32_t Pvar, int32_t L, const int32_t* inc_ptr, const int32_t* inc,
                       const int32_t* obs_landmark, SchurTiles* out, std::string* err);

// Block structure of S in rows of ascending columns: row i couples with the row
// of every factor block of every landmark it has one of, and with itself.
struct SchurRows {
  std::vector<int32_t> row_ptr, col;     // Pvar + 1; one per block
  std::vector<int32_t> diag_pos;         // position of each row's own block
  std::vector<int32_t> upper_pairs;      // per block with column >= row, in row order: incidence pairs
                                         // (x in the row, y in the column, same landmark) summed into it
  int64_t pairs = 0;                     // their sum
  int32_t max_row_blocks = 0;
};
bool build_schur_rows(int32_t Pvar, int32_t L, const SchurTiles& tiles, SchurRows* out, std::string* err);

}  // namespace mlba

#endif  // MAPLAB_AMD_BA_TILES_H_
