// Sort-based histogram accumulation (RF_HIST_SORT): shared definitions.
//
// Instead of one memory-side atomic per sample, the chaos-game kernel writes
// 4-byte records into coarse buckets of 2^19 bins, a second kernel splits
// each bucket into 128 tiles of 2^12 bins, and a third accumulates every tile
// in LDS and adds it to the histogram with one plain read-modify-write per
// touched bin (a tile of many records in segments and parts, below).  Records carry no weight, so the mode needs unit opacities;
// the LDS sums are fixed point, so palette values must lie in [0, 1].
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#include <stdint.h>
#endif

namespace rfk {

constexpr int SORT_COARSE_SHIFT = 19;                                        // bins per bucket: 2^19
constexpr int SORT_TILE_SHIFT = 12;                                          // bins per tile: 2^12
constexpr int SORT_TILES_PER_BUCKET = 1 << (SORT_COARSE_SHIFT - SORT_TILE_SHIFT);  // 128
constexpr int SORT_MAX_BUCKETS = 256;                                        // 2^27 bins
constexpr int SORT_STAGE_SLOTS = 4096;                                       // samples staged in LDS per flush
constexpr int SORT_CHUNK = 16384;                                            // records per rebucketing workgroup
constexpr int SORT_CHUNK_SMALL = 4096;                                       // the same in a small draw's plan
// Tile sums add red | green << 32 and blue | count << 32 per record with
// 64-bit LDS atomics, colours in fixed point.  A tile of at most SORT_SEG16
// records is summed by one workgroup at 2^16 - 1 per unit (a field then
// holds at most 65532 * 65535 < 2^32, so no carry crosses into the next); a
// larger tile is split into segments of at most SORT_SEG15 records, each
// summed by its own workgroup at 2^15 - 1 per unit (131068 * 32767 < 2^32).  A
// plan for a small image may have several workgroups sum a segment in parts
// (part_len): their integers are added in device memory, so a segment's sums
// are the same, and rounded to float once, however it is cut.
// Each sample's colour is rounded by at most 1 / (2 * 65535) or
// 1 / (2 * 32767), about 2^-17 and 2^-16.
constexpr int SORT_SEG16 = 65532;
constexpr int SORT_SEG15 = 131068;
// Records per segment of a tile of capacity cap.
constexpr uint32_t sort_seg_len(uint32_t cap) { return cap > (uint32_t)SORT_SEG16 ? SORT_SEG15 : SORT_SEG16; }
constexpr uint32_t SORT_MAX_SLOTS = 1024;  // segments a plan may cut into parts
constexpr uint32_t SORT_SLOT_WORDS = 2u << SORT_TILE_SHIFT;  // u64 sums of one (64 KiB)
constexpr uint32_t SORT_NONE = 0xffffffffu;

struct SortArgs {
  uint32_t* cbuf;          // bucket records: ((bin mod 2^19) << 8) | palette index
  uint32_t* tbuf;          // tile records:   ((bin mod 2^12) << 8) | palette index
  uint32_t* bcur;          // per bucket: records offered (may exceed the capacity)
  uint32_t* tcur;          // per tile: records offered
  const uint32_t* boff;    // per bucket: first record in cbuf
  const uint32_t* bcap;    // per bucket: capacity
  const uint32_t* toff;    // per tile: first record in tbuf
  const uint32_t* tcap;    // per tile: capacity
  const uint32_t* chunks;  // rebucketing work: (bucket << 16) | chunk index, one per workgroup
  const uint32_t* segs;    // tile work: (tile << 16) | part index over the tile's segments, one per workgroup
  uint32_t n_buckets;
  uint32_t n_tiles;        // n_buckets * SORT_TILES_PER_BUCKET
  uint32_t n_chunks, n_segs;
  uint32_t chunk_len;      // records per chunk: SORT_CHUNK_SMALL, or 0 for SORT_CHUNK
  uint32_t part_len;       // records per part of a segment; 0: whole segments
  // With parts: per slot (tile << 16) | segment of a segment that may have
  // several parts, per tile the slot of its first segment, and per slot
  // SORT_SLOT_WORDS integer sums, zero between draws.
  uint32_t n_slots;
  const uint32_t* slots;
  const uint32_t* tslot;
  unsigned long long* part_sum;
  // Batched rendering: per tile, the offset (in entries) of its frame's
  // palette in the palette array the record passes get; null when one
  // palette serves every tile.
  const uint32_t* tile_pal;
};

#ifndef __HIPCC_RTC__
// Workgroups of a draw of n_batches batches of n_iter iterations each, when a
// flush takes `stage` iterations and `resident` workgroups run at once.  A
// flush of any size reserves its runs with one atomic per bucket on the same
// few cache lines (about 9 ns per workgroup and line, one after another), so
// draws of few iterations are bound by their flushes, and a workgroup takes up
// to four batches if that makes the stages fuller.  One draw of 4 Mi
// particles, one batch against this rule (us):
//   iterations              1          2          3          5          10
//   8 buckets (2048^2)   164 / 116  180 / 154  206 / 198  275 / 279* 493 / 502*
//   32 buckets (4096^2)  197 / 141  214 / 180  229 / 214  294 / 289* 466 / 472*
//   64 buckets           277 / 171  308 / 205  334 / 254  384 / 326  605 / 500
// Where more than half a stage is filled anyway, up to 32 buckets (one line of
// cursors) hide the flushes behind the other workgroups' iterations and the
// coarser grid costs more than it saves (*: not done).  Up to eight batches
// gain nothing over four: 1 and 3 iterations 105 and 195 us instead of 102 and
// 184 into 2048^2, 125 and 205 instead of 122 and 194 into 4096^2, and with
// four times the particles 294 and 560 instead of 296 and 570.  A grid below
// the resident workgroups leaves compute units idle: 262144 particles, 5
// iterations, 68 us with one batch, 79 with three.
inline uint32_t sort_grid(uint32_t n_batches, uint32_t n_iter, uint32_t n_buckets, uint32_t stage,
                          uint32_t resident) {
  if (n_iter == 0 || (n_buckets <= 32 && n_iter > stage / 2)) return n_batches;
  auto flushes = [&](uint64_t m) { return (m * n_iter + stage - 1) / stage; };
  uint64_t per = 1;
  for (uint64_t m = 2; m <= 4; ++m)
    if (flushes(m) * per < flushes(per) * m) per = m;
  const uint32_t grid = (uint32_t)((n_batches + per - 1) / per);
  const uint32_t least = n_batches < resident ? n_batches : resident;
  return grid > least ? grid : least;
}

// Clears the cursors, counter_words words of counter and part_words of the
// parts' sums.
hipError_t launch_sort_reset(const SortArgs& a, hipStream_t s, unsigned long long* counter = nullptr,
                             uint32_t counter_words = 0, uint32_t part_words = 0);
// Copies counter_words 64-bit counters, then (a given) its bucket and tile
// cursors into out, 32-bit words, in one launch; out may be the device address
// of pinned host memory.  With bins the same launch ends a draw whose segments
// were summed in parts (launch_sort_parts).
hipError_t launch_draw_readback(const unsigned long long* counter, uint32_t counter_words, const SortArgs* a,
                                uint32_t* out, hipStream_t s, float* bins = nullptr, uint32_t n_bins = 0);
hipError_t launch_sort_rebucket(const SortArgs& a, float* bins, const float4* palette, hipStream_t s);
// Sums the tiles' records.  With n_slots > 0 the segments in parts are still to
// be added to bins, by launch_sort_parts or launch_draw_readback.
hipError_t launch_sort_tiles(const SortArgs& a, float* bins, uint32_t n_bins, const float4* palette, hipStream_t s);
hipError_t launch_sort_parts(const SortArgs& a, float* bins, uint32_t n_bins, hipStream_t s);
// mass[t] = sum of the count channel over tile t of a histogram (t < n_tiles).
hipError_t launch_sort_tile_mass(const float4* bins, uint32_t n_bins, uint32_t n_tiles, float* mass, hipStream_t s);
#endif

}  // namespace rfk
