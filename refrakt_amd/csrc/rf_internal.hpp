// Internal interface between the host library (rf_host.cpp) and the kernel
// launchers (rf_k_compat.hip, rf_k_fast.hip, rf_k_misc.hip).
#pragma once
#ifndef __HIPCC_RTC__
#include <hip/hip_runtime.h>
#include <stdint.h>
#endif

#include "rf_device.hpp"
#include "rf_sort.hpp"

namespace rfk {

struct CompatArgs {
  const float4* pos_in;
  float4* pos_out;
  const uint32_t* shuf;          // shuffle rows, row-major, ppt entries per row
  uint4* rs;                     // jsf32 state per slot
  const rfd::Block* blocks;      // per temporal sample
  uint32_t block_stride;         // 0: one block for all samples, 1: one per sample
  const float4* palette;
  float* bins;                   // W*H RGBA
  unsigned long long* counter;   // binned samples
  uint32_t ppt;                  // particles per temporal sample
  uint32_t T;                    // temporal samples
  uint32_t in_row, out_row;
  uint32_t random_read, random_write, first_run, do_draw;
  uint32_t W, H;
  float ss[6];                   // screen affine
};

struct FastArgs {
  float4* pos;                   // P particles (x, y, c, 0), read and written
  const rfd::Block* blocks;
  uint32_t block_stride;
  const float4* palette;
  float* bins;
  unsigned long long* counter;
  const uint16_t* perms;         // NPERM rows x (64*waves) slot permutations
  uint64_t seed;
  uint32_t launch;               // launch counter (RNG streams)
  uint32_t ppt;
  uint32_t n_iter;
  uint32_t n_batches;            // batches of 64*waves particles (set by launch_fast)
  uint32_t first_run, do_draw;
  uint32_t W, H;
  float ss[6];
  SortArgs sort;                 // RF_HIST_SORT only
};

// The splat's shape: see k_de_chords.
constexpr int DE_MAX_R = 100;          // largest splat radius
constexpr int DE_CHORD_STRIDE = 128;   // radii per table row
constexpr int DE_C_ROW0 = 108, DE_C_ROWS = 216;
struct DEChord {
  int hl;
  float nx, step, pad;
};
struct DETable {
  DEChord rows[2 * DE_MAX_R + 1][DE_CHORD_STRIDE];
  float c[DE_MAX_R + 1][DE_C_ROWS];
};

// Tonemap parameters; ig = 1 / gamma, rounded once.
struct ToneArgs {
  float ig, brightness, vibrancy, k;
};
#ifndef __HIPCC_RTC__
inline ToneArgs tone_args(float gamma, float brightness, float vibrancy, float k) {
  return ToneArgs{(float)(1.0 / (double)gamma), brightness, vibrancy, k};
}
#endif

struct DEArgs {
  const float4* hist;            // W*H bins (rows bottom-up)
  float4* de_out;                // may be null
  float4* img_out;               // may be null (tonemapped)
  uint32_t W, H;
  int32_t R, rmin;
  float curve;
  int32_t do_tonemap;
  ToneArgs tone;
  // Optional completion stamp (batched rendering): the last workgroup to
  // finish writes the wall clock to *done_ts; *tiles_done counts workgroups.
  uint32_t* tiles_done;
  unsigned long long* done_ts;
  // Work buffer: every bin's splat radius (W*H bytes, see k_de_radius).
  uint8_t* rad;
  // Chord table (launch_de_chords).
  const DETable* tab;
};

constexpr int NPERM = 8;          // permutation rows of the fast engine (held in LDS)
// Draw counters: COUNTER_SLOTS slots of COUNTER_STRIDE u64 (one 128-byte
// line each; slot s holds [binned samples, LDS-table re-hits]).  Memory-side
// atomics on one address serialise (about 80 M/s): one counter for every
// wave of a 2^24-particle draw cost 1.6 ms, spread over 64 lines they cost
// nothing.  The host sums the slots.
constexpr int COUNTER_SLOTS = 64;
constexpr int COUNTER_STRIDE = 16;

#ifndef __HIPCC_RTC__
hipError_t launch_init_rs(uint4* rs, uint64_t n, hipStream_t s);
hipError_t launch_compat_pass(const CompatArgs& a, int hist_mode, hipStream_t s);
hipError_t launch_fast(const FastArgs& a, uint64_t n_particles, int waves, int hist_mode, hipStream_t s);
// Fills n u64 with zero (a kernel, not a memset: safe under graph capture).
hipError_t launch_zero_u64(unsigned long long* p, uint32_t n, hipStream_t s);
hipError_t launch_animate(rfd::Block* blocks, uint32_t T, float tss_width, const float* rot, hipStream_t s);
// Fills the chord table.
hipError_t launch_de_chords(DETable* tab, hipStream_t s);
// Density estimation (+ tonemap): a.rad (W*H bytes) is a device buffer the
// launch may overwrite, a.tab the chord table; R and rmin in [0, DE_MAX_R].
hipError_t launch_de_tonemap(const DEArgs& a, hipStream_t s);
hipError_t launch_tonemap(const float4* in, float4* out, uint32_t n, const ToneArgs& t, hipStream_t s);
hipError_t launch_rgba8(const float4* in, uchar4* out, uint32_t n, hipStream_t s);
hipError_t launch_eval_xform(const rfd::Block* blk, const float* pts, const float* rands, float* out,
                             uint32_t n, hipStream_t s);
hipError_t launch_atomic_probe(float* bins, uint64_t nbins, uint64_t samples, int hist_mode,
                               const float4* palette, hipStream_t s);
#endif

}  // namespace rfk
