// Sort-based histogram accumulation: bucket -> tile split and LDS tile sums.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rf_kern_common.hpp"
#include "rf_sort.hpp"

namespace rfk {
namespace {
using namespace detail;

// Clears the cursors of a sort draw and, on a call's first sub-draw, the
// draw counters (one launch instead of a cursor reset plus a memset) and new
// part sums.
__global__ void k_sort_reset(SortArgs a, unsigned long long* __restrict__ counter, uint32_t counter_words,
                             uint32_t part_words) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < a.n_buckets) a.bcur[i] = 0u;
  if (i < a.n_tiles) a.tcur[i] = 0u;
  if (i < counter_words) counter[i] = 0ull;
  if (i < part_words) a.part_sum[i] = 0ull;
}

// One workgroup per chunk of SORT_CHUNK records of a bucket (the host lists
// the chunks a bucket's capacity can hold): a counting sort of the chunk by
// tile in LDS, one reservation atomic per non-empty tile, then every record
// is written to its tile's run.  Records that do not fit in their tile's
// capacity are added to the histogram directly.  The tile of a sorted record
// is read back from the record itself, so the workgroup needs 69 KiB of LDS
// and two of them (32 waves) fit on a CU.  Larger chunks pay the per-chunk
// work (staging, reservations, scan, barriers) over more records: 8192 and
// 4096 records per workgroup took 12 % and 30 % longer on a 7680x4320 draw.  A
// small draw's plan takes SORT_CHUNK_SMALL: its few chunks leave the chip idle,
// and the pass then takes 6 us instead of 13 (2^18 records).
constexpr int RB_THREADS = 1024;

template <int CHUNK>
__global__ __launch_bounds__(RB_THREADS) void k_sort_rebucket(SortArgs a, float* __restrict__ bins,
                                                              const float4* __restrict__ palette) {
  static_assert(SORT_TILES_PER_BUCKET <= 4 * WAVE, "scan width");
  static_assert(SORT_TILES_PER_BUCKET <= RB_THREADS, "one thread per tile");
  constexpr int RB_PER = CHUNK / RB_THREADS;  // records per thread
  static_assert(RB_PER % 4 == 0, "16-byte loads");
  __shared__ uint32_t s_out[CHUNK];  // tile-ordered records
  __shared__ uint32_t s_cnt[SORT_TILES_PER_BUCKET], s_off[SORT_TILES_PER_BUCKET], s_gb[SORT_TILES_PER_BUCKET];
  __shared__ uint32_t s_total;
  __shared__ uint32_t s_toff[SORT_TILES_PER_BUCKET], s_tcap[SORT_TILES_PER_BUCKET];
  const uint32_t tid = threadIdx.x;
  const uint32_t job = a.chunks[blockIdx.x];
  const uint32_t b = job >> 16;
  const uint32_t cap = a.bcap[b];
  const uint32_t cur = a.bcur[b];
  const uint32_t count = cur < cap ? cur : cap;
  const uint32_t start = (job & 0xffffu) * (uint32_t)CHUNK;
  if (start >= count) return;  // workgroup-uniform
  const uint32_t n = (count - start) < (uint32_t)CHUNK ? (count - start) : (uint32_t)CHUNK;
  // bucket offsets and CHUNK are multiples of 4 records: 16-byte aligned
  const uint32_t* src = a.cbuf + a.boff[b] + start;
  const uint4* src4 = reinterpret_cast<const uint4*>(src);
  if (tid < (uint32_t)SORT_TILES_PER_BUCKET) {
    s_cnt[tid] = 0u;
    s_toff[tid] = a.toff[b * SORT_TILES_PER_BUCKET + tid];
    s_tcap[tid] = a.tcap[b * SORT_TILES_PER_BUCKET + tid];
  }
  // every thread keeps its RB_PER records in registers between the passes;
  // a full chunk (all but a bucket's last) issues its loads without per-lane
  // guards, which would otherwise make each load wait for the one before
  uint32_t rec[RB_PER];
  if (n == (uint32_t)CHUNK) {  // workgroup-uniform
#pragma unroll
    for (int k = 0; k < RB_PER / 4; ++k) {
      const uint4 q = src4[(uint32_t)k * RB_THREADS + tid];
      rec[4 * k] = q.x; rec[4 * k + 1] = q.y; rec[4 * k + 2] = q.z; rec[4 * k + 3] = q.w;
    }
  } else {
#pragma unroll
    for (int k = 0; k < RB_PER / 4; ++k) {
      const uint32_t i4 = (uint32_t)k * RB_THREADS + tid, i = 4u * i4;
      if (i + 3u < n) {
        const uint4 q = src4[i4];
        rec[4 * k] = q.x; rec[4 * k + 1] = q.y; rec[4 * k + 2] = q.z; rec[4 * k + 3] = q.w;
      } else {
#pragma unroll
        for (int e = 0; e < 4; ++e) rec[4 * k + e] = (i + (uint32_t)e) < n ? src[i + e] : SORT_NONE;
      }
    }
  }
  __syncthreads();
  constexpr uint32_t TSH = 8 + SORT_TILE_SHIFT;  // record >> TSH = tile within the bucket
  uint32_t rank[RB_PER];
#pragma unroll
  for (int m = 0; m < RB_PER; ++m) rank[m] = rec[m] != SORT_NONE ? atomicAdd(&s_cnt[rec[m] >> TSH], 1u) : 0u;
  __syncthreads();
  wave0_exclusive_scan<4>(s_cnt, s_off, SORT_TILES_PER_BUCKET, &s_total);
  if (tid < (uint32_t)SORT_TILES_PER_BUCKET) {
    const uint32_t c = s_cnt[tid];
    s_gb[tid] = c ? atomicAdd(a.tcur + b * SORT_TILES_PER_BUCKET + tid, c) : 0u;
  }
  __syncthreads();
#pragma unroll
  for (int m = 0; m < RB_PER; ++m)
    if (rec[m] != SORT_NONE) s_out[s_off[rec[m] >> TSH] + rank[m]] = rec[m];
  __syncthreads();
  // Write-out, four rounds at a time: their LDS reads are issued before the
  // first store, and one ballot per four rounds skips the overflow path.
  const uint32_t total = s_total;
  constexpr int U = 4;
  for (uint32_t q0 = 0; q0 * RB_THREADS < total; q0 += U) {  // uniform
    uint32_t j[U], r[U], gb[U], off[U], cap[U], toff[U];
    bool in[U], ovf[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      j[u] = (q0 + u) * RB_THREADS + tid;
      in[u] = j[u] < total;
      r[u] = s_out[in[u] ? j[u] : 0u];
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t f = r[u] >> TSH;
      gb[u] = s_gb[f];
      off[u] = s_off[f];
      cap[u] = s_tcap[f];
      toff[u] = s_toff[f];
    }
    bool any = false;
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const uint32_t dst = gb[u] + (j[u] - off[u]);
      ovf[u] = in[u] && dst >= cap[u];
      if (in[u] && !ovf[u])
        a.tbuf[toff[u] + dst] = (((r[u] >> 8) & ((1u << SORT_TILE_SHIFT) - 1u)) << 8) | (r[u] & 255u);
      any = any || ovf[u];
    }
    if (__builtin_amdgcn_ballot_w64(any)) {  // wave-uniform and rare
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const uint32_t bin = ovf[u] ? (b << SORT_COARSE_SHIFT) | (r[u] >> 8) : 0u;
        // the tile's frame's palette (batched rendering), from global memory
        const float4* pal = a.tile_pal ? palette + a.tile_pal[bin >> SORT_TILE_SHIFT] : palette;
        bin_quad(bins, bin, ovf[u], r[u] & 255u, 1.0f, pal);
      }
    }
  }
}

// One workgroup per segment of a tile of 2^12 bins (the host lists the
// segments of every tile): the segment's records are summed in LDS with two
// 64-bit atomics per record, red | green << 32 and blue | count << 32, the
// colours in fixed point (see SORT_SEG16 and SORT_SEG15 for why no field
// carries into the next; a palette entry's three fields fit 16 bits each, so
// the table read per record is 8 bytes, which LDS serves in half the cycles
// of the 16-byte addends: 8 % less time per 7680x4320 draw), then the
// touched bins are added to the histogram:
// with a plain read-modify-write when the tile is one segment (tiles are
// disjoint, and every overflow was added by earlier kernels), with quad
// atomics when several segments share the tile.  A workgroup that has only a
// part of a segment adds its integers to the segment's in device memory
// instead (sort_parts).  68 KiB of LDS: two
// workgroups of 16 waves per CU (tiles of 2^11 bins, 36 KiB and four
// workgroups of 8 waves, took 30 % longer on a 1024x1024 draw: the per-tile
// clearing, palette and write-back are paid over half the records).  Each
// thread loads 16 records (four 16-byte loads in flight) before it issues
// their LDS atomics.
constexpr int TILE_THREADS = 1024;
constexpr int TILE_BINS = 1 << SORT_TILE_SHIFT;

struct alignas(8) PalQ {
  uint32_t rg;  // red | green << 16
  uint32_t b;   // blue
};
// the two 64-bit addends of a palette entry
__device__ __forceinline__ uint64_t pal_rg(const PalQ& q) {
  return (uint64_t)(q.rg & 0xffffu) | ((uint64_t)(q.rg >> 16) << 32);
}
__device__ __forceinline__ uint64_t pal_bc(const PalQ& q) { return (uint64_t)q.b | (1ull << 32); }
struct TileSums {
  uint64_t rg[TILE_BINS];  // red | green << 32
  uint64_t bc[TILE_BINS];  // blue | count << 32
  PalQ pal[256];               // per palette entry, one 16-byte LDS read
};

__device__ __forceinline__ void tile_add(TileSums& t, uint32_t r) {
  const uint32_t p = r & 255u, i = r >> 8;
  const PalQ q = t.pal[p];
  lds_add_u64(&t.rg[i], pal_rg(q));
  lds_add_u64(&t.bc[i], pal_bc(q));
}

// Adds K records: every palette read is issued before the first atomic, so a
// record's atomics do not each wait for their own read.
template <int K>
__device__ __forceinline__ void tile_add_batch(TileSums& t, const uint32_t* r) {
  PalQ v[K];
  uint32_t bi[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    bi[k] = r[k] >> 8;
    v[k] = t.pal[r[k] & 255u];
  }
#pragma unroll
  for (int k = 0; k < K; ++k) {
    lds_add_u64(&t.rg[bi[k]], pal_rg(v[k]));
    lds_add_u64(&t.bc[bi[k]], pal_bc(v[k]));
  }
}

// A tile's fixed point: 2^16 - 1 per unit for one of at most SORT_SEG16
// records of room, else 2^15 - 1.
__device__ __forceinline__ float tile_one(uint32_t cap) { return cap > (uint32_t)SORT_SEG16 ? 32767.0f : 65535.0f; }

// A bin's sums as float colours and count.
__device__ __forceinline__ float4 tile_value(uint64_t rg, uint64_t bc, float inv) {
  return make_float4((float)(uint32_t)rg * inv, (float)(uint32_t)(rg >> 32) * inv, (float)(uint32_t)bc * inv,
                     (float)(uint32_t)(bc >> 32));
}

// Records of segment si of a tile that holds count, and their parts.
__device__ __forceinline__ uint32_t seg_parts(uint32_t count, uint32_t si, uint32_t seg, uint32_t part) {
  return (min(count - si * seg, seg) + part - 1) / part;
}

// Segments summed in parts: their integers to float and into the histogram,
// with plain read-modify-writes where the tile has no other segment.  A quarter
// of a tile per workgroup.  The sums are left zero.  (Done by the workgroup
// that adds a segment's last part, behind a fence and a counter, it took 3 to
// 9 us longer a draw than as a launch of its own, which a draw's readback
// saves.)
constexpr int PARTS_THREADS = 256, PARTS_BPT = 4;
constexpr uint32_t PARTS_BLOCKS = TILE_BINS / (PARTS_THREADS * PARTS_BPT);  // per slot
__device__ __forceinline__ void sort_parts(const SortArgs& a, float4* __restrict__ hist, uint32_t n_bins,
                                           uint32_t block) {
  const uint32_t slot = block / PARTS_BLOCKS;
  const uint32_t t = a.slots[slot] >> 16, si = a.slots[slot] & 0xffffu;
  const uint32_t cap = a.tcap[t], count = min(a.tcur[t], cap), seg = sort_seg_len(cap);
  if (si * seg >= count || seg_parts(count, si, seg, a.part_len) < 2u) return;  // workgroup-uniform
  const bool shared = cap > seg;
  const float inv = 1.0f / tile_one(cap);
  const uint32_t i0 = block % PARTS_BLOCKS * (PARTS_THREADS * PARTS_BPT) + threadIdx.x;
  unsigned long long* const p = a.part_sum + (size_t)slot * 2 * TILE_BINS + i0;
  const uint32_t base = (t << SORT_TILE_SHIFT) + i0;
  uint64_t rg[PARTS_BPT], bc[PARTS_BPT];
#pragma unroll
  for (int k = 0; k < PARTS_BPT; ++k) {
    rg[k] = p[k * PARTS_THREADS];
    bc[k] = p[TILE_BINS + k * PARTS_THREADS];
  }
#pragma unroll
  for (int k = 0; k < PARTS_BPT; ++k) {
    const uint32_t b = base + k * PARTS_THREADS;
    const bool add = bc[k] != 0ull && b < n_bins;
    const float4 v = tile_value(rg[k], bc[k], inv);
    if (shared) {  // workgroup-uniform
      bin_quad_vals(reinterpret_cast<float*>(hist), b, add, v);
    } else if (add) {
      float4 h = hist[b];
      h.x += v.x; h.y += v.y; h.z += v.z; h.w += v.w;
      hist[b] = h;
    }
    if (add) { p[k * PARTS_THREADS] = 0ull; p[TILE_BINS + k * PARTS_THREADS] = 0ull; }
  }
}

__global__ __launch_bounds__(PARTS_THREADS) void k_sort_parts(SortArgs a, float4* __restrict__ hist, uint32_t n_bins) {
  sort_parts(a, hist, n_bins, blockIdx.x);
}

// A draw's end in one launch: `copiers` workgroups store the counter words,
// then the bucket and tile cursors, straight into pinned host memory (out is
// its device address), instead of one copy command per array; the workgroups
// behind them add the segments in parts.
__global__ __launch_bounds__(PARTS_THREADS) void k_draw_readback(const unsigned long long* __restrict__ counter,
                                                                uint32_t counter_words, SortArgs a,
                                                                uint32_t* __restrict__ out, uint32_t copiers,
                                                                float4* __restrict__ hist, uint32_t n_bins) {
  if (blockIdx.x >= copiers) {
    sort_parts(a, hist, n_bins, blockIdx.x - copiers);
    return;
  }
  const uint32_t nb = a.n_buckets, cw = 2u * counter_words, n = cw + nb + a.n_tiles;
  const uint32_t* c32 = reinterpret_cast<const uint32_t*>(counter);
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += copiers * blockDim.x)
    out[i] = i < cw ? c32[i] : (i < cw + nb ? a.bcur[i - cw] : a.tcur[i - cw - nb]);
}

__global__ __launch_bounds__(TILE_THREADS) void k_sort_tiles(SortArgs a, float4* __restrict__ hist, uint32_t n_bins,
                                                            const float4* __restrict__ palette) {
  __shared__ TileSums s_t;
  const uint32_t tid = threadIdx.x;
  const uint32_t job = a.segs[blockIdx.x];
  const uint32_t t = job >> 16;
  const uint32_t base = t << SORT_TILE_SHIFT;
  const uint32_t cap = a.tcap[t];
  const uint32_t cur = a.tcur[t];
  const uint32_t count = cur < cap ? cur : cap;
  // workgroup-uniform: a tile of at most SORT_SEG16 records is summed at
  // 2^16 - 1 per unit, a larger one at 2^15 - 1 in segments of SORT_SEG15 (both
  // in parts, a workgroup each, where the plan says so)
  const uint32_t seg = sort_seg_len(cap);
  const float one = tile_one(cap);
  const uint32_t part = a.part_len ? a.part_len : seg, per_seg = (seg + part - 1) / part;
  const uint32_t si = (job & 0xffffu) / per_seg, in_seg = (job & 0xffffu) % per_seg * part;
  const uint32_t start = si * seg + in_seg;
  if (base >= n_bins || start >= count) return;  // workgroup-uniform
  const uint32_t n = min(count - start, min(part, seg - in_seg));
  for (uint32_t i = tid; i < (uint32_t)TILE_BINS; i += TILE_THREADS) {
    s_t.rg[i] = 0ull;
    s_t.bc[i] = 0ull;
  }
  if (tid < 256u) {
    // palette values lie in [0, 1]: each field gets at most `one` (< 2^16)
    // per record
    const float4 c = (a.tile_pal ? palette + a.tile_pal[t] : palette)[tid];
    const uint32_t r = (uint32_t)(c.x * one + 0.5f), g = (uint32_t)(c.y * one + 0.5f),
                   bl = (uint32_t)(c.z * one + 0.5f);
    s_t.pal[tid].rg = r | (g << 16);
    s_t.pal[tid].b = bl;
  }
  __syncthreads();
  // Tile offsets, segments and parts are multiples of 4 records, so the
  // records start 16-byte aligned.
  const uint32_t* src = a.tbuf + a.toff[t] + start;
  const uint4* src4 = reinterpret_cast<const uint4*>(src);
  const uint32_t n4 = n / 4;
  constexpr uint32_t G = 4;  // 16-byte loads per thread and round
  for (uint32_t i0 = 0; i0 < n4; i0 += G * TILE_THREADS) {
    if (i0 + G * TILE_THREADS <= n4) {  // workgroup-uniform: a full round
      uint32_t r[4 * G];
#pragma unroll
      for (uint32_t k = 0; k < G; ++k) {
        const uint4 q = src4[i0 + k * TILE_THREADS + tid];
        r[4 * k] = q.x; r[4 * k + 1] = q.y; r[4 * k + 2] = q.z; r[4 * k + 3] = q.w;
      }
      tile_add_batch<2 * G>(s_t, r);
      tile_add_batch<2 * G>(s_t, r + 2 * G);
    } else {
#pragma unroll
      for (uint32_t k = 0; k < G; ++k) {
        const uint32_t i = i0 + k * TILE_THREADS + tid;
        if (i < n4) {
          const uint4 q = src4[i];
          const uint32_t r[4] = {q.x, q.y, q.z, q.w};
          tile_add_batch<4>(s_t, r);
        }
      }
    }
  }
  for (uint32_t i = n4 * 4 + tid; i < n; i += TILE_THREADS) tile_add(s_t, src[i]);
  __syncthreads();
  const bool shared = cap > seg;  // several segments add to this tile
  const float inv = 1.0f / one;
  constexpr int BPT = TILE_BINS / TILE_THREADS;  // bins per thread
  static_assert(BPT * TILE_THREADS == TILE_BINS, "bins per thread");
  if (a.part_len && seg_parts(count, si, seg, part) > 1u) {  // workgroup-uniform: sort_parts goes on
    unsigned long long* const p = a.part_sum + (size_t)(a.tslot[t] + si) * 2 * TILE_BINS;
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
      const uint32_t i = (uint32_t)k * TILE_THREADS + tid;
      const uint64_t bc = s_t.bc[i];
      if (bc == 0ull) continue;  // no record, no colour
      __hip_atomic_fetch_add(p + i, s_t.rg[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      __hip_atomic_fetch_add(p + TILE_BINS + i, bc, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return;
  }
  float4 v[BPT];
  bool add[BPT];
#pragma unroll
  for (int k = 0; k < BPT; ++k) {
    const uint32_t i = (uint32_t)k * TILE_THREADS + tid;
    const uint64_t bc = s_t.bc[i];
    v[k] = tile_value(s_t.rg[i], bc, inv);
    add[k] = base + i < n_bins && bc != 0ull;
  }
  if (shared) {  // workgroup-uniform
#pragma unroll
    for (int k = 0; k < BPT; ++k)
      bin_quad_vals(reinterpret_cast<float*>(hist), base + (uint32_t)k * TILE_THREADS + tid, add[k], v[k]);
  } else {
    // the touched bins' read-modify-writes, all loads in flight before the
    // first store
    float4 h[BPT];
#pragma unroll
    for (int k = 0; k < BPT; ++k)
      h[k] = add[k] ? hist[base + (uint32_t)k * TILE_THREADS + tid] : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int k = 0; k < BPT; ++k) {
      if (!add[k]) continue;
      h[k].x += v[k].x; h[k].y += v[k].y; h[k].z += v[k].z; h[k].w += v[k].w;
      hist[base + (uint32_t)k * TILE_THREADS + tid] = h[k];
    }
  }
}

// One workgroup per tile: the sum of the count channel over its bins, the
// estimate of where the next draw's samples go when a flame has no sort
// draw to learn from yet.
__global__ __launch_bounds__(256) void k_sort_tile_mass(const float4* __restrict__ hist, uint32_t n_bins,
                                                       float* __restrict__ mass) {
  __shared__ float s_w[256 / WAVE];
  const uint32_t base = blockIdx.x * (uint32_t)TILE_BINS;
  float sum = 0.0f;
  for (uint32_t i = threadIdx.x; i < (uint32_t)TILE_BINS; i += 256u)
    if (base + i < n_bins) sum += hist[base + i].w;
  sum = wave_sum(sum);
  if ((threadIdx.x & (WAVE - 1)) == 0) s_w[threadIdx.x / WAVE] = sum;
  __syncthreads();
  if (threadIdx.x == 0) {
    float t = 0.0f;
    for (int k = 0; k < 256 / WAVE; ++k) t += s_w[k];
    mass[blockIdx.x] = t;
  }
}

}  // namespace

hipError_t launch_sort_tile_mass(const float4* bins, uint32_t n_bins, uint32_t n_tiles, float* mass, hipStream_t s) {
  if (n_tiles == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_tile_mass, dim3(n_tiles), dim3(256), 0, s, bins, n_bins, mass);
  return hipGetLastError();
}

hipError_t launch_sort_reset(const SortArgs& a, hipStream_t s, unsigned long long* counter, uint32_t counter_words,
                             uint32_t part_words) {
  uint32_t n = a.n_tiles > a.n_buckets ? a.n_tiles : a.n_buckets;
  if (!counter) counter_words = 0;
  if (counter_words > n) n = counter_words;
  if (part_words > n) n = part_words;
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_reset, dim3((n + 255) / 256), dim3(256), 0, s, a, counter, counter_words, part_words);
  return hipGetLastError();
}

hipError_t launch_draw_readback(const unsigned long long* counter, uint32_t counter_words, const SortArgs* a,
                                uint32_t* out, hipStream_t s, float* bins, uint32_t n_bins) {
  const SortArgs g = a ? *a : SortArgs{};
  const uint32_t n = 2u * counter_words + g.n_buckets + g.n_tiles;
  const uint32_t copiers = (n + PARTS_THREADS - 1) / PARTS_THREADS < 64u ? (n + PARTS_THREADS - 1) / PARTS_THREADS : 64u;
  const uint32_t grid = copiers + (bins ? g.n_slots * PARTS_BLOCKS : 0u);
  if (grid == 0) return hipSuccess;
  hipLaunchKernelGGL(k_draw_readback, dim3(grid), dim3(PARTS_THREADS), 0, s, counter, counter_words, g, out, copiers,
                     reinterpret_cast<float4*>(bins), n_bins);
  return hipGetLastError();
}

hipError_t launch_sort_rebucket(const SortArgs& a, float* bins, const float4* palette, hipStream_t s) {
  if (a.n_chunks == 0) return hipSuccess;
  if (a.chunk_len == (uint32_t)SORT_CHUNK_SMALL)
    hipLaunchKernelGGL(k_sort_rebucket<SORT_CHUNK_SMALL>, dim3(a.n_chunks), dim3(RB_THREADS), 0, s, a, bins, palette);
  else
    hipLaunchKernelGGL(k_sort_rebucket<SORT_CHUNK>, dim3(a.n_chunks), dim3(RB_THREADS), 0, s, a, bins, palette);
  return hipGetLastError();
}

hipError_t launch_sort_tiles(const SortArgs& a, float* bins, uint32_t n_bins, const float4* palette, hipStream_t s) {
  if (a.n_segs == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_tiles, dim3(a.n_segs), dim3(TILE_THREADS), 0, s, a, reinterpret_cast<float4*>(bins),
                     n_bins, palette);
  return hipGetLastError();
}

hipError_t launch_sort_parts(const SortArgs& a, float* bins, uint32_t n_bins, hipStream_t s) {
  if (a.n_slots == 0) return hipSuccess;
  hipLaunchKernelGGL(k_sort_parts, dim3(a.n_slots * PARTS_BLOCKS), dim3(PARTS_THREADS), 0, s, a,
                     reinterpret_cast<float4*>(bins), n_bins);
  return hipGetLastError();
}

}  // namespace rfk
