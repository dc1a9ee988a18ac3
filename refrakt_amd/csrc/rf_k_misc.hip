// Parameter inflation, density estimation + tonemap, diagnostics.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "rf_kern_common.hpp"

using namespace rfd;

namespace rfk {
namespace {
using namespace detail;

// ---------------------------------------------------------------- animate
// Temporal-sample parameter inflation (shaders/templates/animate.tpl.glsl:18-96):
// block i (one workgroup each) is a copy of the pristine block blocks[T]
// with every xform's affine rotated by theta = 0.31415926535 * dt * rot[k],
// dt = (i - T/2) / float(T/2) * tss:
//   a' = a cos + c sin, b' = b cos + d sin, c' = c cos - a sin, d' = d cos - b sin.
// rot[k] is xform k's rotation_frequency (rot[n_xforms] for the final xform).
// The reference dispatches T/32 groups of 32 lanes, so it defines T >= 32
// only; at T = 1 (half = 0) the single block is the centre sample, dt = 0.
// The division is correctly rounded and sin/cos are evaluated in double and
// rounded to float, so the blocks are a deterministic function of the inputs
// that a CPU computes to the same bits.
__global__ __launch_bounds__(256) void k_animate(Block* blocks, uint32_t T, float tss,
                                                 const float* __restrict__ rot) {
  const uint32_t i = blockIdx.x;
  const Block* src = blocks + T;
  Block* dst = blocks + i;
  const uint32_t* s32 = reinterpret_cast<const uint32_t*>(src);
  uint32_t* d32 = reinterpret_cast<uint32_t*>(dst);
  for (uint32_t k = threadIdx.x; k < sizeof(Block) / 4; k += blockDim.x) d32[k] = s32[k];
  __syncthreads();
  const int nx = (int)src->n_xforms;
  const int k = (int)threadIdx.x;
  if (!(k < nx || (k == nx && src->has_final))) return;
  const int slot = k < nx ? k : FINAL;
  const int half = (int)(T / 2u);
  const int pos = (int)i - half;
  const float dt = half ? rf_div_rn((float)pos, (float)half) * tss : 0.0f;
  const float rps = 0.31415926535f;
  const float th = rps * dt * rot[k];
  const float sn = (float)sin((double)th), cs = (float)cos((double)th);
  const float* a = src->xf[slot].aff;
  float* b = dst->xf[slot].aff;
  const float t0 = a[0] * cs, t1 = a[2] * sn;
  const float t2 = a[1] * cs, t3 = a[3] * sn;
  const float t4 = a[2] * cs, t5 = a[0] * sn;
  const float t6 = a[3] * cs, t7 = a[1] * sn;
  b[0] = t0 + t1;
  b[1] = t2 + t3;
  b[2] = t4 - t5;
  b[3] = t6 - t7;
}

// ------------------------------------------------- density estimation
// Gather form of the reference's point-sprite splat (shaders/density_vert.glsl,
// shaders/density_frag.glsl, src/main.cpp:490-515).  A bin (px, py) with
// alpha a > 0 becomes a sprite centred on render-target texel
// (cx, cy) = (px - 1, H - 1 - py) (glm::ortho(0,W,H,0) maps its vertex at
// (px - 1/(4r+2), py + 1/(4r+2)) there; bins of column 0 have their centre
// outside the clip volume and are dropped).  Texel (cx + j, cy + i) receives
// color * (1 - d) * (2/pi)/r^2 where d = ((2j + 1/S)^2 + (2i + 1/S)^2) / S^2,
// S = 2r + 1, when |i|,|j| <= r and d <= 1; r = 0 copies the bin.
// r = max(rmin, min(R, int(R / a^curve))).
// A splat reaches span = max(R, rmin) texels from its centre.

// x^y for x >= 0: the library's powf without its sign and integer-exponent
// cases, the same bits.
extern "C" __device__ float __ocml_powr_f32(float, float);

// shaders/tonemap.glsl:18-39 with scale_constant k; an empty texel (a = 0,
// where the shader divides 0/0) maps to black.  Bound by VALU issue: four
// powers of about 160 instructions each; powr in their place takes 3840x2160
// with 8-bit conversion from 117 to 110 us, and at vibrancy 1 one power is
// left.
__device__ __forceinline__ float4 tonemap_px(float4 c, const ToneArgs& t) {
  if (!(c.w > 0.0f)) return make_float4(0.f, 0.f, 0.f, 1.0f);
  // log(1 + a k) through log1pf: the shader's float log(1.0 + a*k) loses most
  // digits when a*k is small (k = 1e-4 makes that every sparse texel).
  const float ls = rf_div_rn(((0.5f * t.brightness) * log1pf(c.w * t.k)) * LOG10E, c.w);
  c.x *= ls; c.y *= ls; c.z *= ls; c.w *= ls;
  float o[3] = {c.x, c.y, c.z};
  const float lo = fminf(fminf(c.x, c.y), fminf(c.z, c.w)), hi = fmaxf(c.x, fmaxf(c.y, c.z));
  if (t.ig > 0.0f && t.ig <= 1.0f && lo >= 0.0f && hi < __builtin_inff()) {
    const float gf = rf_div_rn(__ocml_powr_f32(c.w, t.ig), c.w);
#pragma unroll
    for (int q = 0; q < 3; ++q) {
      const float g = gf * o[q];
      // at vibrancy 1 the power has weight 0 (and is finite: 0 <= o < inf, ig <= 1)
      o[q] = t.vibrancy == 1.0f ? g : rf_mix(__ocml_powr_f32(o[q], t.ig), g, t.vibrancy);
    }
  } else {
    const float gf = rf_div_rn(powf(c.w, t.ig), c.w);
#pragma unroll
    for (int q = 0; q < 3; ++q) o[q] = rf_mix(powf(o[q], t.ig), gf * o[q], t.vibrancy);
  }
#pragma unroll
  for (int q = 0; q < 3; ++q) {
    float v = fminf(fmaxf(o[q], 0.0f), 1.0f);
    if (!(v == v)) v = 0.0f;
    o[q] = v;
  }
  return make_float4(o[0], o[1], o[2], 1.0f);
}

// Batched rendering: the last workgroup of a frame's DE stamps its completion.
// Every thread reaches this point (no early return), so the barrier is safe.
__device__ __forceinline__ void de_stamp(const DEArgs& g) {
  if (!g.done_ts) return;  // kernel argument: uniform
  __syncthreads();
  if (threadIdx.x == 0) {
    __threadfence();
    const uint32_t n = gridDim.x * gridDim.y;
    if (atomicAdd(g.tiles_done, 1u) + 1u == n) {
      const unsigned long long t = wall_clock64();
      __hip_atomic_store(g.done_ts, t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
  }
}

// Chord table, constants of the splat's shape.  rows[i + DE_MAX_R][r]
// describes the row of the radius-r splat that lies i texels from its centre:
// the columns j with a positive weight form the interval [hi - len, hi]
// (hl = hi & 0xff | len << 8, -1 where the splat has no such row), and the
// weight of column hi - b is c - (nx - b * step)^2, the reference's
// (1 - nx^2 - ny^2) * norm with sqrt(norm) folded into nx and step and the
// row's share into c = c[r][i + DE_C_ROW0], which is negative outside the splat.
__device__ __forceinline__ float de_chord_weight(float nx, float c) { return fmaf(-nx, nx, c); }

__global__ __launch_bounds__(DE_CHORD_STRIDE) void k_de_chords(DETable* __restrict__ tab) {
  const int r = (int)threadIdx.x, i = (int)blockIdx.x - DE_C_ROW0;
  DEChord e;
  e.hl = -1; e.nx = 0.0f; e.step = 0.0f; e.pad = 0.0f;
  float c = -1.0f;
  if (r == 0 && i == 0) {
    e.hl = 0; c = 1.0f;
  } else if (r <= DE_MAX_R && i >= -r && i <= r) {
    // the weight's terms in double, rounded once
    const double inv = 1.0 / (double)(2 * r + 1), sn = sqrt((double)M_2_PI_F) / (double)r;
    const double ny = (2.0 * i + inv) * inv;
    e.step = (float)(2.0 * inv * sn);
    c = (float)((1.0 - ny * ny) * sn * sn);
    // the chord's ends in real arithmetic, then inwards to the first positive
    // weight as it is evaluated
    const double half = 0.5 * (double)(2 * r + 1) * sqrt(1.0 - ny * ny);
    auto positive = [&](int j) { return de_chord_weight((float)((2.0 * j + inv) * inv * sn), c) > 0.0f; };
    int hi = min(r, (int)ceil(half)), lo = max(-r, (int)floor(-half) - 1);
    while (hi >= lo && !positive(hi)) --hi;
    while (hi >= lo && !positive(lo)) ++lo;
    e.nx = (float)((2.0 * hi + inv) * inv * sn);
    if (hi >= lo) e.hl = (int)((uint32_t)(hi & 0xff) | ((uint32_t)(hi - lo) << 8));
  }
  if (r <= DE_MAX_R) tab->c[r][blockIdx.x] = c;
  if (i >= -DE_MAX_R && i <= DE_MAX_R) tab->rows[i + DE_MAX_R][r] = e;
}

// Every bin's splat radius: DE_EMPTY for an empty bin, DE_ODD added where the
// bin holds an infinity or NaN.
constexpr uint32_t DE_EMPTY = 255u, DE_ODD = 128u;

__global__ __launch_bounds__(256) void k_de_radius(DEArgs g) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)g.W * g.H) return;
  const float4 c = g.hist[i];
  uint32_t v = DE_EMPTY;
  if (c.w != 0.0f) {
    const float q = rf_div_rn((float)g.R, powf(c.w, g.curve));
    int ri = (q >= (float)g.R) ? g.R : (int)q;
    if (!(q == q)) ri = g.R;
    const int r = max(max(ri, g.rmin), 0);
    // one infinity or NaN makes the sum of the products one
    const float z = fmaf(c.x, 0.0f, fmaf(c.y, 0.0f, fmaf(c.z, 0.0f, c.w * 0.0f)));
    v = (uint32_t)r + (z != 0.0f ? DE_ODD : 0u);
  }
  g.rad[i] = (uint8_t)v;
}

// Density estimation of a 64 x (8 V / S) tile of texels per workgroup of eight
// waves, for any radius up to 100 (bound: VALU issue; for an image of few
// tiles the chain of a wave's source rows, which S waves then share).  A wave
// owns V adjacent texel rows of 64 columns and every S-th of their source rows, so the source row, the radius and the splat rows
// it visits are uniform over the wave: the loop over them runs on the scalar
// unit and the chord table is read with scalar loads.  LDS holds, per source
// row, one column mask per radius (the sources whose radius is exactly r) and
// the radii present, for K source rows at a time.  For a radius present in a
// row a lane shifts the mask to its own column, keeps the bits of the widest
// chord of its V rows (32 columns at a time) and adds the sources they name
// to all V texels: the bit scan, the colour's load and the horizontal part of
// the weight are paid once per source and V texels (27 VALU per source and
// four texels; the same gather texel by texel took 10 to 11 per source), and
// the vertical part is one clamped fma per texel, 0 outside the row's own
// chord.  The colours are read straight from the histogram, where the waves
// of a tile find them in L1 or L2: staged in LDS they limited the tile to
// strips of 16 source rows, between which waves waited (7680x4320 radius 9:
// 1637 us against 1525).  Two sources a round, so that two loads are in
// flight: 1525 -> 1416 us.  Tiles are numbered down their columns: neighbours
// in flight share source rows (2048x2048 radius 9: 286 -> 258 us).
constexpr int DR_W = 64, DR_WAVES = 8;

typedef const __attribute__((address_space(4))) DETable CDETable;
typedef int int4_t __attribute__((ext_vector_type(4)));

// One visit's uniform values: the widest chord and the V rows' shares.
template <int V>
struct DEVisit {
  int hl;
  float nx, step, c[V];
};

// Rows i .. i + V - 1 of radius r, the widest of them row iw.
template <int V>
__device__ __forceinline__ DEVisit<V> de_visit(CDETable* tab, int r, int i, int iw) {
  const int4_t q = *reinterpret_cast<const __attribute__((address_space(4))) int4_t*>(&tab->rows[iw + DE_MAX_R][r]);
  DEVisit<V> v;
  v.hl = q.x;
  v.nx = __int_as_float(q.y);
  v.step = __int_as_float(q.z);
#pragma unroll
  for (int k = 0; k < V; ++k) v.c[k] = tab->c[r][i + DE_C_ROW0 + k];
  return v;
}

// LDS of a source row of the tile: the masks' words per radius, then (in bytes,
// dr_row_bytes) those of all radii and the radii present.
__host__ __device__ inline int dr_mask_words(int R) { return ((DR_W - 1 + 2 * R) >> 5) + 2; }
inline uint64_t dr_tiles(uint32_t W, uint32_t H, int V, int S = 1) {
  const int th = DR_WAVES / S * V;
  return ((uint64_t)W + DR_W - 1) / DR_W * (((uint64_t)H + th - 1) / th);
}
inline size_t dr_row_bytes(int R) {
  return (size_t)(R + 1) * dr_mask_words(R) * 4 + (R < 32 ? 4u : 16u);
}

__device__ __forceinline__ float4 de_source(const float4* row, int x) {
  return *reinterpret_cast<const float4*>(reinterpret_cast<const char*>(row) + (uint32_t)(x << 4));
}

// Adds a source of weight v (none where v <= 0).
template <bool ALL>
__device__ __forceinline__ void de_add(float4& acc, const float4& c, float v) {
  const float w = __builtin_amdgcn_fmed3f(v, 0.0f, 1.0f);
  const bool in = ALL || w > 0.0f;  // a select, not a branch: the sums stay in their registers
  acc.x = fmaf(in ? c.x : 0.0f, w, acc.x);
  acc.y = fmaf(in ? c.y : 0.0f, w, acc.y);
  acc.z = fmaf(in ? c.z : 0.0f, w, acc.z);
  acc.w = fmaf(in ? c.w : 0.0f, w, acc.w);
}

// Adds the sources of one visit to the V texels of this lane.  With ALL the
// sources are finite and a texel outside its row's chord adds 0 of them;
// otherwise it must leave them out (0 * inf).
template <int V, bool ALL, bool SHORT>
__device__ __forceinline__ void de_taps(float4 (&acc)[V], const DEVisit<V>& v, int col0, const uint32_t* em,
                                        const float4* cr) {
  const int len = v.hl >> 8;  // the row is within the radius: never empty
  for (int b0 = 0; SHORT ? b0 == 0 : b0 <= len; b0 += 32) {
    const int col = col0 + b0;
    const uint32_t* const ew = em + (col >> 5);
    uint32_t m = __builtin_amdgcn_alignbit(ew[1], ew[0], col & 31);
    if (SHORT || len - b0 < 31) m &= (2u << (len - b0)) - 1u;
    const float nx0 = fmaf(-(float)b0, v.step, v.nx);
    // two sources a round, so that two loads are in flight
    while (m) {
      const int b = __builtin_ctz(m);
      m &= m - 1u;
      const float4 c = de_source(cr, col + b);
      const bool two = m != 0u;
      const int b2 = two ? __builtin_ctz(m) : b;
      m &= m - 1u;
      const float4 c2 = de_source(cr, col + b2);
      const float nx = fmaf(-(float)b, v.step, nx0);
      // a missing second source lies outside every chord
      const float nx2 = two ? fmaf(-(float)b2, v.step, nx0) : 2.0f;
#pragma unroll
      for (int k = 0; k < V; ++k) {
        de_add<ALL>(acc[k], c, de_chord_weight(nx, v.c[k]));
        de_add<ALL>(acc[k], c2, de_chord_weight(nx2, v.c[k]));
      }
    }
  }
}

// Adds a strip's sources to the wave's V texel rows.
template <int V, int NRW, int S, bool ALL, bool SHORT>
__device__ __forceinline__ void de_strip(float4 (&acc)[V], CDETable* tab, const float4* src, int W, const uint32_t* s_e,
                                         const uint32_t* s_rp, int R, int K, int s0, int rows) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int nwd = dr_mask_words(R), mrow = (R + 1) * nwd;
  // this wave's texel rows lie i0 - k .. i0 - k + V - 1 rows from source row k;
  // it takes every S-th of their source rows
  const int i0 = wave / S * V + R - s0;
  const int k0 = max(0, i0 - R), k1 = min(rows, i0 + V + R);
#pragma unroll
  for (int w = 0; w < NRW; ++w) {
    if (32 * w > R) break;
    // lane k holds the radii present in source row k of the strip
    const int rpv = (int)s_rp[w * K + (lane < rows ? lane : 0)];
    for (int k = k0 + wave % S; k < k1; k += S) {
      const int i = i0 - k;
      const int iw = i > 0 ? i : (i + V - 1 < 0 ? i + V - 1 : 0);  // the row nearest the centre
      const int low = (iw < 0 ? -iw : iw) - 32 * w;
      uint32_t radii = (uint32_t)__builtin_amdgcn_readlane(rpv, k);
      if constexpr (NRW == 1) radii &= ~0u << low;
      else radii = low <= 0 ? radii : (low < 32 ? radii & (~0u << low) : 0u);
      if (!radii) continue;
      const uint32_t* const er = s_e + k * mrow;
      const float4* const cr = src - (ptrdiff_t)(s0 + k) * W;  // bins run bottom-up
      if (SHORT && (radii & 1u)) {
        // radius 0 (iw is 0): the source is its own texel, in one of the rows
        // (above 15 radii are many and this saves less than it costs)
        const int col = lane + R;
        float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
        if (er[col >> 5] >> (col & 31) & 1u) c = de_source(cr, col);
#pragma unroll
        for (int q = 0; q < V; ++q)
          if (q == -i) {  // wave-uniform
            acc[q].x += c.x; acc[q].y += c.y; acc[q].z += c.z; acc[q].w += c.w;
          }
        radii &= ~1u;
        if (!radii) continue;
      }
      int r = 32 * w + __builtin_ctz(radii);
      DEVisit<V> next = de_visit<V>(tab, r, i, iw);
      for (;;) {
        // the next radius' values are on their way while this one's are used
        const DEVisit<V> v = next;
        const uint32_t* const em = er + r * nwd;
        radii &= radii - 1u;
        r = radii ? 32 * w + __builtin_ctz(radii) : r;
        next = de_visit<V>(tab, r, i, iw);
        const int col0 = lane + R - (int)(signed char)(v.hl & 0xff);  // column of j = hi
        de_taps<V, ALL, SHORT>(acc, v, col0, em, cr);
        if (!radii) break;
      }
    }
  }
}

// SHORT: chords of at most 31 columns (radius below 16).  NRW words of 32
// radii each.  S: waves that share a texel row.
template <int V, int NRW, bool SHORT, int S>
__global__ __launch_bounds__(64 * DR_WAVES) __attribute__((amdgpu_waves_per_eu(8))) void k_de_rows(DEArgs g, int K) {
  constexpr int TH = DR_WAVES / S * V;  // texel rows of the tile
  extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
  __shared__ int s_odd;  // the strip holds a source that is not finite
  const int R = max(g.R, g.rmin);  // span
  const int SW = DR_W + 2 * R, nwd = dr_mask_words(R);
  const int mrow = (R + 1) * nwd;  // mask words per source row
  uint32_t* s_e = reinterpret_cast<uint32_t*>(smem);  // [row][radius][word]
  uint32_t* s_rp = s_e + K * mrow;                    // [word][row]
  const int lane = threadIdx.x & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int W = (int)g.W, H = (int)g.H;
  const uint32_t ny = (uint32_t)(H + TH - 1) / TH;
  const uint32_t tile = blockIdx.x;  // down the columns of tiles: neighbours share source rows in L2
  const int tx0 = (int)(tile / ny) * DR_W, ty0 = (int)(tile % ny) * TH;
  CDETable* const tab = (CDETable*)g.tab;
  float4 acc[V];
#pragma unroll
  for (int q = 0; q < V; ++q) acc[q] = make_float4(0.f, 0.f, 0.f, 0.f);
  if (threadIdx.x == 0) s_odd = 0;
  // the bin of source row 0, window column 0 (read only where a mask bit is set)
  const float4* const src = g.hist + ((ptrdiff_t)(H - 1 - ty0 + R) * W + tx0 - R + 1);
  // source row s of the tile is texel row ty0 - R + s of the image
  const int s_begin = max(0, R - ty0), s_end = min(TH + 2 * R, H - ty0 + R);
  for (int s0 = s_begin; s0 < s_end; s0 += K) {  // workgroup-uniform
    const int rows = min(K, s_end - s0);
    __syncthreads();  // the previous strip is read
    // radius of window column x of strip row k, DE_EMPTY outside the image
    // (bins of column 0 have no texel)
    auto radius_at = [&](int k, int x) -> uint32_t {
      const int px = tx0 - R + x + 1;
      if (k >= rows || x >= SW || px < 1 || px >= W) return DE_EMPTY;
      return g.rad[(size_t)(H - 1 - (ty0 - R + s0 + k)) * W + px];
    };
    // this row's masks of 64 columns from x0, one round per radius among them
    auto put_masks = [&](uint32_t* er, uint32_t v, int x0, uint32_t (&rp)[NRW]) {
      const int r = v == DE_EMPTY ? -1 : (int)(v & (DE_ODD - 1u));
      uint64_t left = __builtin_amdgcn_ballot_w64(r >= 0);
      uint32_t* const ex = er + (x0 >> 5);
      const bool put = lane < 2 && (x0 >> 5) + lane < nwd;
      while (left) {
        const int rr = __builtin_amdgcn_readlane(r, __builtin_ctzll(left));
        const uint64_t m = __builtin_amdgcn_ballot_w64(r == rr);
        left &= ~m;
        if (put) ex[rr * nwd + lane] = (uint32_t)(m >> (32 * lane));
        if constexpr (NRW == 1) {
          rp[0] |= 1u << rr;
        } else {
#pragma unroll
          for (int w = 0; w < NRW; ++w) rp[w] |= (rr >> 5) == w ? 1u << (rr & 31) : 0u;
        }
      }
    };
    auto is_odd = [](uint32_t v) { return v != DE_EMPTY && v >= DE_ODD; };
    if constexpr (SHORT) {
      // The 2 R columns beyond the first 64 of several rows in one go: `tw`
      // lanes for each of G rows, a round per radius for all of them.  A pass
      // of its own for each row took nearly half of the masks' time, which at
      // small radii is a third of the kernel's: with this and the shorter way
      // of radius 0 (de_strip) 7680x4320 at 0.3 samples a texel takes 585 us
      // instead of 635 at radius 1, 1130 instead of 1185 at radius 9.
      const int ts = R <= 4 ? 3 : R <= 8 ? 4 : 5, tw = 1 << ts, G = WAVE >> ts;
      bool odd = false;
      uint32_t v0 = radius_at(wave, lane);
      for (int k0 = wave; k0 < rows; k0 += DR_WAVES * G) {
        const int tk = k0 + DR_WAVES * (lane >> ts);
        const uint32_t vt = radius_at(tk, WAVE + (lane & (tw - 1)));
        for (int k = k0; k < min(rows, k0 + DR_WAVES * G); k += DR_WAVES) {
          uint32_t* const er = s_e + k * mrow;
          for (int q = lane; q < mrow; q += WAVE) er[q] = 0u;
          uint32_t rp[NRW] = {0u};
          const uint32_t v = v0;
          v0 = radius_at(k + DR_WAVES, lane);  // the next row's, under way
          odd = odd || is_odd(v);
          put_masks(er, v, 0, rp);
          if (lane == 0) s_rp[k] = rp[0];
        }
        odd = odd || is_odd(vt);
        const int r = vt == DE_EMPTY ? -1 : (int)(vt & (DE_ODD - 1u));
        uint32_t rpt = 0u;
        uint64_t left = __builtin_amdgcn_ballot_w64(r >= 0);
        while (left) {
          const int rr = __builtin_amdgcn_readlane(r, __builtin_ctzll(left));
          const uint64_t m = __builtin_amdgcn_ballot_w64(r == rr);
          left &= ~m;
          const uint32_t bits = (uint32_t)(m >> lane) & (uint32_t)((1ull << tw) - 1ull);
          if ((lane & (tw - 1)) == 0 && bits != 0u) {
            s_e[tk * mrow + rr * nwd + WAVE / 32] = bits;
            rpt |= 1u << rr;
          }
        }
        if (rpt != 0u) s_rp[tk] |= rpt;
      }
      if (odd) s_odd = 1;
    } else {
      uint32_t v0 = radius_at(wave, lane), v1 = radius_at(wave, WAVE + lane);
      for (int k = wave; k < rows; k += DR_WAVES) {
        uint32_t* const er = s_e + k * mrow;
        for (int q = lane; q < mrow; q += WAVE) er[q] = 0u;
        uint32_t rp[NRW];
#pragma unroll
        for (int w = 0; w < NRW; ++w) rp[w] = 0u;
        bool odd = false;
        for (int x0 = 0; x0 < SW; x0 += WAVE) {
          // this row's first 128 columns were loaded during the previous row
          const uint32_t v = x0 == 0 ? v0 : (x0 == WAVE ? v1 : radius_at(k, x0 + lane));
          if (x0 == 0) v0 = radius_at(k + DR_WAVES, lane);
          if (x0 == WAVE) v1 = radius_at(k + DR_WAVES, WAVE + lane);
          odd = odd || is_odd(v);
          put_masks(er, v, x0, rp);
        }
        if (odd) s_odd = 1;
#pragma unroll
        for (int w = 0; w < NRW; ++w)
          if (lane == 0) s_rp[w * K + k] = rp[w];
      }
    }
    __syncthreads();
    if (__builtin_amdgcn_readfirstlane(s_odd) == 0) de_strip<V, NRW, S, true, SHORT>(acc, tab, src, W, s_e, s_rp, R, K, s0, rows);
    else de_strip<V, NRW, S, false, SHORT>(acc, tab, src, W, s_e, s_rp, R, K, s0, rows);
  }
  if constexpr (S > 1) {  // the shares of a row's waves, added in their order
    float4* const s_part = reinterpret_cast<float4*>(smem);  // [q][wave][lane], over the masks
    __syncthreads();  // the last strip is read
#pragma unroll
    for (int q = 0; q < V; ++q) s_part[(q * DR_WAVES + wave) * WAVE + lane] = acc[q];
    __syncthreads();
    if (wave % S == 0) {
#pragma unroll
      for (int q = 0; q < V; ++q)
#pragma unroll
        for (int p = 1; p < S; ++p) {
          const float4 v = s_part[(q * DR_WAVES + wave + p) * WAVE + lane];
          acc[q].x += v.x; acc[q].y += v.y; acc[q].z += v.z; acc[q].w += v.w;
        }
    }
  }
  const int tx = tx0 + lane;
#pragma unroll
  for (int q = 0; q < V; ++q) {
    __builtin_amdgcn_sched_barrier(0);  // one tonemap's registers at a time
    if (wave % S != 0) break;
    const int ty = ty0 + wave / S * V + q;
    if (tx < W && ty < H) {
      const size_t o = (size_t)ty * W + tx;
      if (g.de_out) g.de_out[o] = acc[q];
      if (g.img_out && g.do_tonemap) g.img_out[o] = tonemap_px(acc[q], g.tone);
    }
  }
  de_stamp(g);
}

// Radius 0 everywhere: every bin is its own texel.
__global__ __launch_bounds__(256) void k_de_copy(DEArgs g) {
  const uint32_t tx = blockIdx.x * 64 + (threadIdx.x & 63u), ty = blockIdx.y * 4 + threadIdx.x / 64;
  if (tx < g.W && ty < g.H) {
    float4 c = make_float4(0.f, 0.f, 0.f, 0.f);
    if (tx + 1 < g.W) {
      const float4 b = g.hist[(size_t)(g.H - 1 - ty) * g.W + tx + 1];
      if (b.w != 0.0f) c = b;
    }
    const size_t o = (size_t)ty * g.W + tx;
    if (g.de_out) g.de_out[o] = c;
    if (g.img_out && g.do_tonemap) g.img_out[o] = tonemap_px(c, g.tone);
  }
  de_stamp(g);
}

__global__ void k_tonemap(const float4* __restrict__ in, float4* __restrict__ out, uint32_t n, ToneArgs t) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = tonemap_px(in[i], t);
}

// RGBA float -> RGBA8: clamp to [0, 1], x255, round to nearest (NaN -> 0);
// one thread per pixel, 16 bytes in, 4 bytes out.
__global__ void k_rgba8(const float4* __restrict__ in, uchar4* __restrict__ out, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float4 v = in[i];
  const float c[4] = {v.x, v.y, v.z, v.w};
  uint8_t o[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const float t = c[k] > 0.0f ? (c[k] < 1.0f ? c[k] : 1.0f) : 0.0f;
    o[k] = (uint8_t)(t * 255.0f + 0.5f);
  }
  out[i] = make_uchar4(o[0], o[1], o[2], o[3]);
}

// ------------------------------------------------------------ diagnostics
__global__ void k_eval_xform(const Block* __restrict__ blk, const float* __restrict__ pts,
                             const float* __restrict__ rands, float* __restrict__ out, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  TableRng rng{rands + (size_t)i * 16, 0};
  const XOut o = apply_xform(blk, 0, pts[3 * i], pts[3 * i + 1], pts[3 * i + 2], false, rng);
  out[4 * i + 0] = o.x;
  out[4 * i + 1] = o.y;
  out[4 * i + 2] = o.c;
  out[4 * i + 3] = o.w;
}

__device__ __forceinline__ uint32_t fmix32(uint32_t h) {
  h ^= h >> 16; h *= 0x85ebca6bu; h ^= h >> 13; h *= 0xc2b2ae35u; h ^= h >> 16;
  return h;
}

template <int HM>
__global__ __launch_bounds__(256) void k_atomic_probe(float* bins, uint64_t nbins, uint32_t per_lane,
                                                      const float4* __restrict__ palette) {
  __shared__ float4 s_pal[256];
  s_pal[threadIdx.x] = palette[threadIdx.x];
  __syncthreads();
  const uint32_t t = blockIdx.x * 256u + threadIdx.x;
  for (uint32_t k = 0; k < per_lane; ++k) {
    const uint32_t h = fmix32(t * 0x9E3779B9u ^ (k * 0x632BE5ABu));
    const uint32_t b = (uint32_t)(((uint64_t)h * nbins) >> 32);
    bin_sample<HM>(bins, b, true, h & 255u, 1.0f, s_pal);
  }
}

}  // namespace

__global__ void k_zero_u64(unsigned long long* __restrict__ p, uint32_t n) {
  const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0ull;
}

hipError_t launch_zero_u64(unsigned long long* p, uint32_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero_u64, dim3((n + 255) / 256), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t launch_animate(Block* blocks, uint32_t T, float tss_width, const float* rot, hipStream_t s) {
  hipLaunchKernelGGL(k_animate, dim3(T), dim3(256), 0, s, blocks, T, tss_width, rot);
  return hipGetLastError();
}

hipError_t launch_de_chords(DETable* tab, hipStream_t s) {
  hipLaunchKernelGGL(k_de_chords, dim3(DE_C_ROWS), dim3(DE_CHORD_STRIDE), 0, s, tab);
  return hipGetLastError();
}

// RMAX: the largest radius that is launched with this V and S.
template <int V, int S, int RMAX>
static void launch_de_rows(const DEArgs& a, int R, hipStream_t s) {
  // all source rows of the tile at once while their masks fit 32 KiB (four
  // workgroups per CU, as many as its waves allow)
  const size_t row = dr_row_bytes(R);
  const int K = (int)std::min<size_t>({(size_t)(DR_WAVES / S * V + 2 * R), (size_t)WAVE, (size_t)32768 / row});
  const size_t lds = std::max(K * row, S > 1 ? (size_t)V * DR_WAVES * WAVE * 16 : 0);
  const dim3 grid((unsigned)dr_tiles(a.W, a.H, V, S));
  if (R < 16) {
    hipLaunchKernelGGL((k_de_rows<V, 1, true, S>), grid, dim3(64 * DR_WAVES), lds, s, a, K);
  } else if constexpr (RMAX >= 16) {
    if (R < 32) hipLaunchKernelGGL((k_de_rows<V, 1, false, S>), grid, dim3(64 * DR_WAVES), lds, s, a, K);
    else hipLaunchKernelGGL((k_de_rows<V, 4, false, S>), grid, dim3(64 * DR_WAVES), lds, s, a, K);
  }
}

hipError_t launch_de_tonemap(const DEArgs& a, hipStream_t s) {
  const int R = a.R > a.rmin ? a.R : a.rmin;
  const uint64_t n = (uint64_t)a.W * a.H;
  if (!a.rad || !a.tab || R < 0 || R > DE_MAX_R) return hipErrorInvalidValue;
  if (n == 0) return hipSuccess;
  if (R == 0) {
    hipLaunchKernelGGL(k_de_copy, dim3((a.W + 63) / 64, (a.H + 3) / 4), dim3(256), 0, s, a);
    return hipGetLastError();
  }
  hipLaunchKernelGGL(k_de_radius, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, a);
  // Texel rows per wave (V) and waves per texel row (S), by the 64 x 32 tiles
  // of the image.  Four rows share the most work per source but leave the fewest
  // waves; several waves a row put back the waves, and shorten the chain of
  // source rows that bounds an image of few tiles, for a sum through LDS and
  // masks built for fewer texels.  Measured (us, the tonemap included; V/S):
  //               4/1   4/2   4/4   2/1   2/2   2/8
  //   320x240  R9   63    49    41    49    39    28   (1/1, one wave a row: 44)
  //           R24  180   108    77   141    91    54
  //   900x480  R4   52    50    48    48    43    50
  //            R9   86    74    64    79    66    72
  //           R24  334   215   175   282   225   189
  //   1900x1000 R1  50    56    64    50    57    85
  //            R9  122   109   107   120   111   149
  //           R24  414   316   271   431   338   407
  //   2600x1400 R1  76    93   113    78    98   157
  //            R7  150   151   174   162   171   265
  //           R24  620   522   522   739   677   945
  //   3000x1600 R9 277   284   334   330   356   542
  //           R15  469   443   490   597   603   847
  // and at 5000x2700 radius 15 857 with 4/1.
  const uint64_t t = dr_tiles(a.W, a.H, 4);
  if (t < 192) launch_de_rows<2, 8, DE_MAX_R>(a, R, s);
  else if (R < 4 && t < 2560) launch_de_rows<2, 1, 3>(a, R, s);
  else if (t < 1280 && R < 9) launch_de_rows<2, 2, 8>(a, R, s);
  else if (t < 1280) launch_de_rows<4, 4, DE_MAX_R>(a, R, s);
  else if (t < 4096 && R >= 12) launch_de_rows<4, 2, DE_MAX_R>(a, R, s);
  else launch_de_rows<4, 1, DE_MAX_R>(a, R, s);
  return hipGetLastError();
}

hipError_t launch_tonemap(const float4* in, float4* out, uint32_t n, const ToneArgs& t, hipStream_t s) {
  hipLaunchKernelGGL(k_tonemap, dim3((n + 255) / 256), dim3(256), 0, s, in, out, n, t);
  return hipGetLastError();
}

hipError_t launch_rgba8(const float4* in, uchar4* out, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_rgba8, dim3((n + 255) / 256), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t launch_eval_xform(const Block* blk, const float* pts, const float* rands, float* out,
                             uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_eval_xform, dim3((n + 255) / 256), dim3(256), 0, s, blk, pts, rands, out, n);
  return hipGetLastError();
}

hipError_t launch_atomic_probe(float* bins, uint64_t nbins, uint64_t samples, int hm,
                               const float4* palette, hipStream_t s) {
  const uint32_t per_lane = 64;
  const uint64_t lanes = samples / per_lane;
  dim3 grid((uint32_t)(lanes / 256u)), block(256);
  switch (hm) {
    case 2: hipLaunchKernelGGL(k_atomic_probe<2>, grid, block, 0, s, bins, nbins, per_lane, palette); break;
    case 3: hipLaunchKernelGGL(k_atomic_probe<3>, grid, block, 0, s, bins, nbins, per_lane, palette); break;
    default: hipLaunchKernelGGL(k_atomic_probe<1>, grid, block, 0, s, bins, nbins, per_lane, palette); break;
  }
  return hipGetLastError();
}

}  // namespace rfk
