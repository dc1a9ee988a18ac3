// Denoiser network kernels (gfx950): bf16 MFMA convolutions with fp32
// accumulation, weight gradients, pooling, loss and Adam.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "rf_nn.hpp"

namespace rfn {
namespace {

typedef short short4_t __attribute__((ext_vector_type(4)));
typedef float float4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float bf2f(bf16 h) { return __uint_as_float((uint32_t)h << 16); }

// Round to nearest even; NaN stays NaN.  (v_cvt_pk_bf16_f32; the same bits as
// rounding by integer arithmetic for every value but NaN.)
typedef float float2_t __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t f2bf2(float lo, float hi) {
  const float2_t v = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2_t));
}
__device__ __forceinline__ bf16 f2bf(float f) { return (bf16)f2bf2(f, 0.0f); }

// Workgroup barrier that orders LDS only: __syncthreads() would also wait for
// every global load and store under way.
__device__ __forceinline__ void lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// ------------------------------------------------------------ convolution
// Implicit GEMM: M = pixels, N = output channels, K = 9 * Cin.  A workgroup
// of 4 waves covers 64 consecutive pixels of one image row (16 per wave) and
// 16*NT output channels.  Per (r, s, 16-channel step) each wave issues NT
// v_mfma_f32_16x16x16_bf16 with one A fragment (16 pixels x 16 channels) and
// NT B fragments (16 channels x 16 outputs).  Operand layout of that
// instruction (wave64): lane l holds A[l % 16][4 (l / 16) + e] and
// B[4 (l / 16) + e][l % 16] for e = 0..3, and D[4 (l / 16) + e][l % 16].
// NHWC activations and [r][s][Cout][Cin] weights make both fragments one
// 8-byte load per lane.
template <int NT>
__global__ __launch_bounds__(256) void k_conv3x3(View in, const bf16* __restrict__ w, const float* __restrict__ bias,
                                                 View out, int H, int W, int Cin, int Cout, int relu) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int n = blockIdx.y / H, y = blockIdx.y % H;
  const int x0 = blockIdx.x * 64 + wave * 16;
  const int co0 = blockIdx.z * 16 * NT;
  const int i = lane & 15, kq = lane >> 4;
  float4_t acc[NT];
#pragma unroll
  for (int t = 0; t < NT; ++t) acc[t] = float4_t{0.f, 0.f, 0.f, 0.f};
  const int xa = x0 + i;
  for (int r = 0; r < 3; ++r) {
    const int yy = y + r - 1;
    const bool rok = yy >= 0 && yy < H;
    for (int s = 0; s < 3; ++s) {
      const int xx = xa + s - 1;
      const bool ok = rok && xx >= 0 && xx < W;
      const bf16* ap = in.p + ((size_t)(n * H + (rok ? yy : 0)) * W + (ok ? xx : 0)) * in.cs + in.co + 4 * kq;
      const bf16* wp = w + ((size_t)(r * 3 + s) * Cout + co0 + i) * Cin + 4 * kq;
      for (int c0 = 0; c0 < Cin; c0 += 16) {
        short4_t a = short4_t{0, 0, 0, 0};
        if (ok) a = *reinterpret_cast<const short4_t*>(ap + c0);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const short4_t b = *reinterpret_cast<const short4_t*>(wp + (size_t)t * 16 * Cin + c0);
          acc[t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc[t], 0, 0, 0);
        }
      }
    }
  }
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int co = co0 + 16 * t + i;
    const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int px = x0 + 4 * kq + e;
      if (px < W) {
        float v = acc[t][e] + bv;
        if (relu) v = fmaxf(v, 0.0f);
        out.p[((size_t)(n * H + y) * W + px) * out.cs + out.co + co] = f2bf(v);
      }
    }
  }
}

__device__ __forceinline__ float bf_lo(uint32_t u) { return __uint_as_float(u << 16); }
__device__ __forceinline__ float bf_hi(uint32_t u) { return __uint_as_float(u & 0xffff0000u); }

// LDS-tiled implicit GEMM.  A workgroup of 4 waves covers 4 RW image rows
// x CT_W = 64 pixels (RW rows per wave, four 16-pixel A fragments per row) and
// 16*NT output channels.  Per KC-channel step of Cin (KC = 32 with gfx950's
// v_mfma_f32_16x16x32_bf16 for the wide layers, else 16 with the 16x16x16 form)
// it stages the (4 RW + 2) x (CT_W + 2) input patch (zero halo) and the
// step's 3x3 x 16*NT x KC weights in LDS (strides: ConvStage); every A fragment then feeds NT MFMAs and every B
// fragment four per output row it reaches.  With RW = 2 a wave's four input
// rows serve six (row, tap row) pairs, so each A fragment read from LDS feeds
// up to 2 NT MFMAs: the narrow layers, whose NT is small, read a third fewer
// A fragments and half the B fragments per output.  The next step's operands
// are loaded into registers while the MFMAs of the current one run.  Needs
// 16-byte aligned channel runs (Cin, channel strides and offsets multiples of
// 8).  At 1024^2 the 192 -> 64 layer takes 269 us and the 384 -> 128 layer at
// 512^2 207 us (860 and 1120 TFLOP/s, the latter near a large matrix
// product's rate on this card); with places and bounds recomputed every step,
// LDS rows of 80 bytes and fragments read as they were needed 287 and 232.
// Operand layouts (wave64, i = lane % 16, kq = lane / 16): 16x16x16 lane
// holds A[i][4 kq + e], B[4 kq + e][i] (e < 4); 16x16x32 lane holds
// A[i][8 kq + e], B[8 kq + e][i] (e < 8); both give D[4 kq + e][i] (e < 4).
constexpr int CT_W = 64;
// staged input pixels of a tile of 4 RW rows
__host__ __device__ constexpr int ct_in_pix(int RW) { return (4 * RW + 2) * (CT_W + 2); }

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));

template <int NT, int KC, int RW>
struct ConvStage {
  // LDS strides (bf16) of a pixel and of a weight row.  A 16-byte LDS read of
  // a wave takes four cycles when each of its groups of 16 lanes (lanes 0..3,
  // 12..15 and 20..27, and so on) covers all banks, else eight or more: the
  // 16 lanes of a fragment and the four 16-byte pieces of their rows do so at
  // 96 bytes a row, or at 64 with the pieces swizzled (w_piece) where rows
  // start at multiples of 16.  80 bytes, the smallest odd multiple of 16,
  // take eight.
  static constexpr int PS = KC == 32 ? 48 : 24, WS = KC == 32 ? 32 : 24;
  static __device__ __forceinline__ int w_piece(int row, int piece) {
    return KC == 32 ? piece ^ (-(row >> 2) & 3) : piece;
  }
  static constexpr int PQ = KC / 8;             // 16-byte pieces per pixel / weight row
  static constexpr int IN_Q = ct_in_pix(RW) * PQ;
  static constexpr int W_Q = 9 * 16 * NT * PQ;
  static constexpr int IN_PER = (IN_Q + 255) / 256;
  static constexpr int W_PER = (W_Q + 255) / 256;
  uint4 vin[IN_PER];
  uint4 vw[W_PER];
  uint32_t place[IN_PER];  // see conv_places
};

// Buffer loads: an offset at or beyond BUF_RANGE reads zeros, which is how the
// halo outside the image is filled without branches.
constexpr uint32_t BUF_RANGE = 0x7fffffffu, BUF_NONE = 0x80000000u;
typedef uint32_t uint4_t __attribute__((ext_vector_type(4)));
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_at(const bf16* p) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<bf16*>(p), 0, (int)BUF_RANGE, 0x00020000);
}
__device__ __forceinline__ uint4 buf_load(__amdgpu_buffer_rsrc_t r, uint32_t lane, uint32_t uniform) {
  const uint4_t v = __builtin_amdgcn_raw_buffer_load_b128(r, (int)lane, (int)uniform, 0);
  return make_uint4(v.x, v.y, v.z, v.w);
}

// This thread's input pieces in `in`, or (up = 1) in the half-resolution `up`:
// bytes from the patch's first pixel or (FAR, where 32 bits need not hold them)
// row, column and piece; BUF_NONE outside the image.  They are computed once per view and
// tile: recomputed for every channel step, places and bounds were 300 vector
// instructions a wave and step beside 144 MFMAs.
template <int NT, int KC, int RW, bool FAR>
__device__ __forceinline__ void conv_places(ConvStage<NT, KC, RW>& st, int cs, int up, int y0, int x0, int H, int W) {
  using S = ConvStage<NT, KC, RW>;
#pragma unroll
  for (int k = 0; k < S::IN_PER; ++k) {
    const int q = (int)threadIdx.x + 256 * k;
    const int piece = q % S::PQ, pix = q / S::PQ;
    const int yy = y0 + pix / (CT_W + 2) - 1, gx = x0 + pix % (CT_W + 2) - 1;
    // (from the patch's row y0 - 1, column x0 - 1, halved with rounding down for `up`)
    const uint32_t dy = (uint32_t)((yy >> up) - ((y0 - 1) >> up)), dx = (uint32_t)((gx >> up) - ((x0 - 1) >> up));
    const bool in_image = q < S::IN_Q && yy >= 0 && yy < H && gx >= 0 && gx < W;
    const uint32_t at = FAR ? dy << 10 | dx << 3 | (uint32_t)piece
                            : 16u * ((dy * (uint32_t)(W >> up) + dx) * (uint32_t)(cs / 8) + (uint32_t)piece);
    st.place[k] = in_image ? at : BUF_NONE;
  }
}

// A 16-byte piece (the piece-th of a pixel `pixels` pixels behind the first) of
// a row: its place, BUF_NONE for zeros, and its load.  FAR: 64-bit addresses, at
// any channel stride.
template <bool FAR>
__device__ __forceinline__ uint32_t piece_place(int pixels, int cs, int piece) {
  return FAR ? (uint32_t)(16 * pixels + piece) : 2u * (uint32_t)(pixels * cs + 8 * piece);
}
template <bool FAR>
__device__ __forceinline__ uint4 piece_load(const bf16* row, int cs, uint32_t place) {
  if constexpr (FAR) {
    uint4 v = make_uint4(0u, 0u, 0u, 0u);
    if (place != BUF_NONE) v = *reinterpret_cast<const uint4*>(row + (size_t)(place / 16) * cs + 8 * (place % 16));
    return v;
  }
  return buf_load(buf_at(row), place, 0);
}

// The loads of one channel step.  Channels [0, Cup) come from the
// half-resolution `up` (nearest-neighbour upsampling read in place), the rest
// from `in`; a KC step never straddles the two (Cup is a multiple of 32).
// `src` is the patch's first pixel in the step's view of `width` columns and
// channel stride cs, c its first channel.
template <int NT, int KC, int RW, bool FAR>
__device__ __forceinline__ void conv_load(ConvStage<NT, KC, RW>& st, const bf16* src, int width, int cs, int c,
                                          const bf16* w, int c0, int Cin, int Cout) {
  using S = ConvStage<NT, KC, RW>;
  // weight row = tap * 16 NT + output channel; a round of 256 threads covers
  // whole taps
  constexpr int ROWS = 256 / S::PQ, TAPS = ROWS / (16 * NT);
  static_assert(TAPS * 16 * NT == ROWS, "whole taps");
  const int row0 = (int)threadIdx.x / S::PQ, piece = (int)threadIdx.x % S::PQ;
  if constexpr (FAR) {
#pragma unroll
    for (int k = 0; k < S::IN_PER; ++k) {
      st.vin[k] = make_uint4(0u, 0u, 0u, 0u);
      if (st.place[k] != BUF_NONE)
        st.vin[k] = *reinterpret_cast<const uint4*>(
            src + ((size_t)(st.place[k] >> 10) * width + (st.place[k] >> 3 & 127u)) * cs + 8 * (st.place[k] & 7u) + c);
    }
#pragma unroll
    for (int k = 0; k < S::W_PER; ++k) {
      st.vw[k] = make_uint4(0u, 0u, 0u, 0u);
      if ((int)threadIdx.x + 256 * k < S::W_Q)
        st.vw[k] = *reinterpret_cast<const uint4*>(
            w + ((size_t)(k * TAPS + row0 / (16 * NT)) * Cout + row0 % (16 * NT)) * Cin + c0 + 8 * piece);
    }
    return;
  }
  const __amdgpu_buffer_rsrc_t rin = buf_at(src), rw = buf_at(w);
#pragma unroll
  for (int k = 0; k < S::IN_PER; ++k) st.vin[k] = buf_load(rin, st.place[k], 2u * (uint32_t)c);
  const uint32_t lane = 2u * (uint32_t)((row0 / (16 * NT) * Cout + row0 % (16 * NT)) * Cin + 8 * piece);
#pragma unroll
  for (int k = 0; k < S::W_PER; ++k) {
    const bool some = S::W_Q >= 256 * (k + 1) || (int)threadIdx.x + 256 * k < S::W_Q;
    st.vw[k] = buf_load(rw, some ? lane : BUF_NONE, 2u * (uint32_t)(k * TAPS * Cout * Cin + c0));
  }
}

// One lane's operand fragment: 4 (16x16x16) or 8 (16x16x32) bf16 values.
template <int KC>
struct ConvFrag;
template <>
struct ConvFrag<16> {
  typedef short4_t T;
  static __device__ __forceinline__ float4_t mfma(T a, T b, float4_t acc) {
    return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(a, b, acc, 0, 0, 0);
  }
};
template <>
struct ConvFrag<32> {
  typedef bf16x8_t T;
  static __device__ __forceinline__ float4_t mfma(T a, T b, float4_t acc) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, acc, 0, 0, 0);
  }
};

// Two bf16 values, each kept where the other word's value in its place is
// positive (ReLU's backward).
__device__ __forceinline__ uint32_t relu_keep(uint32_t v, uint32_t y) {
  const uint32_t lo = bf_lo(y) > 0.0f ? 0xffffu : 0u, hi = bf_hi(y) > 0.0f ? 0xffff0000u : 0u;
  return v & (lo | hi);
}
__device__ __forceinline__ uint2 relu_keep(const uint2& v, const uint2& y) {
  return make_uint2(relu_keep(v.x, y.x), relu_keep(v.y, y.y));
}
__device__ __forceinline__ uint4 relu_keep(const uint4& v, const uint4& y) {
  return make_uint4(relu_keep(v.x, y.x), relu_keep(v.y, y.y), relu_keep(v.z, y.z), relu_keep(v.w, y.w));
}

// Output of one tile: bias, ReLU and bf16 in LDS (tile row RW * wave + rr is
// image row y0 + RW * wave + rr), then 16-byte stores per pixel, the fused
// 2x2 averages or the fused fp32 residual.  The output tile reuses the
// staging buffer: the caller's next step waits on a barrier before staging.
template <int NT, int RW>
__device__ __forceinline__ void conv_store_lds(const float4_t (&acc)[RW][4][NT], bf16* s_buf,
                                               const float* __restrict__ bias, const View& out, const ConvFuse& fz,
                                               int relu, int n, int y0, int x0, int co0, int H, int W) {
  constexpr int OC = 16 * NT, OS = OC + 8, TR = 4 * RW;
  constexpr int PQ = OC / 8;  // 16-byte pieces per pixel
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i = lane & 15, kq = lane >> 4;
  __syncthreads();  // the last step's fragment reads are done: the staging buffer is free
#pragma unroll
  for (int rr = 0; rr < RW; ++rr) {
    bf16* const s_o = s_buf + (RW * wave + rr) * CT_W * OS;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const float bv = bias ? bias[co0 + 16 * t + i] : 0.0f;
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          float v = acc[rr][f][t][e] + bv;
          if (relu) v = fmaxf(v, 0.0f);
          s_o[(16 * f + 4 * kq + e) * OS + 16 * t + i] = f2bf(v);
        }
    }
  }
  __syncthreads();
  if (fz.y) {  // workgroup-uniform: the residual output replaces `out`
    const int px = x0 + lane;
#pragma unroll
    for (int rr = 0; rr < RW; ++rr) {
      const int y = y0 + RW * wave + rr;
      if (y < H && px < W) {
        const size_t p = (size_t)(n * H + y) * W + px;
        const uint2 xv = *reinterpret_cast<const uint2*>(fz.res.p + p * fz.res.cs + fz.res.co);
        const uint2 ov = *reinterpret_cast<const uint2*>(s_buf + ((RW * wave + rr) * CT_W + lane) * OS);
        *reinterpret_cast<float4*>(fz.y + p * 4) =
            make_float4(bf_lo(xv.x) + bf_lo(ov.x), bf_hi(xv.x) + bf_hi(ov.x), bf_lo(xv.y) + bf_lo(ov.y),
                        bf_hi(xv.y) + bf_hi(ov.y));
      }
    }
  } else {
    const bool down = co0 < fz.Cdown;  // workgroup-uniform
#pragma unroll
    for (int rr = 0; rr < RW; ++rr) {
      const int y = y0 + RW * wave + rr;
      const bf16* const s_o = s_buf + (RW * wave + rr) * CT_W * OS;
      if (y < H && !down) {
#pragma unroll
        for (int q = lane; q < CT_W * PQ; q += 64) {
          const int px = q / PQ, piece = q % PQ;
          if (x0 + px < W) {
            const size_t p = (size_t)(n * H + y) * W + x0 + px;
            uint4 v = *reinterpret_cast<const uint4*>(s_o + px * OS + 8 * piece);
            if (fz.mask.p)  // workgroup-uniform
              v = relu_keep(v, *reinterpret_cast<const uint4*>(fz.mask.p + p * fz.mask.cs + fz.mask.co + co0 + 8 * piece));
            *reinterpret_cast<uint4*>(out.p + p * out.cs + out.co + co0 + 8 * piece) = v;
          }
        }
      }
    }
    // workgroup-uniform: the tile's 2x2 averages or masked sums, added in
    // k_avgpool2_v8's order
    if (fz.pool.p || down) {
      const View pool = down ? fz.down : fz.pool;
      const float scale = down ? 1.0f : 0.25f;
      constexpr int PW = CT_W / 2, NPQ = (TR / 2) * PW * PQ;
      for (int q = tid; q < NPQ; q += 256) {
        const int piece = q % PQ, pp = (q / PQ) % PW, pr = q / (PQ * PW);
        const int yo = (y0 >> 1) + pr, xo = (x0 >> 1) + pp;
        if (yo < (H >> 1) && xo < (W >> 1)) {
          float sum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
          for (int a = 0; a < 2; ++a)
#pragma unroll
            for (int b = 0; b < 2; ++b) {
              const uint4 v =
                  *reinterpret_cast<const uint4*>(s_buf + (2 * pr + a) * CT_W * OS + (2 * pp + b) * OS + 8 * piece);
              const uint32_t qv[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
              for (int k = 0; k < 4; ++k) { sum[2 * k] += bf_lo(qv[k]); sum[2 * k + 1] += bf_hi(qv[k]); }
            }
          uint32_t r[4];
#pragma unroll
          for (int k = 0; k < 4; ++k)
            r[k] = f2bf2(scale * sum[2 * k], scale * sum[2 * k + 1]);
          const size_t p = (size_t)(n * (H >> 1) + yo) * (W >> 1) + xo;
          uint4 v = make_uint4(r[0], r[1], r[2], r[3]);
          if (down)
            v = relu_keep(v, *reinterpret_cast<const uint4*>(fz.down_mask.p + p * fz.down_mask.cs + fz.down_mask.co + co0 +
                                                             8 * piece));
          *reinterpret_cast<uint4*>(pool.p + p * pool.cs + pool.co + co0 + 8 * piece) = v;
        }
      }
    }
  }
}

// One workgroup per tile (x block, row block of 4 RW rows of image n, 16 NT
// output channel block): workgroup t has channel block t % nbz, x block
// (t / nbz) % nbx and row block t / (nbz nbx), so the workgroups that read
// the same input patch for different output channels run next to each other.
// (A persistent variant, each workgroup walking tiles b, b + G, ... with the
// next tile's first step prefetched during the last step of the current one,
// and outputs stored straight from the accumulators, took 10 % fewer cycles on
// the wide layers but 1 % less time, the clock falling as the stalls went, and
// 10 % more time on the 64 -> 32 layer.)
template <int NT, int KC, int RW, bool FAR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(RW == 2 ? (KC == 16 ? 3 : 2) : 1))) void k_conv3x3_lds(
    View in, const bf16* __restrict__ w, const float* __restrict__ bias, View out, int H, int W, int Cin, int Cout,
    int relu, int vec_out, ConvFuse fz, int nbx, int nbz, int n_tiles) {
  const View& up = fz.up;
  const int Cup = fz.Cup;
  using S = ConvStage<NT, KC, RW>;
  using F = ConvFrag<KC>;
  constexpr int PS = S::PS, WS = S::WS, KE = KC / 4;  // fragment elements per lane
  constexpr int OC = 16 * NT, OS = OC + 8;  // output tile: channels per pixel, LDS row stride
  constexpr int TR = 4 * RW;                // tile rows
  constexpr int IN_PIX = ct_in_pix(RW);
  static_assert(TR * CT_W * OS <= IN_PIX * PS + 9 * 16 * NT * WS, "output tile fits the staging buffer");
  __shared__ __attribute__((aligned(16))) bf16 s_buf[IN_PIX * PS + 9 * 16 * NT * WS];
  bf16* const s_in = s_buf;
  bf16* const s_w = s_buf + IN_PIX * PS;
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int nrb = (H + TR - 1) / TR;
  const int i = lane & 15, kq = lane >> 4;
  const int tile = blockIdx.x;
  if (tile >= n_tiles) return;  // workgroup-uniform
  const int bz = tile % nbz, rest = tile / nbz;
  const int bx = rest % nbx, by = rest / nbx;
  const int n = by / nrb, y0 = (by % nrb) * TR, x0 = bx * CT_W, co0 = bz * 16 * NT;
  // this lane's channels of a weight row (rows 16 t + i)
  const int wk = KC == 32 ? 8 * S::w_piece(i, kq) : KE * kq;
  float4_t acc[RW][4][NT];
#pragma unroll
  for (int rr = 0; rr < RW; ++rr)
#pragma unroll
    for (int f = 0; f < 4; ++f)
#pragma unroll
      for (int t = 0; t < NT; ++t) acc[rr][f][t] = float4_t{0.f, 0.f, 0.f, 0.f};
  S st;
  // the patch's first pixel in each view (outside the image for a tile at its
  // edge), the pieces' places in the view being read, the weights
  auto patch = [&](const View& v, int u) {
    return v.p + ((ptrdiff_t)(n * (H >> u) + ((y0 - 1) >> u)) * (W >> u) + ((x0 - 1) >> u)) * v.cs + v.co;
  };
  const bf16* const wsrc = w + (size_t)co0 * Cin;
  const bf16* src = Cup ? patch(up, 1) : patch(in, 0);
  conv_places<NT, KC, RW, FAR>(st, Cup ? up.cs : in.cs, Cup ? 1 : 0, y0, x0, H, W);
  conv_load<NT, KC, RW, FAR>(st, src, Cup ? W >> 1 : W, Cup ? up.cs : in.cs, 0, wsrc, 0, Cin, Cout);
  for (int c0 = 0; c0 < Cin; c0 += KC) {
    __syncthreads();  // the previous step's fragment reads are done
#pragma unroll
    for (int k = 0; k < S::IN_PER; ++k) {
      const int q = tid + 256 * k;
      if (q < S::IN_Q) *reinterpret_cast<uint4*>(s_in + (q / S::PQ) * PS + 8 * (q % S::PQ)) = st.vin[k];
    }
#pragma unroll
    for (int k = 0; k < S::W_PER; ++k) {
      const int q = tid + 256 * k;
      if (q < S::W_Q) *reinterpret_cast<uint4*>(s_w + (q / S::PQ) * WS + 8 * S::w_piece(q / S::PQ, q % S::PQ)) = st.vw[k];
    }
    __syncthreads();
    if (c0 + KC < Cin) {
      if (c0 + KC == Cup) {  // on to the other view
        src = patch(in, 0);
        conv_places<NT, KC, RW, FAR>(st, in.cs, 0, y0, x0, H, W);
      }
      const bool of_up = c0 + KC < Cup;
      conv_load<NT, KC, RW, FAR>(st, src, of_up ? W >> 1 : W, of_up ? up.cs : in.cs, of_up ? c0 + KC : c0 + KC - Cup,
                                 wsrc, c0 + KC, Cin, Cout);
    }
    // A fragment's LDS read takes as long as several MFMAs: the next group's
    // are under way while a group runs (and no more, for the registers; left
    // to itself the compiler reads them two at a time and waits for each).
    typedef typename F::T Frag;
    if constexpr (RW == 1) {
      // group = tap
      Frag a[2][4], b[2][NT];
      auto frags = [&](int tap) {
        const bf16* ap = s_in + ((wave + tap / 3) * (CT_W + 2) + i + tap % 3) * PS + KE * kq;
        const bf16* bp = s_w + (tap * 16 * NT + i) * WS + wk;
#pragma unroll
        for (int f = 0; f < 4; ++f) a[tap & 1][f] = *reinterpret_cast<const Frag*>(ap + 16 * f * PS);
#pragma unroll
        for (int t = 0; t < NT; ++t) b[tap & 1][t] = *reinterpret_cast<const Frag*>(bp + 16 * t * WS);
      };
      frags(0);
#pragma unroll
      for (int tap = 0; tap < 9; ++tap) {
        if (tap + 1 < 9) frags(tap + 1);
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int t = 0; t < NT; ++t) acc[0][f][t] = F::mfma(a[tap & 1][f], b[tap & 1][t], acc[0][f][t]);
        __builtin_amdgcn_sched_barrier(0);
      }
    } else {
      // Staged input row j of the wave's RW + 2 rows is tap row r = j - rr
      // of its output row rr: per tap column s, the 3 NT B fragments are
      // read once and every A fragment once, for all the rows it reaches.
      // Group = (tap column, input row).
      constexpr int G = 3 * (RW + 2);
      Frag a[2][4], b[2][3][NT];
      auto frags_a = [&](int g) {
        const bf16* ap = s_in + ((RW * wave + g % (RW + 2)) * (CT_W + 2) + i + g / (RW + 2)) * PS + KE * kq;
#pragma unroll
        for (int f = 0; f < 4; ++f) a[g & 1][f] = *reinterpret_cast<const Frag*>(ap + 16 * f * PS);
      };
      auto frags_b = [&](int s, int r) {
#pragma unroll
        for (int t = 0; t < NT; ++t)
          b[s & 1][r][t] = *reinterpret_cast<const Frag*>(s_w + ((r * 3 + s) * 16 * NT + 16 * t + i) * WS + wk);
      };
      frags_a(0);
#pragma unroll
      for (int r = 0; r < 3; ++r) frags_b(0, r);
#pragma unroll
      for (int g = 0; g < G; ++g) {
        const int s = g / (RW + 2), j = g % (RW + 2);
        if (g + 1 < G) frags_a(g + 1);
        if (s < 2 && j > 0) frags_b(s + 1, j - 1);
#pragma unroll
        for (int f = 0; f < 4; ++f)
#pragma unroll
          for (int rr = 0; rr < RW; ++rr) {
            const int r = j - rr;
            if (r >= 0 && r < 3) {
#pragma unroll
              for (int t = 0; t < NT; ++t) acc[rr][f][t] = F::mfma(a[g & 1][f], b[s & 1][r][t], acc[rr][f][t]);
            }
          }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
  }
  if (vec_out) {  // workgroup-uniform
    conv_store_lds<NT, RW>(acc, s_buf, bias, out, fz, relu, n, y0, x0, co0, H, W);
  } else {
#pragma unroll
    for (int rr = 0; rr < RW; ++rr) {
      const int y = y0 + RW * wave + rr;
      if (y < H) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          const int co = co0 + 16 * t + i;
          const float bv = bias ? bias[co] : 0.0f;
#pragma unroll
          for (int f = 0; f < 4; ++f) {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int px = x0 + 16 * f + 4 * kq + e;
              if (px < W) {
                float v = acc[rr][f][t][e] + bv;
                if (relu) v = fmaxf(v, 0.0f);
                out.p[((size_t)(n * H + y) * W + px) * out.cs + out.co + co] = f2bf(v);
              }
            }
          }
        }
      }
    }
  }
}

// Persistent convolution of the narrow layers (Cin 16 or 32, at most 32
// output channels per block), which memory bounds (a 32 -> 32 layer at 2048^2
// moves 537 MB for 77 GFLOP).  A workgroup of 4 waves keeps its 9 x Cin x
// 16 NT weights in registers and walks tiles of 8 rows x 64 pixels, first
// tile blockIdx / nbz, step gridDim / nbz; the next tile's input (halo
// included) is loaded into registers while the MFMAs of the current one run,
// so loads are in flight all the time, and only the input goes through LDS.
// The weights are the A operand: a lane's four (NT = 1) or eight consecutive
// output channels of one pixel leave as one store, without LDS; for NT = 2
// fragment t's row m is channel 8 (m / 4) + 4 t + m % 4, which makes the
// eight consecutive.
//
// Every output sums 16-channel products in k_conv3x3_lds<NT, 16, 2>'s order
// (input channel halves, then tap columns, then tap rows) and has its bits:
// v_mfma_f32_16x16x32_bf16 adds its first sixteen products, then the others,
// exactly as two chained 16x16x16 instructions do, so two successive taps
// share one instruction at twice the rate.  Lanes 0..31 hold the first tap's
// eight channels each, lanes 32..63 the second's: in a pair of successive
// taps the second lies one of three distances behind the first, and with one
// base address for each all fragment offsets are constants.
//
// One tile a workgroup (k_conv3x3_lds) exposes each tile's first load and its
// store: at 2048^2 the 16 -> 32, 32 -> 32 and 32 -> 16 layers took 132, 206
// and 116 us there and take 98, 144 and 98 us here (3.7 to 4.1 TB/s).
constexpr int CF_PIX = ct_in_pix(2);

template <int NT>
constexpr int conv_few_waves() { return NT == 2 ? 2 : 3; }  // workgroups per CU, by registers

// DOWN: the launch has fz.Cdown (and no mask or pool, whose registers it would
// not leave).
template <int CIN, int NT, bool RELU, bool DOWN>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(conv_few_waves<NT>()))) void k_conv3x3_few(
    View in, const bf16* __restrict__ w, const float* __restrict__ bias, View out, int H, int W, int Cout,
    ConvFuse fz, int nbx, int nbz, int n_tiles) {
  // (strides as in ConvStage; three workgroups of <32, 1> fit LDS at 80 bytes only)
  constexpr int PQ = CIN / 8, PS = CIN == 16 ? 16 : NT == 2 ? 48 : 40, PW = CT_W + 2;
  constexpr int IN_Q = CF_PIX * PQ, IN_PER = (IN_Q + 255) / 256;
  constexpr int NP = 9 * CIN / 16, NQ = NP / 2;  // products of 16 channels and pairs of them per output
  __shared__ __attribute__((aligned(16))) bf16 s_in[CF_PIX * PS];
  __shared__ __attribute__((aligned(16))) float s_bias[16 * NT];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int i = lane & 15, kq = lane >> 4;
  const int nrb = (H + 7) / 8;
  const int bz = blockIdx.x % nbz, step = gridDim.x / nbz;
  const int co0 = bz * 16 * NT;
  const bool hi = kq >= 2;
  // product p: channel half, tap column, tap row
  auto half = [](int p) { return p / 9; };
  auto tap = [](int p) { return (p % 3) * 3 + (p % 9) / 3; };
  auto at = [&](int p) { return ((p % 3) * PW + (p % 9) / 3) * PS + 16 * half(p); };

  bf16x8_t wf[NQ][NT];
  short4_t wl[NT];  // the odd product's weights
#pragma unroll
  for (int t = 0; t < NT; ++t) {
    const int co = co0 + (NT == 2 ? 8 * (i >> 2) + 4 * t + (i & 3) : i);
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
      const bf16* const wa = w + ((size_t)tap(2 * q) * Cout + co) * CIN + 16 * half(2 * q);
      const bf16* const wb = w + ((size_t)tap(2 * q + 1) * Cout + co) * CIN + 16 * half(2 * q + 1);
      wf[q][t] = *reinterpret_cast<const bf16x8_t*>((hi ? wb : wa) + 8 * (kq & 1));
    }
    if constexpr (NP % 2)
      wl[t] = *reinterpret_cast<const short4_t*>(w + ((size_t)tap(NP - 1) * Cout + co) * CIN + 4 * kq);
  }
  if (tid < 16 * NT) s_bias[tid] = bias ? bias[co0 + tid] : 0.0f;
  // four outputs of one pixel: bias, ReLU, bf16
  auto out4 = [&](const float4_t& a, const float4_t& b) {
    float v[4];
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      v[e] = a[e] + b[e];
      if (RELU) v[e] = fmaxf(v[e], 0.0f);
    }
    return make_uint2(f2bf2(v[0], v[1]), f2bf2(v[2], v[3]));
  };
  uint4 st[IN_PER];
  auto load = [&](int tile) {
    const int bx = tile % nbx, by = tile / nbx;
    const int n = by / nrb, y0 = (by % nrb) * 8, x0 = bx * CT_W;
    // the patch's first pixel (outside the image for a tile at its edge) and
    // the pieces' offsets from it (conv3x3 takes this kernel if 31 bits hold
    // ten rows)
    const bf16* const src = in.p + ((ptrdiff_t)(n * H + y0 - 1) * W + (x0 - 1)) * in.cs + in.co;
    int q0 = tid;
    asm volatile("" : "+v"(q0));  // the pieces' places computed here, not held over the tiles
    if (y0 > 0 && y0 + 9 <= H && x0 > 0 && x0 + CT_W + 1 <= W) {  // workgroup-uniform: no pixel outside
#pragma unroll
      for (int k = 0; k < IN_PER; ++k) {
        // (the last round's spare threads read the patch's last piece again)
        const int q = k + 1 < IN_PER ? q0 + 256 * k : min(q0 + 256 * k, IN_Q - 1);
        const int piece = q % PQ, pix = q / PQ;
        st[k] = *reinterpret_cast<const uint4*>(src + (uint32_t)((pix / PW * W + pix % PW) * in.cs + 8 * piece));
      }
      return;
    }
#pragma unroll
    for (int k = 0; k < IN_PER; ++k) {
      const int q = q0 + 256 * k;
      const int piece = q % PQ, pix = q / PQ;
      const int yy = y0 + pix / PW - 1, gx = x0 + pix % PW - 1;
      uint4 v = make_uint4(0u, 0u, 0u, 0u);
      if (q < IN_Q && yy >= 0 && yy < H && gx >= 0 && gx < W)
        v = *reinterpret_cast<const uint4*>(src + (uint32_t)((pix / PW * W + pix % PW) * in.cs + 8 * piece));
      st[k] = v;
    }
  };
  int tile = blockIdx.x / nbz;
  if (tile < n_tiles) load(tile);
  for (; tile < n_tiles; tile += step) {  // workgroup-uniform
    int q0 = tid;
    asm volatile("" : "+v"(q0));  // as in load
    lds_barrier();                // the last tile's fragment reads are done
#pragma unroll
    for (int k = 0; k < IN_PER; ++k) {
      const int q = q0 + 256 * k;
      if (q < IN_Q) *reinterpret_cast<uint4*>(s_in + (q / PQ) * PS + 8 * (q % PQ)) = st[k];
    }
    lds_barrier();
    if (tile + step < n_tiles) load(tile + step);
    const int bx = tile % nbx, by = tile / nbx;
    const int n = by / nrb, y0 = (by % nrb) * 8 + 2 * wave, x0 = bx * CT_W;
    // a pixel's place in a view: that of the wave's first pixel, and an offset
    auto row = [&](const View& v) { return v.p + ((size_t)(n * H + y0) * W + x0) * v.cs + v.co; };
    uint2 xv[2] = {make_uint2(0u, 0u), make_uint2(0u, 0u)};  // the residual's input, under way during the MFMAs
    if (NT == 1 && fz.y) {
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
        if (y0 + rr < H && x0 + lane < W)
          xv[rr] = *reinterpret_cast<const uint2*>(row(fz.res) + (ptrdiff_t)rr * W * fz.res.cs + lane * fz.res.cs);
    }

    float4_t acc[2][4][NT];
#pragma unroll
    for (int rr = 0; rr < 2; ++rr)
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t) acc[rr][f][t] = float4_t{0.f, 0.f, 0.f, 0.f};
    const bf16* const base = s_in + (2 * wave * PW + i) * PS + 8 * (kq & 1);
    const bf16* const base_r = base + (hi ? PW * PS : 0);                  // the next tap row
    const bf16* const base_s = base + (hi ? PS - 2 * PW * PS : 0);         // the next tap column's first row
    const bf16* const base_h = base + (hi ? 16 - (2 * PW + 2) * PS : 0);   // the next channel half's first tap
    // group g = (pair q, output row rr): its four fragments are read while
    // the group before runs
    auto frags = [&](int g, bf16x8_t (&b)[4]) {
      const int q = g / 2, d = at(2 * q + 1) - at(2 * q);
      const bf16* const bp = (d == PW * PS ? base_r : d == PS - 2 * PW * PS ? base_s : base_h) + at(2 * q) + (g % 2) * PW * PS;
#pragma unroll
      for (int f = 0; f < 4; ++f) b[f] = *reinterpret_cast<const bf16x8_t*>(bp + 16 * f * PS);
    };
    bf16x8_t b[2][4];
    frags(0, b[0]);
#pragma unroll
    for (int g = 0; g < 2 * NQ; ++g) {
      if (g + 1 < 2 * NQ) frags(g + 1, b[(g + 1) & 1]);
#pragma unroll
      for (int f = 0; f < 4; ++f)
#pragma unroll
        for (int t = 0; t < NT; ++t)
          acc[g % 2][f][t] =
              __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[g / 2][t], b[g & 1][f], acc[g % 2][f][t], 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);  // no fragments read further ahead: they would spill
    }
    if constexpr (NP % 2) {
      const bf16* const bp = s_in + (2 * wave * PW + i) * PS + 4 * kq + at(NP - 1);
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const short4_t bl = *reinterpret_cast<const short4_t*>(bp + (rr * PW + 16 * f) * PS);
#pragma unroll
          for (int t = 0; t < NT; ++t)
            acc[rr][f][t] = __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(wl[t], bl, acc[rr][f][t], 0, 0, 0);
        }
      __builtin_amdgcn_sched_barrier(0);
    }

    float4_t bv[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) bv[t] = *reinterpret_cast<const float4_t*>(s_bias + 4 * NT * kq + 4 * t);
    if (NT == 1 && fz.y) {  // workgroup-uniform: the residual output replaces `out`
      // channels 0..3 are lanes 0..15's; lane l takes pixel l of the row
#pragma unroll
      for (int rr = 0; rr < 2; ++rr) {
        uint2 o = make_uint2(0u, 0u);
#pragma unroll
        for (int f = 0; f < 4; ++f) {
          const uint2 v = out4(acc[rr][f][0], bv[0]);
          const uint32_t vx = (uint32_t)__shfl((int)v.x, i), vy = (uint32_t)__shfl((int)v.y, i);
          if (kq == f) o = make_uint2(vx, vy);
        }
        if (y0 + rr < H && x0 + lane < W)
          *reinterpret_cast<float4*>(fz.y + ((size_t)(n * H + y0 + rr) * W + x0 + lane) * 4) =
              make_float4(bf_lo(xv[rr].x) + bf_lo(o.x), bf_hi(xv[rr].x) + bf_hi(o.x), bf_lo(xv[rr].y) + bf_lo(o.y),
                          bf_hi(xv[rr].y) + bf_hi(o.y));
      }
      continue;
    }
    typedef typename std::conditional<NT == 2, uint4, uint2>::type Out;
    // (uniform) row and fragment, this lane's pixel and channels in it
    const bf16* const mrow = row(fz.mask);
    bf16* const orow = row(out);
    const uint32_t mlane = (uint32_t)(i * fz.mask.cs + co0 + 4 * NT * kq), olane = (uint32_t)(i * out.cs + co0 + 4 * NT * kq);
    auto inside = [&](int f, int rr) { return y0 + rr < H && x0 + 16 * f + i < W; };
    const bool down = DOWN && co0 < fz.Cdown;  // workgroup-uniform
    // the mask of this fragment and, where registers allow, the next
    constexpr int MD = conv_few_waves<NT>() == 2 ? 2 : 1;
    Out m[MD][2];
    auto mask = [&](int f) {
#pragma unroll
      for (int rr = 0; rr < 2; ++rr)
        if (inside(f, rr))
          m[f % MD][rr] = *reinterpret_cast<const Out*>(mrow + (ptrdiff_t)(rr * W + 16 * f) * fz.mask.cs + mlane);
    };
    if (!DOWN && MD == 2 && fz.mask.p) mask(0);  // workgroup-uniform
#pragma unroll
    for (int f = 0; f < 4; ++f) {
      __builtin_amdgcn_sched_barrier(0);
      if (!DOWN && fz.mask.p && f + MD - 1 < 4) mask(f + MD - 1);
      Out o[2];
#pragma unroll
      for (int rr = 0; rr < 2; ++rr) {
        if constexpr (NT == 2) {
          const uint2 a = out4(acc[rr][f][0], bv[0]), c = out4(acc[rr][f][1], bv[1]);
          o[rr] = make_uint4(a.x, a.y, c.x, c.y);
        } else {
          o[rr] = out4(acc[rr][f][0], bv[0]);
        }
        if (down || !inside(f, rr)) continue;
        Out v = o[rr];
        if (!DOWN && fz.mask.p) v = relu_keep(v, m[f % MD][rr]);
        *reinterpret_cast<Out*>(orow + (ptrdiff_t)(rr * W + 16 * f) * out.cs + olane) = v;
      }
      // workgroup-uniform: the 2x2 averages or masked sums, added in
      // k_avgpool2_v8's order
      if (DOWN ? down : fz.pool.p != nullptr) {
        const View pool = down ? fz.down : fz.pool;
        const float scale = down ? 1.0f : 0.25f;
        const uint32_t* const r0 = reinterpret_cast<const uint32_t*>(&o[0]);
        const uint32_t* const r1 = reinterpret_cast<const uint32_t*>(&o[1]);
        Out pv;
        uint32_t* const r = reinterpret_cast<uint32_t*>(&pv);
#pragma unroll
        for (int h = 0; h < 2 * NT; ++h) {
          // the neighbouring pixel's values, from the neighbouring lane
          const uint32_t a1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)r0[h], 0xB1, 0xf, 0xf, true);
          const uint32_t b1 = (uint32_t)__builtin_amdgcn_mov_dpp((int)r1[h], 0xB1, 0xf, 0xf, true);
          const float lo = (((0.0f + bf_lo(r0[h])) + bf_lo(a1)) + bf_lo(r1[h])) + bf_lo(b1);
          const float hi2 = (((0.0f + bf_hi(r0[h])) + bf_hi(a1)) + bf_hi(r1[h])) + bf_hi(b1);
          r[h] = f2bf2(scale * lo, scale * hi2);
        }
        const int yo = y0 >> 1, xo = (x0 + 16 * f + i) >> 1;
        if ((i & 1) == 0 && yo < (H >> 1) && xo < (W >> 1)) {
          const size_t p = (size_t)(n * (H >> 1) + yo) * (W >> 1) + xo;
          const int c = co0 + 4 * NT * kq;
          if (down)
            pv = relu_keep(pv, *reinterpret_cast<const Out*>(fz.down_mask.p + p * fz.down_mask.cs + fz.down_mask.co + c));
          *reinterpret_cast<Out*>(pool.p + p * pool.cs + pool.co + c) = pv;
        }
      }
    }
  }
}

// Weight gradient on MFMA: an implicit GEMM per tap (r, s) with M = output
// channels, N = input channels, K = pixels:
//   dw[r][s][k][c] = sum_p dy[p][k] x[p + (r - 1, s - 1)][c].
// A workgroup owns a TCO x TCI channel tile, all nine taps, and a run of
// "units" (one 64-pixel strip of one dy row; units are strip-major, so a
// run walks down the rows of a strip).  LDS holds pixels as they lie in
// memory (all channels of a pixel together), a ring of three input rows of 66
// pixels and two dy rows, the next being filled while the others are read.  The
// matrix
// operands need eight consecutive pixels of one channel per lane; gfx950's
// transposing LDS read delivers them from that layout, so staging is one
// 16-byte store per eight channels and a column shift is a pixel offset.
// (Stored channel-major at three column shifts, staging took 24 two-byte
// stores per eight channels and most of the kernel's time.)  An input row's
// fragments stay in registers for the three dy rows they serve: one row down
// reads three shifts of one input row.  v_mfma_f32_16x16x32_bf16: lane l
// holds A[l % 16][8 (l / 16) + e], B[8 (l / 16) + e][l % 16], D[4 (l / 16) +
// e][l % 16].  Waves own SPW 16-channel output blocks x one 16-channel input
// block; when the tile has fewer such groups than waves, WK = 2 waves split
// each strip's two 32-pixel K steps and add in LDS at the end.  The bias
// gradient is the product with an all-ones B.  Each run's sums go to its own
// slice of `part` (no atomics); k_wgrad_reduce adds the slices to dw and db
// in a fixed order.  Rows are loaded two ahead: a row's products take a third
// of a load's time, and one row ahead the waves waited two thirds of theirs.
// Per 8 x 256^2 training step the twelve layers take 0.31 ms (0.37 ms one row
// ahead, 0.62 ms channel-major), those of 64 outputs at 580 TFLOP/s.
constexpr int WG_SEG = 64;  // strip width

template <int TCO, int TCI, int SPW>
struct WgradCfg {
  static constexpr int NCI = TCI / 16, GROUPS = NCI * (TCO / (16 * SPW));  // wave groups of the tile
  static constexpr int WK = GROUPS >= 4 ? 1 : 2;                          // waves per group (K split)
  static constexpr int KS = 2 / WK;                                       // K steps of a strip per wave
  static_assert(GROUPS * WK <= 4 && (GROUPS == 4 || WK == 2), "four waves cover the tile");
  static constexpr int PQO = TCO / 8, PQI = TCI / 8;                      // 16-byte pieces per pixel
  static constexpr int DY_Q = WG_SEG * PQO, XROW_Q = (WG_SEG + 2) * PQI;
  static constexpr int DY_PER = (DY_Q + 255) / 256, X_PER = (XROW_Q + 255) / 256;  // pieces per thread
  // LDS pixel strides: 16 bytes of padding spread the transposing reads' rows
  // over the banks and keep the stores aligned
  static constexpr int OS = TCO + 8, IS = TCI + 8;
  static constexpr int X_ROW = (WG_SEG + 2) * IS, DY_ROW = WG_SEG * OS;
  static constexpr int LDS = 3 * X_ROW + 2 * DY_ROW;  // bf16 elements
  static constexpr int RED_Q = 5;                     // taps per round of the K-split reduction
  static_assert(WK == 1 || GROUPS * RED_Q * SPW * 4 * 64 * 4 <= LDS * 2, "the reduction fits the staging buffers");
};

// A lane's eight consecutive pixels of one channel from pixel-major LDS: p
// points at the lane's piece (pixel 8 (l / 16) + (l % 16) / 4 of the K step,
// channels 4 (l % 4) .. + 3 of the block).
typedef __attribute__((address_space(3))) short4_t* lds_short4_p;
template <int STRIDE>
__device__ __forceinline__ bf16x8_t wgrad_frag(const bf16* p) {
  const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_p)p);
  const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_p)(p + 4 * STRIDE));
  return __builtin_bit_cast(bf16x8_t, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Waves per SIMD that the registers must allow: with three, <32, 32> spills (934
// against 874 us for the 32-output layers of eight 8 x 256^2 training steps).
constexpr int wgrad_waves(int TCO, int TCI) { return TCI == 16 ? 4 : TCO >= 32 ? 2 : 3; }

template <int TCO, int TCI, int SPW, bool FAR>
__global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(wgrad_waves(TCO, TCI)))) void k_wgrad_mfma(
    View x, View up, int Cup, View dy, float* __restrict__ part, int N, int H, int W, int Cin, int Cout, int runs,
    int with_bias) {
  using C = WgradCfg<TCO, TCI, SPW>;
  __shared__ __attribute__((aligned(16))) bf16 s_buf[C::LDS];
  bf16* const s_x = s_buf;                  // [row of three][pixel][ci]
  bf16* const s_dy = s_buf + 3 * C::X_ROW;  // [row & 1][pixel][co]
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int i = lane & 15, kq = lane >> 4;
  const int run = blockIdx.x, cb = blockIdx.y, kb = blockIdx.z;
  const int ci0 = cb * TCI, co0 = kb * TCO;
  const int rows = N * H, strips = (W + WG_SEG - 1) / WG_SEG, units = rows * strips;
  const int u0 = (int)((long long)units * run / runs), u1 = (int)((long long)units * (run + 1) / runs);
  // this wave's group: output blocks sco0 .. sco0 + SPW - 1, input block sci, K steps kw, kw + WK, ...
  const int kw = wave % C::WK, grp = wave / C::WK;
  const bool active = grp < C::GROUPS;
  const int sci = grp % C::NCI, sco0 = (grp / C::NCI) * SPW;
  const bool bias = with_bias && cb == 0 && sci == 0 && active;
  // this lane's piece within a K step (see wgrad_frag)
  const int fpx = 32 * kw + 8 * kq + (i >> 2), fch = 4 * (i & 3);
  const bf16* const fdy = s_dy + fpx * C::OS + 16 * (active ? sco0 : 0) + fch;
  const bf16* const fx = s_x + fpx * C::IS + 16 * sci + fch;
  float4_t acc[9][SPW], accb[SPW];
#pragma unroll
  for (int q = 0; q < 9; ++q)
#pragma unroll
    for (int t = 0; t < SPW; ++t) acc[q][t] = float4_t{0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int t = 0; t < SPW; ++t) accb[t] = float4_t{0.f, 0.f, 0.f, 0.f};
  const uint4 one4 = make_uint4(0x3f803f80u, 0x3f803f80u, 0x3f803f80u, 0x3f803f80u);
  const bf16x8_t ones = __builtin_bit_cast(bf16x8_t, one4);
  // The input's view: half-resolution for a block of upsampled channels (TCI
  // divides Cup).  Written out by a pass of their own they cost 33 us an 8 x
  // 256^2 training step, and as much again in reading four copies.
  const int us = ci0 < Cup ? 1 : 0;  // workgroup-uniform
  const bf16* const xp = us ? up.p + up.co + ci0 : x.p + x.co + ci0 - Cup;
  const int xcs = us ? up.cs : x.cs, Wx = W >> us, Hx = H >> us;
  // Rows on their way to LDS, by the row's place in the ring of three: one
  // being stored while the next is under way (a row's products take a third of
  // a load's time, so one row ahead left the waves waiting).
  uint4 vd[3][C::DY_PER], vx[3][C::X_PER];
  uint32_t pd[C::DY_PER], px[C::X_PER];  // this thread's pieces of a strip's rows (piece_load)
  auto places = [&](int xs) {
#pragma unroll
    for (int k = 0; k < C::DY_PER; ++k) {
      const int q = tid + 256 * k, p = q / C::PQO, pc = q % C::PQO;
      pd[k] = q < C::DY_Q && xs + p < W ? piece_place<FAR>(p, dy.cs, pc) : BUF_NONE;
    }
#pragma unroll
    for (int k = 0; k < C::X_PER; ++k) {
      const int q = tid + 256 * k, p = q / C::PQI, pc = q % C::PQI, gx = xs + p - 1;
      px[k] = q < C::XROW_Q && gx >= 0 && gx < W ? piece_place<FAR>((gx >> us) - ((xs - 1) >> us), xcs, pc) : BUF_NONE;
    }
  };
  auto load_dy = [&](uint4 (&v)[C::DY_PER], int n, int y, int xs) {
    const bf16* const src = dy.p + ((size_t)(n * H + y) * W + xs) * dy.cs + dy.co + co0;
#pragma unroll
    for (int k = 0; k < C::DY_PER; ++k) v[k] = piece_load<FAR>(src, dy.cs, pd[k]);
  };
  auto store_dy = [&](const uint4 (&v)[C::DY_PER], int y) {
#pragma unroll
    for (int k = 0; k < C::DY_PER; ++k) {
      const int q = tid + 256 * k, p = q / C::PQO, pc = q % C::PQO;
      if (q < C::DY_Q) *reinterpret_cast<uint4*>(s_dy + (y & 1) * C::DY_ROW + p * C::OS + 8 * pc) = v[k];
    }
  };
  auto load_x = [&](uint4 (&v)[C::X_PER], int n, int yy, int xs) {
    const bf16* const src = xp + ((ptrdiff_t)(n * Hx + (yy >> us)) * Wx + ((xs - 1) >> us)) * xcs;
#pragma unroll
    for (int k = 0; k < C::X_PER; ++k) v[k] = piece_load<FAR>(src, xcs, px[k]);
  };
  auto store_x = [&](const uint4 (&v)[C::X_PER], int slot) {
#pragma unroll
    for (int k = 0; k < C::X_PER; ++k) {
      const int q = tid + 256 * k, p = q / C::PQI, pc = q % C::PQI;
      if (q < C::XROW_Q) *reinterpret_cast<uint4*>(s_x + slot * C::X_ROW + p * C::IS + 8 * pc) = v[k];
    }
  };
  // fragments of the input rows around the current dy row: [row][shift][K step]
  bf16x8_t xf[3][3][C::KS];
  auto read_x = [&](bf16x8_t (&f)[3][C::KS], int slot) {
    const bf16* const fr = fx + slot * C::X_ROW;
#pragma unroll
    for (int sh = 0; sh < 3; ++sh)
#pragma unroll
      for (int ks = 0; ks < C::KS; ++ks) f[sh][ks] = wgrad_frag<C::IS>(fr + (sh + 32 * ks) * C::IS);
  };
  // One dy row, R = its number in the strip modulo 3.  xf[R] holds input row
  // y - 1, xf[R + 1] row y, and row y + 1 is read from ring place R + 2 into
  // xf[R + 2] (indices modulo 3).  Ends with dy row y + 1 and input row y + 2
  // (ring place R) in LDS and the rows behind them under way, as far as the
  // run's `left` rows of the strip go on.
  auto unit = [&](auto rot, int n, int y, int xs, int left) {
    constexpr int R = decltype(rot)::value;
    if (left > 2) {
      load_dy(vd[(R + 2) % 3], n, y + 2, xs);
      if (y + 3 < H) load_x(vx[(R + 1) % 3], n, y + 3, xs);
    }
    if (active) {
      if (y + 1 < H) read_x(xf[(R + 2) % 3], (R + 2) % 3);
#pragma unroll
      for (int ks = 0; ks < C::KS; ++ks) {
        bf16x8_t a[SPW];
#pragma unroll
        for (int t = 0; t < SPW; ++t)
          a[t] = wgrad_frag<C::OS>(fdy + (y & 1) * C::DY_ROW + 32 * ks * C::OS + 16 * t);
#pragma unroll
        for (int r = 0; r < 3; ++r) {
          if (y + r < 1 || y + r > H) continue;  // zero padding: no products
#pragma unroll
          for (int sh = 0; sh < 3; ++sh)
#pragma unroll
            for (int t = 0; t < SPW; ++t)
              acc[r * 3 + sh][t] =
                  __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], xf[(R + r) % 3][sh][ks], acc[r * 3 + sh][t], 0, 0, 0);
        }
        if (bias) {
#pragma unroll
          for (int t = 0; t < SPW; ++t)
            accb[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[t], ones, accb[t], 0, 0, 0);
        }
      }
    }
    if (left > 1) {
      store_dy(vd[(R + 1) % 3], y + 1);
      if (y + 2 < H) store_x(vx[R], R);
      lds_barrier();
    }
  };
  for (int u = u0; u < u1;) {
    // a new strip or image
    const int row = u % rows, n = row / H, y0 = row % H, xs = (u / rows) * WG_SEG;
    const int y1 = min(H, y0 + (u1 - u));  // this run's dy rows of it: y0 .. y1 - 1
    places(xs);
    // the first rows, all loads at once
    load_dy(vd[0], n, y0, xs);
    if (y0 > 0) load_x(vx[0], n, y0 - 1, xs);
    load_x(vx[1], n, y0, xs);
    if (y0 + 1 < H) load_x(vx[2], n, y0 + 1, xs);
    if (y0 + 1 < y1) load_dy(vd[1], n, y0 + 1, xs);
    lds_barrier();  // the previous rows are read
    store_dy(vd[0], y0);
    if (y0 > 0) store_x(vx[0], 0);
    if (y0 + 1 < y1 && y0 + 2 < H) load_x(vx[0], n, y0 + 2, xs);
    store_x(vx[1], 1);
    if (y0 + 1 < H) store_x(vx[2], 2);
    lds_barrier();
    if (active) {
      if (y0 > 0) read_x(xf[0], 0);
      read_x(xf[1], 1);
    }
    // row y0 + 2 is stored over row y0 - 1 at the end of the first unit
    if (y0 > 0 && y0 + 1 < y1) lds_barrier();
    for (int y = y0; y < y1;) {
      unit(std::integral_constant<int, 0>(), n, y, xs, y1 - y);
      if (++y >= y1) break;
      unit(std::integral_constant<int, 1>(), n, y, xs, y1 - y);
      if (++y >= y1) break;
      unit(std::integral_constant<int, 2>(), n, y, xs, y1 - y);
      ++y;
    }
    u += y1 - y0;
  }
  // K-split groups: the second wave of each group adds its sums to the first's
  if constexpr (C::WK == 2) {
    float* const s_red = reinterpret_cast<float*>(s_buf);
#pragma unroll
    for (int q0 = 0; q0 < 10; q0 += C::RED_Q) {  // taps 0..8, then the bias
      __syncthreads();
      if (active && kw == 1) {
#pragma unroll
        for (int q = q0; q < q0 + C::RED_Q; ++q)
#pragma unroll
          for (int t = 0; t < SPW; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              s_red[(((grp * C::RED_Q + q - q0) * SPW + t) * 4 + e) * 64 + lane] =
                  q < 9 ? acc[q < 9 ? q : 0][t][e] : accb[t][e];
      }
      __syncthreads();
      if (active && kw == 0) {
#pragma unroll
        for (int q = q0; q < q0 + C::RED_Q; ++q)
#pragma unroll
          for (int t = 0; t < SPW; ++t)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const float o = s_red[(((grp * C::RED_Q + q - q0) * SPW + t) * 4 + e) * 64 + lane];
              if (q < 9) acc[q < 9 ? q : 0][t][e] += o;
              else accb[t][e] += o;
            }
      }
    }
  }
  if (!active || kw != 0) return;
  // part[run][q][co][ci]; the bias sums of every run follow all runs' weights
  const size_t per = (size_t)9 * Cout * Cin;
  float* const pr = part + (size_t)run * per;
#pragma unroll
  for (int q = 0; q < 9; ++q)
#pragma unroll
    for (int t = 0; t < SPW; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int co = co0 + 16 * (sco0 + t) + 4 * kq + e, ci = ci0 + 16 * sci + i;
        pr[((size_t)q * Cout + co) * Cin + ci] = acc[q][t][e];
      }
  if (bias && i == 0) {
    // every column of the all-ones product holds the row sums
#pragma unroll
    for (int t = 0; t < SPW; ++t)
#pragma unroll
      for (int e = 0; e < 4; ++e)
        part[(size_t)runs * per + (size_t)run * Cout + co0 + 16 * (sco0 + t) + 4 * kq + e] = accb[t][e];
  }
}

// dw[i] += sum over runs of part (bias entries after the weights): 64
// outputs per workgroup, 16 lanes per output summing every 16th run, the 16
// sums added in a fixed order (deterministic).  Four loads in flight per lane
// (17.6 -> 11.0 us a layer); eight, or 16 outputs per workgroup for the small
// layers, took 13 us.
__global__ __launch_bounds__(1024) void k_wgrad_reduce(const float* __restrict__ part, float* __restrict__ dw,
                                                       float* __restrict__ db, int runs, int n_w, int n_b) {
  __shared__ float s_sum[16][65];
  const int o = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int idx = blockIdx.x * 64 + o;
  float acc = 0.0f;
  if (idx < n_w + n_b) {
    const float* const src = idx < n_w ? part + idx : part + (size_t)runs * n_w + (idx - n_w);
    const size_t step = idx < n_w ? (size_t)n_w : (size_t)n_b;
    int k = g;
    for (; k + 48 < runs; k += 64) {
      const float v0 = src[(size_t)k * step], v1 = src[(size_t)(k + 16) * step], v2 = src[(size_t)(k + 32) * step],
                  v3 = src[(size_t)(k + 48) * step];
      acc += v0;
      acc += v1;
      acc += v2;
      acc += v3;
    }
    for (; k < runs; k += 16) acc += src[(size_t)k * step];
  }
  s_sum[g][o] = acc;
  __syncthreads();
  if (g == 0) {
    float t = 0.0f;
#pragma unroll
    for (int k = 0; k < 16; ++k) t += s_sum[k][o];
    if (idx < n_w) dw[idx] += t;
    else if (idx < n_w + n_b) db[idx - n_w] += t;
  }
}

__device__ __forceinline__ bf16 flipped(const bf16* __restrict__ w, int i, int Cin, int Cout) {
  // index i: [r][s][c][k] with k fastest
  const int k = i % Cout, c = (i / Cout) % Cin, rs = i / (Cout * Cin);
  return w[((size_t)(8 - rs) * Cout + k) * Cin + c];
}

__global__ void k_flip(const bf16* __restrict__ w, bf16* __restrict__ wt, int Cin, int Cout) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < 9 * Cin * Cout) wt[i] = flipped(w, i, Cin, Cout);
}

// Every layer's weights in one launch (one launch per layer took 58 us of
// the 2.17 ms of an 8 x 256^2 training step): blockIdx.y is the layer.
__global__ void k_flip_all(FlipLayers L, const bf16* __restrict__ w, bf16* __restrict__ wt) {
  const FlipLayers::Layer y = L.layer[blockIdx.y];
  const int n = 9 * y.cin * y.cout;
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x)
    wt[y.wt_off + i] = flipped(w + y.w_off, i, y.cin, y.cout);
}

__global__ void k_avgpool2(View in, View out, int N, int H, int W, int C) {
  const int Ho = H / 2, Wo = W / 2;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)N * Ho * Wo * C) return;
  const int c = (int)(i % C);
  const size_t po = i / C;
  const int xo = (int)(po % Wo), yo = (int)((po / Wo) % Ho), n = (int)(po / ((size_t)Wo * Ho));
  float s = 0.0f;
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) s += bf2f(in.p[((size_t)(n * H + 2 * yo + a) * W + 2 * xo + b) * in.cs + in.co + c]);
  out.p[po * out.cs + out.co + c] = f2bf(0.25f * s);
}

// 8-channel (16-byte) version of pooling: one thread per output pixel and
// channel group.

__global__ void k_avgpool2_v8(View in, View out, int N, int H, int W, int C) {
  const int Ho = H / 2, Wo = W / 2, G = C / 8;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)N * Ho * Wo * G) return;
  const int g = (int)(i % G);
  const size_t po = i / G;
  const int xo = (int)(po % Wo), yo = (int)((po / Wo) % Ho), n = (int)(po / ((size_t)Wo * Ho));
  float s[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
  for (int a = 0; a < 2; ++a)
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const uint4 v = *reinterpret_cast<const uint4*>(
          in.p + ((size_t)(n * H + 2 * yo + a) * W + 2 * xo + b) * in.cs + in.co + 8 * g);
      const uint32_t q[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
      for (int k = 0; k < 4; ++k) { s[2 * k] += bf_lo(q[k]); s[2 * k + 1] += bf_hi(q[k]); }
    }
  uint32_t r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    r[k] = f2bf2(0.25f * s[2 * k], 0.25f * s[2 * k + 1]);
  *reinterpret_cast<uint4*>(out.p + po * out.cs + out.co + 8 * g) = make_uint4(r[0], r[1], r[2], r[3]);
}

// Gradient of the 2x2 average added to din (8 channels per thread), then
// ReLU's mask of y.
__global__ void k_avgpool2_bwd_v8(View dout, View din, View y, int N, int H, int W, int C) {
  const int G = C / 8;
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= (size_t)N * H * W * G) return;
  const int g = (int)(i % G);
  const size_t p = i / G;
  const int x = (int)(p % W), yy = (int)((p / W) % H), n = (int)(p / ((size_t)W * H));
  const uint4 v = *reinterpret_cast<const uint4*>(
      dout.p + ((size_t)(n * (H / 2) + yy / 2) * (W / 2) + x / 2) * dout.cs + dout.co + 8 * g);
  uint4* const d = reinterpret_cast<uint4*>(din.p + p * din.cs + din.co + 8 * g);
  const uint4 o = *d;
  const uint32_t q[4] = {v.x, v.y, v.z, v.w}, a[4] = {o.x, o.y, o.z, o.w};
  uint32_t r[4];
#pragma unroll
  for (int k = 0; k < 4; ++k)
    r[k] = (uint32_t)f2bf(bf_lo(a[k]) + 0.25f * bf_lo(q[k])) |
           ((uint32_t)f2bf(bf_hi(a[k]) + 0.25f * bf_hi(q[k])) << 16);
  *d = relu_keep(make_uint4(r[0], r[1], r[2], r[3]), *reinterpret_cast<const uint4*>(y.p + p * y.cs + y.co + 8 * g));
}

inline bool v8_ok(const View& a, const View& b, int C) {
  return C % 8 == 0 && a.cs % 8 == 0 && a.co % 8 == 0 && b.cs % 8 == 0 && b.co % 8 == 0 &&
         ((uintptr_t)a.p & 15u) == 0 && ((uintptr_t)b.p & 15u) == 0;
}

// One pixel per thread and round.  The loss goes out as one atomic per
// workgroup: one per wave (8192 to one address at 8 x 256^2) held the kernel
// for 125 us.  VEC: 16-byte aligned buffers, 8- and 16-byte accesses.
constexpr int RES_GRID = 1024;

template <bool VEC>
__global__ __launch_bounds__(256) void k_residual_loss(View x, View o, const bf16* __restrict__ t,
                                                       float* __restrict__ y_out, float* __restrict__ loss_sum,
                                                       bf16* __restrict__ dO, int npix, float inv_count) {
  __shared__ float s_l[4];
  auto load4 = [](const bf16* p, float (&v)[4]) {
    if constexpr (VEC) {
      const uint2 q = *reinterpret_cast<const uint2*>(p);
      v[0] = bf_lo(q.x); v[1] = bf_hi(q.x); v[2] = bf_lo(q.y); v[3] = bf_hi(q.y);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c) v[c] = bf2f(p[c]);
    }
  };
  float l = 0.0f;
  for (int p = blockIdx.x * 256 + threadIdx.x; p < npix; p += gridDim.x * 256) {
    float y[4], ov[4];
    load4(x.p + (size_t)p * x.cs + x.co, y);
    load4(o.p + (size_t)p * o.cs + o.co, ov);
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      y[c] = y[c] + ov[c];
      if (y_out) y_out[(size_t)p * 4 + c] = y[c];
    }
    if (t) {
      float tv[4];
      bf16 g[4];
      load4(t + (size_t)p * 16, tv);
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        const float d = y[c] - tv[c];
        l += d * d;
        g[c] = f2bf(2.0f * d * inv_count);
      }
      if constexpr (VEC) {
        uint4* q = reinterpret_cast<uint4*>(dO + (size_t)p * 16);
        q[0] = make_uint4((uint32_t)g[0] | ((uint32_t)g[1] << 16), (uint32_t)g[2] | ((uint32_t)g[3] << 16), 0u, 0u);
        q[1] = make_uint4(0u, 0u, 0u, 0u);
      } else {
#pragma unroll
        for (int c = 0; c < 16; ++c) dO[(size_t)p * 16 + c] = c < 4 ? g[c] : (bf16)0;
      }
    }
  }
  if (t) {
#pragma unroll
    for (int off = 32; off >= 1; off >>= 1) l += __shfl_xor(l, off);
    if ((threadIdx.x & 63) == 0) s_l[threadIdx.x >> 6] = l;
    __syncthreads();
    if (threadIdx.x == 0) atomicAdd(loss_sum, (s_l[0] + s_l[1]) + (s_l[2] + s_l[3]));
  }
}

__global__ void k_adam(float* __restrict__ p, const float* __restrict__ g, float* __restrict__ m,
                       float* __restrict__ v, bf16* __restrict__ pb, int n, float lr, float b1, float b2, float eps,
                       float c1, float c2) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  const float gi = g[i];
  const float mi = b1 * m[i] + (1.0f - b1) * gi;
  const float vi = b2 * v[i] + (1.0f - b2) * gi * gi;
  m[i] = mi;
  v[i] = vi;
  // bias-corrected step: c1 = 1 - b1^t, c2 = 1 - b2^t
  const float pi = p[i] - lr * (mi / c1) / (sqrtf(vi / c2) + eps);
  p[i] = pi;
  if (pb) pb[i] = f2bf(pi);
}

__global__ void k_to_bf16(const float* __restrict__ in, bf16* __restrict__ out, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) out[i] = f2bf(in[i]);
}

// Network input: channels 0-3 the normalised log-density log10(1 + v scale)
// of the bin's RGBA, channel 4 the noise level log10(1 + scale) (what one
// sample in a bin reads: scale = W H / n is the inverse samples per pixel),
// channels 5-15 zero.
__global__ void k_log_density(const float* __restrict__ hist, bf16* __restrict__ out, int npix, float scale) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix * 16) return;
  const int p = i >> 4, c = i & 15;
  out[i] = c < 4 ? f2bf(log10f(1.0f + hist[(size_t)p * 4 + c] * scale))
                 : (c == 4 ? f2bf(log10f(1.0f + scale)) : (bf16)0);
}

// The same values, one pixel per thread: one 16-byte load of the bin and two
// 16-byte stores of its 16 channels (16-byte aligned buffers).
__global__ void k_log_density_v(const float4* __restrict__ hist, uint4* __restrict__ out, int npix, float scale) {
  const int p = blockIdx.x * blockDim.x + threadIdx.x;
  if (p >= npix) return;
  const float4 h = hist[p];
  const uint32_t lo = f2bf2(log10f(1.0f + h.x * scale), log10f(1.0f + h.y * scale));
  const uint32_t hi = f2bf2(log10f(1.0f + h.z * scale), log10f(1.0f + h.w * scale));
  const uint32_t nl = (uint32_t)f2bf(log10f(1.0f + scale));
  out[2 * (size_t)p] = make_uint4(lo, hi, nl, 0u);
  out[2 * (size_t)p + 1] = make_uint4(0u, 0u, 0u, 0u);
}

__global__ void k_bf16_to_f32_4(const bf16* __restrict__ in, int cs, float* __restrict__ out, int npix) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= npix * 4) return;
  out[i] = bf2f(in[(size_t)(i >> 2) * cs + (i & 3)]);
}

__global__ void k_zero(float* __restrict__ p, size_t n) {
  const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0.0f;
}

inline dim3 grid1(size_t n) { return dim3((unsigned)((n + 255) / 256)); }

}  // namespace

hipError_t conv3x3(View in, const bf16* w, const float* bias, View out, int N, int H, int W, int Cin, int Cout,
                   int relu, hipStream_t s, const ConvFuse& fuse) {
  const View& up = fuse.up;
  const int Cup = fuse.Cup;
  const View& pool = fuse.pool;
  if (Cin % 16 || Cout % 16 || in.cs % 4 || in.co % 4 || out.cs < out.co + Cout || in.cs < in.co + Cin - Cup)
    return hipErrorInvalidValue;
  const int nt = (Cout % 64 == 0) ? 4 : (Cout % 32 == 0) ? 2 : 1;
  const bool lds = Cin % 8 == 0 && in.cs % 8 == 0 && in.co % 8 == 0 && ((uintptr_t)in.p & 15u) == 0 &&
                   ((uintptr_t)w & 15u) == 0;
  if (Cup) {  // the fused upsampling exists on the LDS path only
    if (!lds || Cup < 0 || Cup % 32 || Cup >= Cin || H % 2 || W % 2 || up.cs % 8 || up.co % 8 ||
        up.cs < up.co + Cup || ((uintptr_t)up.p & 15u) != 0)
      return hipErrorInvalidValue;
  }
  if (lds) {
    // K = 32 steps (v_mfma_f32_16x16x32_bf16: twice the products per
    // instruction) pay off where each staged step feeds 64 output channels or
    // the input has 64 channels or more: the 96 -> 32 decoder layer at full
    // resolution takes 320 us at 2048^2 with them, 389 us without.  The
    // narrow layers with 16, 32 or 48 input channels keep the smaller K = 16
    // tiles, whose LDS and registers fit three workgroups per CU instead of
    // two.  The narrow layers give each wave two rows (RW = 2), whose shared
    // input rows halve the B and cut the A fragment reads per output by a
    // third.
    const bool k32 = Cin % 32 == 0 && (nt == 4 || Cin >= 64);
    const int rw = nt <= 2 ? 2 : 1;
    const int nbx = (W + CT_W - 1) / CT_W, nbz = Cout / (16 * nt);
    const long long tiles = (long long)nbx * N * ((H + 4 * rw - 1) / (4 * rw)) * nbz;
    if (tiles >= (1ll << 24)) return hipErrorInvalidValue;  // a 1-D grid of 256-thread workgroups
    const int n_tiles = (int)tiles;
    const int vec_out = out.cs % 8 == 0 && out.co % 8 == 0 && ((uintptr_t)out.p & 15u) == 0;
    // the fused pooling needs the LDS epilogue; otherwise pool afterwards
    const bool fuse_pool = pool.p && vec_out && H % 2 == 0 && W % 2 == 0 && pool.cs % 8 == 0 &&
                           pool.co % 8 == 0 && ((uintptr_t)pool.p & 15u) == 0;
    // the residual output needs the LDS epilogue of a single 16-channel block;
    // otherwise the output is written and the residual computed afterwards
    const bool fuse_res = fuse.y && vec_out && Cout == 16 && fuse.res.cs % 4 == 0 && fuse.res.co % 4 == 0 &&
                          ((uintptr_t)fuse.res.p & 7u) == 0 && ((uintptr_t)fuse.y & 15u) == 0 && !pool.p;
    // so does the mask of a gradient
    if (fuse.mask.p && (!vec_out || fuse.y || fuse.mask.cs % 8 || fuse.mask.co % 8 ||
                        ((uintptr_t)fuse.mask.p & 15u) != 0))
      return hipErrorInvalidValue;
    if (fuse.Cdown && (!vec_out || fuse.y || pool.p || fuse.Cdown % (16 * nt) || fuse.Cdown >= Cout || H % 2 || W % 2 ||
                       fuse.down.cs % 8 || fuse.down.co % 8 || ((uintptr_t)fuse.down.p & 15u) != 0 ||
                       fuse.down_mask.cs % 8 || fuse.down_mask.co % 8 || ((uintptr_t)fuse.down_mask.p & 15u) != 0))
      return hipErrorInvalidValue;
    ConvFuse fz = fuse;
    if (!fuse_pool) fz.pool = View{nullptr, 0, 0};
    if (!fuse_res) { fz.res = View{nullptr, 0, 0}; fz.y = nullptr; }
    // Weights that fit the registers (Cin 16 or 32) and no part that needs
    // another path: the persistent kernel, faster at every size (32 -> 32,
    // with the call's 17 us: 2048^2 223 -> 162 us, 8 x 256^2 43 -> 33, 517 x
    // 333 28 -> 23; 16 -> 32 at 64^2 20.6 -> 17.3).
    // (Its 32-bit offsets reach ten rows of the input, and of the other views a
    // tile's 64 pixels.)
    const bool few = (long long)10 * W * in.cs < (1ll << 31) &&
                     std::max({out.cs, fuse.mask.cs, fuse.res.cs}) < (1 << 24) && !k32 && nt <= 2 && Cin <= 32 && !Cup && vec_out && (!pool.p || fuse_pool) && (!fuse.y || fuse_res) &&
                     (!fuse.Cdown || (Cin == 32 && nt == 2 && !relu && !fuse.mask.p));
    if (few) {
      int dev = 0, cus = 0;
      hipError_t e = hipGetDevice(&dev);
      if (e == hipSuccess) e = hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev);
      if (e != hipSuccess) return e;
#define RF_CONV_FEW(CIN_, NT_, RELU_, DOWN_)                                                                      \
  hipLaunchKernelGGL((k_conv3x3_few<CIN_, NT_, RELU_, DOWN_>),                                                    \
                     dim3((unsigned)(std::min(n_tiles / nbz, std::max(1, conv_few_waves<NT_>() * cus / nbz)) * nbz)), \
                     dim3(256), 0, s, in, w, bias, out, H, W, Cout, fz, nbx, nbz, n_tiles / nbz)
      if (fuse.Cdown) {
        RF_CONV_FEW(32, 2, false, true);
      } else if (relu) {
        if (Cin == 32) { if (nt == 2) RF_CONV_FEW(32, 2, true, false); else RF_CONV_FEW(32, 1, true, false); }
        else { if (nt == 2) RF_CONV_FEW(16, 2, true, false); else RF_CONV_FEW(16, 1, true, false); }
      } else {
        if (Cin == 32) { if (nt == 2) RF_CONV_FEW(32, 2, false, false); else RF_CONV_FEW(32, 1, false, false); }
        else { if (nt == 2) RF_CONV_FEW(16, 2, false, false); else RF_CONV_FEW(16, 1, false, false); }
      }
#undef RF_CONV_FEW
      return hipGetLastError();
    }
    // Buffer loads reach 2 GiB from a tile's first pixel (of at most ten rows
    // are read) and from the first weight; wider images and larger weights
    // take the same kernel with 64-bit addresses.
    const bool far = 20ll * W * std::max(in.cs, Cup ? up.cs : 0) >= (1ll << 31) - 65536 ||
                     18ll * Cin * Cout >= (1ll << 31) - 65536;
#define RF_CONV_LDS(NT_, KC_, RW_)                                                                                  \
  do {                                                                                                              \
    if (far)                                                                                                        \
      hipLaunchKernelGGL((k_conv3x3_lds<NT_, KC_, RW_, true>), dim3((unsigned)n_tiles), dim3(256), 0, s, in, w,     \
                         bias, out, H, W, Cin, Cout, relu, vec_out, fz, nbx, nbz, n_tiles);                         \
    else                                                                                                            \
      hipLaunchKernelGGL((k_conv3x3_lds<NT_, KC_, RW_, false>), dim3((unsigned)n_tiles), dim3(256), 0, s, in, w,    \
                         bias, out, H, W, Cin, Cout, relu, vec_out, fz, nbx, nbz, n_tiles);                         \
  } while (0)
    if (k32) {
      switch (nt) {
        case 4: RF_CONV_LDS(4, 32, 1); break;
        case 2: RF_CONV_LDS(2, 32, 2); break;
        default: RF_CONV_LDS(1, 32, 2); break;
      }
    } else {
      switch (nt) {
        case 4: RF_CONV_LDS(4, 16, 1); break;
        case 2: RF_CONV_LDS(2, 16, 2); break;
        default: RF_CONV_LDS(1, 16, 2); break;
      }
    }
#undef RF_CONV_LDS
    hipError_t e = hipGetLastError();
    if (e == hipSuccess && pool.p && !fuse_pool) e = avgpool2(out, pool, N, H, W, Cout, s);
    if (e == hipSuccess && fuse.y && !fuse_res)
      e = residual_loss(fuse.res, out, nullptr, fuse.y, nullptr, nullptr, N * H * W, 0.0f, s);
    return e;
  }
  if (fuse.mask.p || fuse.Cdown) return hipErrorInvalidValue;
  const dim3 grid((W + 63) / 64, N * H, Cout / (16 * nt));
  switch (nt) {
    case 4: hipLaunchKernelGGL(k_conv3x3<4>, grid, dim3(256), 0, s, in, w, bias, out, H, W, Cin, Cout, relu); break;
    case 2: hipLaunchKernelGGL(k_conv3x3<2>, grid, dim3(256), 0, s, in, w, bias, out, H, W, Cin, Cout, relu); break;
    default: hipLaunchKernelGGL(k_conv3x3<1>, grid, dim3(256), 0, s, in, w, bias, out, H, W, Cin, Cout, relu); break;
  }
  hipError_t e = hipGetLastError();
  if (e == hipSuccess && pool.p) e = avgpool2(out, pool, N, H, W, Cout, s);
  if (e == hipSuccess && fuse.y) e = residual_loss(fuse.res, out, nullptr, fuse.y, nullptr, nullptr, N * H * W, 0.0f, s);
  return e;
}

namespace {
// Channel tile of the weight gradient: TCO x TCI, SPW output blocks per wave.
struct WgradTile {
  int tco, tci;
};
WgradTile wgrad_tile(int Cin, int Cout) {
  const int tci = Cin % 32 == 0 ? 32 : 16;
  const int tco = (Cout % 64 == 0 && tci == 32) ? 64 : Cout % 32 == 0 ? 32 : 16;
  return WgradTile{tco, tci};
}
// Runs (row-strip ranges with their own partial sums): about 2048
// workgroups, at least 4 units per run, at most 2^23 partial sums.
int wgrad_runs(int N, int H, int W, int Cin, int Cout) {
  const WgradTile t = wgrad_tile(Cin, Cout);
  const int blocks = (Cout / t.tco) * (Cin / t.tci);
  const long long units = (long long)N * H * ((W + WG_SEG - 1) / WG_SEG);
  const size_t per = (size_t)9 * Cout * Cin + Cout;
  long long runs = std::min<long long>((2048 + blocks - 1) / blocks, std::max<long long>(1, units / 4));
  runs = std::min<long long>(runs, (long long)std::max<size_t>(1, ((size_t)1 << 23) / per));
  return (int)std::max<long long>(1, runs);
}

template <int TCO, int TCI, int SPW>
void launch_wgrad(dim3 grid, hipStream_t s, View x, View up, int Cup, View dy, float* work, int N, int H, int W,
                  int Cin, int Cout, int runs, int with_bias) {
  // buffer loads reach 2 GiB from a strip's first pixel, and take whole pieces
  // (views at multiples of 8 channels)
  auto whole = [](const View& v) { return ((uintptr_t)v.p & 15u) == 0 && v.cs % 8 == 0 && v.co % 8 == 0; };
  if (2ll * (WG_SEG + 2) * std::max({x.cs, Cup ? up.cs : 0, dy.cs}) < (1ll << 31) - 65536 && whole(x) && whole(dy) &&
      whole(up))
    hipLaunchKernelGGL((k_wgrad_mfma<TCO, TCI, SPW, false>), grid, dim3(256), 0, s, x, up, Cup, dy, work, N, H, W, Cin,
                       Cout, runs, with_bias);
  else
    hipLaunchKernelGGL((k_wgrad_mfma<TCO, TCI, SPW, true>), grid, dim3(256), 0, s, x, up, Cup, dy, work, N, H, W, Cin,
                       Cout, runs, with_bias);
}
}  // namespace

size_t conv3x3_wgrad_work(int N, int H, int W, int Cin, int Cout) {
  return (size_t)wgrad_runs(N, H, W, Cin, Cout) * ((size_t)9 * Cout * Cin + Cout);
}

hipError_t conv3x3_wgrad(View x, View up, int Cup, View dy, float* dw, float* db, int N, int H, int W, int Cin,
                         int Cout, float* work, size_t work_floats, hipStream_t s) {
  if (Cin % 16 || Cout % 16 || N <= 0 || H <= 0 || W <= 0 || !work) return hipErrorInvalidValue;
  if (Cup && (Cup < 0 || Cup % 32 || Cup >= Cin || H % 2 || W % 2)) return hipErrorInvalidValue;
  if (work_floats < conv3x3_wgrad_work(N, H, W, Cin, Cout)) return hipErrorInvalidValue;
  const WgradTile t = wgrad_tile(Cin, Cout);
  const int runs = wgrad_runs(N, H, W, Cin, Cout);
  const dim3 grid((unsigned)runs, (unsigned)(Cin / t.tci), (unsigned)(Cout / t.tco));
  const int wb = db ? 1 : 0;
  if (t.tco == 64) launch_wgrad<64, 32, 2>(grid, s, x, up, Cup, dy, work, N, H, W, Cin, Cout, runs, wb);
  else if (t.tco == 32 && t.tci == 32) launch_wgrad<32, 32, 1>(grid, s, x, up, Cup, dy, work, N, H, W, Cin, Cout, runs, wb);
  else if (t.tco == 32) launch_wgrad<32, 16, 1>(grid, s, x, up, Cup, dy, work, N, H, W, Cin, Cout, runs, wb);
  else if (t.tci == 32) launch_wgrad<16, 32, 1>(grid, s, x, up, Cup, dy, work, N, H, W, Cin, Cout, runs, wb);
  else launch_wgrad<16, 16, 1>(grid, s, x, up, Cup, dy, work, N, H, W, Cin, Cout, runs, wb);
  const int n_w = 9 * Cout * Cin, n_b = db ? Cout : 0;
  hipLaunchKernelGGL(k_wgrad_reduce, dim3((unsigned)((n_w + n_b + 63) / 64)), dim3(1024), 0, s, work, dw, db, runs,
                     n_w, n_b);
  return hipGetLastError();
}

hipError_t flip_weights(const bf16* w, bf16* wt, int Cin, int Cout, hipStream_t s) {
  hipLaunchKernelGGL(k_flip, grid1((size_t)9 * Cin * Cout), dim3(256), 0, s, w, wt, Cin, Cout);
  return hipGetLastError();
}

hipError_t flip_weights_all(const FlipLayers& L, int n_layers, const bf16* w, bf16* wt, hipStream_t s) {
  if (n_layers < 1 || n_layers > FlipLayers::kMax) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_flip_all, dim3(128, (unsigned)n_layers), dim3(256), 0, s, L, w, wt);
  return hipGetLastError();
}

hipError_t avgpool2(View in, View out, int N, int H, int W, int C, hipStream_t s) {
  if (v8_ok(in, out, C))
    hipLaunchKernelGGL(k_avgpool2_v8, grid1((size_t)N * (H / 2) * (W / 2) * (C / 8)), dim3(256), 0, s, in, out, N, H,
                       W, C);
  else
    hipLaunchKernelGGL(k_avgpool2, grid1((size_t)N * (H / 2) * (W / 2) * C), dim3(256), 0, s, in, out, N, H, W, C);
  return hipGetLastError();
}

hipError_t avgpool2_bwd(View dout, View din, View y, int N, int H, int W, int C, hipStream_t s) {
  if (!v8_ok(dout, din, C) || !v8_ok(y, y, C)) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_avgpool2_bwd_v8, grid1((size_t)N * H * W * (C / 8)), dim3(256), 0, s, dout, din, y, N, H, W, C);
  return hipGetLastError();
}

hipError_t residual_loss(View x, View o, const bf16* t, float* y_out, float* loss_sum, bf16* dO, int npix,
                         float inv_count, hipStream_t s) {
  const dim3 grid((unsigned)std::min((npix + 255) / 256, RES_GRID));
  const bool vec = (((uintptr_t)x.p | (uintptr_t)o.p | (uintptr_t)t | (uintptr_t)dO) & 15u) == 0 && x.cs % 4 == 0 &&
                   x.co % 4 == 0 && o.cs % 4 == 0 && o.co % 4 == 0;
  if (vec)
    hipLaunchKernelGGL(k_residual_loss<true>, grid, dim3(256), 0, s, x, o, t, y_out, loss_sum, dO, npix, inv_count);
  else
    hipLaunchKernelGGL(k_residual_loss<false>, grid, dim3(256), 0, s, x, o, t, y_out, loss_sum, dO, npix, inv_count);
  return hipGetLastError();
}

hipError_t adam(float* p, const float* g, float* m, float* v, bf16* pb, int n, float lr, float b1, float b2,
                float eps, float c1, float c2, hipStream_t s) {
  hipLaunchKernelGGL(k_adam, grid1((size_t)n), dim3(256), 0, s, p, g, m, v, pb, n, lr, b1, b2, eps, c1, c2);
  return hipGetLastError();
}

hipError_t to_bf16(const float* in, bf16* out, int n, hipStream_t s) {
  hipLaunchKernelGGL(k_to_bf16, grid1((size_t)n), dim3(256), 0, s, in, out, n);
  return hipGetLastError();
}

hipError_t log_density_bf16(const float* hist, bf16* out, int npix, float scale, hipStream_t s) {
  if (npix < 0 || (size_t)npix * 16 > (size_t)INT32_MAX) return hipErrorInvalidValue;
  if ((((uintptr_t)hist | (uintptr_t)out) & 15u) == 0)
    hipLaunchKernelGGL(k_log_density_v, grid1((size_t)npix), dim3(256), 0, s, reinterpret_cast<const float4*>(hist),
                       reinterpret_cast<uint4*>(out), npix, scale);
  else
    hipLaunchKernelGGL(k_log_density, grid1((size_t)npix * 16), dim3(256), 0, s, hist, out, npix, scale);
  return hipGetLastError();
}

hipError_t bf16_to_f32_4(const bf16* in, int cs, float* out, int npix, hipStream_t s) {
  hipLaunchKernelGGL(k_bf16_to_f32_4, grid1((size_t)npix * 4), dim3(256), 0, s, in, cs, out, npix);
  return hipGetLastError();
}

hipError_t zero_f32(float* p, size_t n, hipStream_t s) {
  if (n == 0) return hipSuccess;
  hipLaunchKernelGGL(k_zero, grid1(n), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

}  // namespace rfn
