// Mapped convolution over images of very few channels (first layers: grey, RGB, RGB-D), float32.
//
// The matrix-unit kernels (conv_fused.hip, conv_window_gemm.hip) contract 32 gather-side
// channels per chunk; with Cg <= 4 a chunk is at most an eighth full, and both the gathers and
// the MFMAs of the padding are wasted.  Here the reduction index (c, k) is packed instead:
//
//   small_forward_kernel   pix[b][n][m] = bias[n] + sum_{c,k} Wm[n][c][k] * col[b][(c,k)][m]
//   small_wgrad_kernel     gW[n][c][k] += sum_{b,m} pix[b][n][m] * col[b][(c,k)][m]
//   small_scatter_kernel   the transpose of the forward, with float atomics
//
// col[b][(c,k)][m] = sum over the points and taps of sample k of pixel m of
// coefficient * img[b][c][tap], as in common/mapped_im2col.h:13-63 of the reference.
//
// Forward and weight gradient build the column values the same way.  A workgroup owns a tile of
// pixels, 32 consecutive ones of a row per wave; lane l and lane l + 32 share a pixel and take
// half of its samples each, which is the operand layout of v_mfma_f32_32x32x2_f32 (reduction
// index = lane half).  The taps of a lane's samples are worked out once and serve every batch
// element; per batch element the window of the image they fall into is copied to LDS, all
// channels of an element side by side, so a tap is one LDS read and the blend one multiply-add
// per channel.  What bounded the kernels before was exactly that: the forward gathered every
// tap and channel from global memory (17 cycles of the CU's address path each), the weight
// gradient also worked the taps out once per channel.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>

#include "conv_small.hpp"
#include "sdk_host.hpp"
#include "sdk_mfma.hpp"
#include "sdk_taps.hpp"

namespace sdk {
namespace {

constexpr int kSmThreads = 256;
// Waves per SIMD a kernel's registers are cut for, by the accumulators it holds.
constexpr int small_waves(int NG, int blocks) { return NG > 1 || blocks > 2 ? 2 : 5 - blocks; }

// Kernel launch with dynamic LDS as an expression (for the dispatch macros).
template <typename... KArgs, typename... Args>
inline void launch_lds(void (*kernel)(KArgs...), dim3 grid, dim3 block, size_t smem,
                       hipStream_t stream, Args... args) {
  if (smem > 64 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),
                              hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);
  kernel<<<grid, block, smem, stream>>>(args...);
}

// Keeps a loaded value in a register here and now: without it the compiler moves the load
// behind the test of the tap it belongs to, one branch, one load and one wait per tap.
__device__ __forceinline__ void pin(float& x) { asm volatile("" : "+v"(x)); }

// Between the LDS writes of some lanes of a wave and the reads of others.  The hardware serves a
// wave's LDS accesses in order; this keeps the compiler from moving them past each other.
__device__ __forceinline__ void wave_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// ----------------------------------------------------------------------------- column values
// Pixel tiles: `waves` rows of 32 pixels where the grid has that many rows, else one row of
// 32 * waves pixels (vertex lists).
struct SmallTiling {
  int waves;    // of a workgroup
  int stacked;  // 1: a tile's waves lie in consecutive rows
  int nx, ny;   // tiles across and down
  int batches;  // batch elements a workgroup takes
  int workgroups;
};

constexpr int kSmPix = 32;       // pixels of a wave
constexpr int kSmGroup = 5;      // samples of a lane whose taps are held at a time
// Image elements of a tile's window.  32 x 4 pixels of a 3 x 3 kernel need 7 x 36 at the equator;
// 7 x 132 where the kernel is 18 degrees wide, five rows from a pole of a 512-row image.  20 KB
// with 16-byte elements leave room for six workgroups per CU.  A tile that needs more (the rows
// next to a pole, incoherent maps) reads its taps from global memory.
constexpr int kSmWindow = 1280;

typedef float f32x4 __attribute__((ext_vector_type(4)));
// Last word of a buffer descriptor: raw 32-bit data, no swizzle.  A store through one takes the
// channel's row as a scalar offset, where a flat address would cost two 64-bit additions per
// value (with them the 16 stores of a wave were a third of the forward's instructions).
constexpr int kRawBuffer = 0x00027000;

// A window element: the channels of an image element side by side.
template <int CG>
struct SmallElem {
  using type = f32x4;
  static constexpr int kFloats = 4;
  static __device__ __forceinline__ float channel(type v, int c) { return v[c]; }
};
template <>
struct SmallElem<1> {
  using type = float;
  static constexpr int kFloats = 1;
  static __device__ __forceinline__ float channel(type v, int) { return v; }
};

// A lane's samples of one point each, before the window is known: row and (anchored) column of the
// first tap, coefficients of all (0: inactive).  The other taps lie one row down and one column on.
template <int INTERP, int G>
struct LaneSamples {
  static constexpr int N = PointTaps<float, INTERP>::N;
  int y[G], d[G];
  float co[G][N];
};
// The same ready for use: LDS byte offset of the window element (window tiles) or flat image
// offset (others, -1: none), and coefficient.  Inactive taps point at the window's zero element,
// so no value they would have named can reach the sum.
template <int INTERP, int G>
struct LaneTaps {
  static constexpr int N = PointTaps<float, INTERP>::N;
  int off[G][N];
  float co[G][N];
};

struct TileWindow {
  int y0, x0;   // first row; first column relative to the anchor
  int rows, cols;
  int anchor;
  bool fits;
};

// Column distance from the anchor, modulo the image width: a tile at the wrap seam stays compact.
__device__ __forceinline__ int wrapped_distance(int x, int anchor, int W) {
  int d = x - anchor;
  if (d >= W - W / 2) d -= W;
  if (d < -(W / 2)) d += W;
  return d;
}
template <int INTERP>
__device__ __forceinline__ int tile_anchor(float x, float y, int H, int W) {
  PointTaps<float, INTERP> t;
  t.set(x, y, H, W);
  return __builtin_amdgcn_readfirstlane(t.off[0] >= 0 ? t.tx[0] : 0);
}

// Map entries of samples k0 .. k0 + G - 1 (point p) of pixel m; past K the last repeats.
template <bool WEIGHTED, int G>
struct LanePoints {
  float x[G], y[G], wt[G];
  __device__ __forceinline__ void read(const float* __restrict__ map,
                                       const float* __restrict__ wts, size_t m, int k0, int K,
                                       int P, int p) {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      size_t s = m * K + min(k0 + g, K - 1);
      if constexpr (WEIGHTED) s = s * P + p;
      x[g] = map[s * 2];
      y[g] = map[s * 2 + 1];
      if constexpr (WEIGHTED) wt[g] = wts[s];
    }
  }
};

// Their taps; samples from `live` on do not exist.
template <int INTERP, bool WEIGHTED, int G>
__device__ __forceinline__ void decode(const LanePoints<WEIGHTED, G>& pt, int live, int anchor,
                                       int H, int W, LaneSamples<INTERP, G>& out) {
#pragma unroll
  for (int g = 0; g < G; ++g) {
    // PointTaps<float, INTERP>::set without the offsets: what is out of the image, or a sample
    // that does not exist, gets coefficient 0
    const float x = pt.x[g], y = pt.y[g];
    const float wt = WEIGHTED ? pt.wt[g] : 1.0f;
    if constexpr (INTERP == 0) {
      const int xi = to_int_clamped(round_t(x)), yi = to_int_clamped(round_t(y));
      const bool on = g < live && (unsigned)xi < (unsigned)W && (unsigned)yi < (unsigned)H;
      out.y[g] = yi;
      out.d[g] = wrapped_distance(xi, anchor, W);
      out.co[g][0] = on ? wt : 0.0f;
    } else {
      const float fx = floor_t(x), fy = floor_t(y);
      const int x1 = to_int_clamped(fx), y1 = to_int_clamped(fy);
      const float A = (fy + 1.0f) - y, B = (fx + 1.0f) - x, C = x - fx, D = y - fy;
      const bool y1ok = g < live && (unsigned)y1 < (unsigned)H;
      const bool y2ok = g < live && (unsigned)(y1 + 1) < (unsigned)H;
      const bool x1ok = INTERP == 2 || (unsigned)x1 < (unsigned)W;
      const bool x2ok = INTERP == 2 || (unsigned)(x1 + 1) < (unsigned)W;
      out.y[g] = y1;
      out.d[g] = wrapped_distance(INTERP == 2 ? wrap_index(x1, W) : x1, anchor, W);
      const float w0 = A * B, w1 = A * C, w2 = D * B, w3 = D * C;
      out.co[g][0] = y1ok && x1ok ? (WEIGHTED ? wt * w0 : w0) : 0.0f;
      out.co[g][1] = y1ok && x2ok ? (WEIGHTED ? wt * w1 : w1) : 0.0f;
      out.co[g][2] = y2ok && x1ok ? (WEIGHTED ? wt * w2 : w2) : 0.0f;
      out.co[g][3] = y2ok && x2ok ? (WEIGHTED ? wt * w3 : w3) : 0.0f;
    }
    __builtin_amdgcn_sched_barrier(0);   // a sample at a time: registers
  }
}

// Bounding box of active taps.
struct TapBox {
  int y_lo = 1 << 30, y_hi = -1, x_lo = 1 << 30, x_hi = -(1 << 30);
  template <int INTERP, int G>
  __device__ __forceinline__ void add(const LaneSamples<INTERP, G>& s) {
    constexpr int kFar = 1 << 30;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      bool on[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) on[i] = i < s.N && s.co[g][i < s.N ? i : 0] != 0.0f;
      const bool top = on[0] || on[1], bottom = on[2] || on[3];
      const bool left = on[0] || on[2], right = on[1] || on[3];
      y_lo = min(y_lo, top ? s.y[g] : (bottom ? s.y[g] + 1 : kFar));
      y_hi = max(y_hi, bottom ? s.y[g] + 1 : (top ? s.y[g] : -1));
      x_lo = min(x_lo, left ? s.d[g] : (right ? s.d[g] + 1 : kFar));
      x_hi = max(x_hi, right ? s.d[g] + 1 : (left ? s.d[g] : -kFar));
    }
  }
  // over the workgroup; red: 4 ints per wave in LDS
  __device__ __forceinline__ TileWindow window(int anchor, int waves, int* red) {
#pragma unroll
    for (int d = 32; d >= 1; d >>= 1) {
      y_lo = min(y_lo, __shfl_xor(y_lo, d));
      y_hi = max(y_hi, __shfl_xor(y_hi, d));
      x_lo = min(x_lo, __shfl_xor(x_lo, d));
      x_hi = max(x_hi, __shfl_xor(x_hi, d));
    }
    const int wave = threadIdx.x >> 6;
    if ((threadIdx.x & 63) == 0) {
      red[wave * 4] = y_lo;
      red[wave * 4 + 1] = y_hi;
      red[wave * 4 + 2] = x_lo;
      red[wave * 4 + 3] = x_hi;
    }
    __syncthreads();
    for (int w = 0; w < waves; ++w) {
      y_lo = min(y_lo, red[w * 4]);
      y_hi = max(y_hi, red[w * 4 + 1]);
      x_lo = min(x_lo, red[w * 4 + 2]);
      x_hi = max(x_hi, red[w * 4 + 3]);
    }
    TileWindow win;
    win.anchor = anchor;
    win.y0 = __builtin_amdgcn_readfirstlane(y_lo);
    win.x0 = __builtin_amdgcn_readfirstlane(x_lo);
    win.rows = __builtin_amdgcn_readfirstlane(y_hi) - win.y0 + 1;
    win.cols = __builtin_amdgcn_readfirstlane(x_hi) - win.x0 + 1;
    if (win.rows <= 0) win.rows = win.cols = 0;   // no active tap
    win.fits = win.rows * (int64_t)win.cols <= kSmWindow;
    return win;
  }
};

template <int INTERP, int G>
__device__ __forceinline__ void place(const LaneSamples<INTERP, G>& s, const TileWindow& win, int W,
                                      int elem_bytes, LaneTaps<INTERP, G>& out) {
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int i = 0; i < s.N; ++i) out.co[g][i] = s.co[g][i];
  if (win.fits) {
    const int zero = win.rows * win.cols * elem_bytes, row = win.cols * elem_bytes;
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const int e0 = ((s.y[g] - win.y0) * win.cols + (s.d[g] - win.x0)) * elem_bytes;
#pragma unroll
      for (int i = 0; i < s.N; ++i)
        out.off[g][i] = s.co[g][i] != 0.0f ? e0 + (i >> 1) * row + (i & 1) * elem_bytes : zero;
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < s.N; ++i) {
        int col = win.anchor + s.d[g] + (i & 1);
        if (col < 0) col += W;
        if (col >= W) col -= W;
        out.off[g][i] = s.co[g][i] != 0.0f ? (s.y[g] + (i >> 1)) * W + col : -1;
      }
  }
}

// The window of a workgroup's tile from the taps of all its lanes' samples.  TAPS (one group, one
// point: `first` holds them): and the taps themselves, which then serve every batch element.
template <int INTERP, bool WEIGHTED, bool TAPS>
__device__ __forceinline__ TileWindow tile_window(const LanePoints<WEIGHTED, kSmGroup>& first,
                                                  const float* __restrict__ map,
                                                  const float* __restrict__ wts, size_t m,
                                                  int k_first, int samples, int K, int P,
                                                  int anchor, int H, int W, int waves, int* red,
                                                  int elem_bytes,
                                                  LaneTaps<INTERP, kSmGroup>& taps) {
  TapBox box;
  LaneSamples<INTERP, kSmGroup> s;
  if constexpr (TAPS) {
    decode<INTERP, WEIGHTED, kSmGroup>(first, samples, anchor, H, W, s);
    box.add(s);
    const TileWindow win = box.window(anchor, waves, red);
    place(s, win, W, elem_bytes, taps);
    return win;
  } else {
    const int q = WEIGHTED ? P : 1;
    for (int k0 = 0; k0 < samples; k0 += kSmGroup)
      for (int p = 0; p < q; ++p) {
        LanePoints<WEIGHTED, kSmGroup> pt;
        pt.read(map, wts, m, k_first + k0, K, P, p);
        decode<INTERP, WEIGHTED, kSmGroup>(pt, samples - k0, anchor, H, W, s);
        box.add(s);
      }
    return box.window(anchor, waves, red);
  }
}

// Elements of one batch element's window, the zero element behind it included, and how many
// batch elements the window space holds at a time.
__device__ __forceinline__ int window_stride(const TileWindow& win) {
  return win.rows * win.cols + 1;
}
__device__ __forceinline__ int windows_at_once(const TileWindow& win, int batches) {
  if (!win.fits) return 1;
  return __builtin_amdgcn_readfirstlane(min(batches, (kSmWindow + 1) / window_stride(win)));
}

// Copies the windows of `count` batch elements from img0 on into LDS, all channels of an element
// together, a zero element behind each.  A wave takes 64 columns of a row at a time, of four
// batch elements together; everything but a lane's column is uniform over the wave.
// PAD: there may be fewer channels than CG (two at least), and the others have to read as zero: their
// weights are zero, but zero times an infinity is not.
template <int CG, bool PAD>
__device__ __forceinline__ void stage_windows(const TileWindow& win, const float* __restrict__ img0,
                                              int count, size_t HW, int Cg, int W, int waves,
                                              float* __restrict__ lds) {
  using Elem = typename SmallElem<CG>::type;
  Elem* out = reinterpret_cast<Elem*>(lds);
  constexpr int U = 4;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int stride = window_stride(win);
  for (int c0 = 0; c0 < win.cols; c0 += 64) {
    const int c = c0 + lane;
    const bool on = c < win.cols;
    int col = win.anchor + win.x0 + (on ? c : 0);
    if (col < 0) col += W;
    if (col >= W) col -= W;
    for (int r = wave; r < win.rows; r += waves) {
      const float* row = img0 + (size_t)(win.y0 + r) * W;
      const int at = r * win.cols + c;
      for (int j0 = 0; j0 < count; j0 += U) {
        float v[U][CG];
#pragma unroll
        for (int i = 0; i < U; ++i) {
          const float* src = row + (size_t)min(j0 + i, count - 1) * Cg * HW;
#pragma unroll
          for (int ch = 0; ch < CG; ++ch) v[i][ch] = (src + (size_t)(ch < Cg ? ch : 0) * HW)[col];
          if constexpr (PAD) {
#pragma unroll
            for (int ch = 2; ch < CG; ++ch) v[i][ch] = ch < Cg ? v[i][ch] : 0.0f;
          }
        }
        if (on) {
#pragma unroll
          for (int i = 0; i < U; ++i) {
            if (j0 + i < count) {
              Elem* dst = out + (j0 + i) * stride + at;
              if constexpr (CG == 1) *dst = v[i][0];
              else *dst = f32x4{v[i][0], v[i][1], CG > 2 ? v[i][CG > 2 ? 2 : 0] : 0.0f, CG > 3 ? v[i][CG - 1] : 0.0f};
            }
          }
        }
      }
    }
  }
  for (int j = threadIdx.x; j < count; j += 64 * waves) out[j * stride + stride - 1] = Elem{};
}

// An integer the compiler must take as it is, here: what is computed from it stays in its loop
// (hoisted out of the loop over the batch, the addresses of the path below would not fit in
// registers).
__device__ __forceinline__ int opaque(int x) {
  asm volatile("" : "+v"(x));
  return x;
}

// col[g][c] += the lane's column values of G samples.  The reads of a sample are requested before
// the blend of the one before it.
template <int INTERP, int CG, int G, bool PAD>
__device__ __forceinline__ void add_columns(const LaneTaps<INTERP, G>& t, bool fits,
                                            const float* __restrict__ window,
                                            const float* __restrict__ img_b, size_t HW, int Cg,
                                            float (&col)[G][CG]) {
  constexpr int N = LaneTaps<INTERP, G>::N;
  using Elem = typename SmallElem<CG>::type;
  if (fits) {
    const char* base = reinterpret_cast<const char*>(window);
    Elem d[2][N];
#pragma unroll
    for (int i = 0; i < N; ++i) d[0][i] = *reinterpret_cast<const Elem*>(base + t.off[0][i]);
#pragma unroll
    for (int g = 0; g < G; ++g) {
      if (g + 1 < G) {
#pragma unroll
        for (int i = 0; i < N; ++i)
          d[(g + 1) & 1][i] = *reinterpret_cast<const Elem*>(base + t.off[g + 1][i]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < CG; ++c)
          col[g][c] = __builtin_fmaf(t.co[g][i], SmallElem<CG>::channel(d[g & 1][i], c), col[g][c]);
      __builtin_amdgcn_sched_barrier(0);
    }
  } else {
#pragma unroll
    for (int g = 0; g < G; ++g) {
      float d[N][CG];
      int o[N];
#pragma unroll
      for (int i = 0; i < N; ++i) {
        o[i] = opaque(t.off[g][i]);
#pragma unroll
        for (int c = 0; c < CG; ++c)
          d[i][c] = img_b[(size_t)(c < Cg ? c : 0) * HW + max(o[i], 0)];
      }
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < CG; ++c) pin(d[i][c]);
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < CG; ++c)
          col[g][c] = __builtin_fmaf(t.co[g][i], o[i] >= 0 && (!PAD || c < 2 || c < Cg) ? d[i][c] : 0.0f,
                                     col[g][c]);
      __builtin_amdgcn_sched_barrier(0);   // one sample's reads in flight: registers
    }
  }
}

// What a lane knows about its place in tile t.
struct LanePixel {
  int m;          // its pixel (a valid one also where `valid` is false)
  bool valid;
  int first;      // first pixel of its wave
  int count;      // pixels of its wave that exist
  int k_first;    // first of the lane's samples
  int samples;    // how many it has (none without a pixel)
  size_t anchor_sample;
};
__device__ __forceinline__ LanePixel lane_pixel(const SmallTiling& tl, int tile, int OW, int M,
                                                int K, int points, int half_samples) {
  LanePixel p;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int tx = tile % tl.nx, ty = tile / tl.nx;
  const int row0 = tl.stacked ? ty * tl.waves : ty;
  const int x0 = (tl.stacked ? tx : tx * tl.waves) * kSmPix;
  const int row = row0 + (tl.stacked ? wave : 0), x = x0 + (tl.stacked ? 0 : wave * kSmPix);
  const int lane = threadIdx.x & 63, px = lane & 31, h = lane >> 5;
  const int OH = M / OW;
  p.count = row < OH ? max(0, min(kSmPix, OW - x)) : 0;
  p.first = p.count > 0 ? row * OW + x : 0;
  p.valid = px < p.count;
  p.m = p.valid ? p.first + px : row0 * OW + x0;
  p.k_first = h * half_samples;
  p.samples = p.valid ? max(0, min(half_samples, K - p.k_first)) : 0;
  p.anchor_sample = ((size_t)(row0 * OW + x0) * K + K / 2) * points;
  return p;
}

// The weight matrix Wm[Cp][Cg][K] into LDS as wl[Cp][CG][KMAX], zero where c >= Cg or k >= K, so
// the loops over (c, k) need no guards and address with constants.  Every lane reads the same
// element at a time, which the LDS serves as a broadcast.
template <int CG, int KMAX>
__device__ __forceinline__ void stage_weights(const float* __restrict__ Wm, int Cp, int Cg, int K,
                                              float* __restrict__ wl) {
  for (int e = threadIdx.x; e < Cp * CG * KMAX; e += blockDim.x) {
    const int k = e % KMAX, c = (e / KMAX) % CG, n = e / (KMAX * CG);
    wl[e] = (c < Cg && k < K) ? Wm[((size_t)n * Cg + c) * K + k] : 0.0f;
  }
  __syncthreads();
}

// Column values of G consecutive samples (first: sample0; only the first `valid` exist, the
// others repeat the last) of one pixel for CG channels: v[g][c].  All map reads of the group
// are issued together, then all image reads, then the blend.
template <int INTERP, bool WEIGHTED, int CG, int G>
__device__ __forceinline__ void column_group(const float* __restrict__ img_b, size_t HW,
                                             const float* __restrict__ map,
                                             const float* __restrict__ wts, size_t sample0,
                                             int valid, int P, int H, int W, int Cg,
                                             float (&v)[G][CG]) {
  constexpr int N = PointTaps<float, INTERP>::N;
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int c = 0; c < CG; ++c) v[g][c] = 0.0f;
  const int q = WEIGHTED ? P : 1;
  for (int p = 0; p < q; ++p) {
    float mx[G], my[G], wt[G];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      const size_t s = (sample0 + (g < valid ? g : valid - 1)) * q + p;
      mx[g] = map[s * 2];
      my[g] = map[s * 2 + 1];
      wt[g] = WEIGHTED ? wts[s] : 1.0f;
    }
    PointTaps<float, INTERP> t[G];
    float d[G][N][CG];
#pragma unroll
    for (int g = 0; g < G; ++g) {
      t[g].set(mx[g], my[g], H, W);
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const size_t o = t[g].off[i] >= 0 ? (size_t)t[g].off[i] : 0;
#pragma unroll
        for (int c = 0; c < CG; ++c) d[g][i][c] = img_b[(size_t)(c < Cg ? c : 0) * HW + o];
      }
    }
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int i = 0; i < N; ++i)
#pragma unroll
        for (int c = 0; c < CG; ++c) pin(d[g][i][c]);
#pragma unroll
    for (int g = 0; g < G; ++g) {
#pragma unroll
      for (int i = 0; i < N; ++i) {
        const float co = WEIGHTED ? wt[g] * t[g].w[i] : t[g].w[i];
        const bool on = t[g].off[i] >= 0 && co != 0.0f;
#pragma unroll
        for (int c = 0; c < CG; ++c)
          v[g][c] = __builtin_fmaf(on ? co : 0.0f, on ? d[g][i][c] : 0.0f, v[g][c]);
      }
    }
  }
}

// One thread per pixel gathers its Cg * K column values once into registers and forms every
// output channel from them on the vector unit.  grid (pixel blocks, batch); KMAX bounds K
// (register array).  For layers of few outputs: see small_forward.
template <int INTERP, bool WEIGHTED, int CG, int KMAX>
__global__ __launch_bounds__(kSmThreads) void small_pixel_forward_kernel(
    const float* __restrict__ img, const float* __restrict__ map, const float* __restrict__ wts,
    const float* __restrict__ Wm, const float* __restrict__ bias, float* __restrict__ pix, int Cg,
    int H, int W, int Cp, int M, int K, int P) {
  extern __shared__ __align__(16) float wl[];
  stage_weights<CG, KMAX>(Wm, Cp, Cg, K, wl);
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const size_t HW = (size_t)H * W;
  const float* img_b = img + (size_t)blockIdx.y * Cg * HW;
  constexpr int G = 3;                      // samples whose reads are in flight together
  constexpr int KPAD = (KMAX + G - 1) / G * G;
  float col[KPAD][CG];
#pragma unroll
  for (int k0 = 0; k0 < KPAD; k0 += G) {
    if (k0 < K) {
      float grp[G][CG];
      column_group<INTERP, WEIGHTED, CG, G>(img_b, HW, map, wts, (size_t)m * K + k0,
                                            min(G, K - k0), P, H, W, Cg, grp);
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < CG; ++c) col[k0 + g][c] = grp[g][c];
    } else {
#pragma unroll
      for (int g = 0; g < G; ++g)
#pragma unroll
        for (int c = 0; c < CG; ++c) col[k0 + g][c] = 0.0f;
    }
  }
  // what has no sample or channel of its own (the group's last repeated, channel 0) meets weights of
  // zero, but zero times an infinity is not zero
  if (K < KPAD || Cg < CG) {
#pragma unroll
    for (int k = 0; k < KPAD; ++k)
#pragma unroll
      for (int c = 0; c < CG; ++c) col[k][c] = k < K && c < Cg ? col[k][c] : 0.0f;
  }
  float* out = pix + (size_t)blockIdx.y * Cp * M + m;
  for (int n = 0; n < Cp; ++n) {
    const float* wrow = wl + n * (CG * KMAX);
    float acc = bias != nullptr ? bias[n] : 0.0f;
#pragma unroll
    for (int c = 0; c < CG; ++c) {
#pragma unroll
      for (int k = 0; k < KMAX; ++k) acc = __builtin_fmaf(wrow[c * KMAX + k], col[k][c], acc);
    }
    out[(size_t)n * M] = acc;
  }
}

// img[b][c][tap] += coefficient * sum_n Wm[n][c][k] * pix[b][n][m] over the taps of (m, k): the
// transpose of the forward.  One thread per pixel forms its Cg * K products with the weights
// in LDS and splats them with float atomics; img must hold the values to add to.
template <int INTERP, bool WEIGHTED, int CG, int KMAX>
__global__ __launch_bounds__(kSmThreads) void small_scatter_kernel(
    const float* __restrict__ pix, const float* __restrict__ map, const float* __restrict__ wts,
    const float* __restrict__ Wm, float* __restrict__ img, int Cg, int H, int W, int Cp, int M,
    int K, int P) {
  extern __shared__ __align__(16) float wl[];
  stage_weights<CG, KMAX>(Wm, Cp, Cg, K, wl);
  const int m = blockIdx.x * blockDim.x + threadIdx.x;
  if (m >= M) return;
  const size_t HW = (size_t)H * W;
  float* img_b = img + (size_t)blockIdx.y * Cg * HW;
  const float* in = pix + (size_t)blockIdx.y * Cp * M + m;
  float t[KMAX][CG];
#pragma unroll
  for (int k = 0; k < KMAX; ++k)
#pragma unroll
    for (int c = 0; c < CG; ++c) t[k][c] = 0.0f;
  for (int n = 0; n < Cp; ++n) {
    const float g = in[(size_t)n * M];
    const float* wrow = wl + n * (CG * KMAX);
#pragma unroll
    for (int c = 0; c < CG; ++c) {
#pragma unroll
      for (int k = 0; k < KMAX; ++k) t[k][c] = __builtin_fmaf(wrow[c * KMAX + k], g, t[k][c]);
    }
  }
  const int q = WEIGHTED ? P : 1;
  PointTaps<float, INTERP> tp;
  for (int p = 0; p < q; ++p) {
    // the map entries of all samples first (one round trip), then taps and atomics
    float mx[KMAX], my[KMAX], wt[KMAX];
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      const size_t s = ((size_t)m * K + (k < K ? k : K - 1)) * q + p;
      mx[k] = map[s * 2];
      my[k] = map[s * 2 + 1];
      wt[k] = WEIGHTED ? wts[s] : 1.0f;
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      pin(mx[k]);
      pin(my[k]);
      pin(wt[k]);
    }
#pragma unroll
    for (int k = 0; k < KMAX; ++k) {
      if (k < K) {
        tp.set(mx[k], my[k], H, W);
#pragma unroll
        for (int i = 0; i < PointTaps<float, INTERP>::N; ++i) {
          const float co = WEIGHTED ? wt[k] * tp.w[i] : tp.w[i];
          if (tp.off[i] >= 0 && co != 0.0f) {
#pragma unroll
            for (int c = 0; c < CG; ++c)
              if (c < Cg) atomic_add_noret(img_b + (size_t)c * HW + tp.off[i], co * t[k][c]);
          }
        }
      }
    }
  }
}

// grid (tiles, batch parts, channel chunks of 32 NB).  NG: groups of kSmGroup samples a lane half
// takes.  The weights of step (sample, c) lie in LDS as the A operands of the MFMAs.
//
// 3 -> 32 channels at 512 x 1024, B = 4, bilinear, K = 9 (268 MB written): 148 us with a thread
// per pixel that gathered from global memory and multiplied on the vector unit, 101 us now, of
// which 32 us are vector (1015 instructions a wave) and 31 us matrix instructions; those add up, and
// four waves per SIMD do not cover all of a tile's serial start (map, box, window): waves wait 0.42
// of their cycles.  A window per wave instead of
// per workgroup saves the two barriers and doubles the window reads: 119 us.
template <int INTERP, bool WEIGHTED, int CG, int NG, int NB>
__global__ __launch_bounds__(kSmThreads, small_waves(NG, NB)) void small_forward_kernel(
    const float* __restrict__ img, const float* __restrict__ map, const float* __restrict__ wts,
    const float* __restrict__ Wm, const float* __restrict__ bias, float* __restrict__ pix, int Cg,
    int H, int W, int Cp, int M, int OW, int K, int P, int B, SmallTiling tl) {
  constexpr int E = SmallElem<CG>::kFloats, HALF = NG * kSmGroup, STEPS = HALF * CG;
  constexpr bool kPad = NG > 1;   // (CG is the image's own number of channels otherwise)
  extern __shared__ __align__(16) float lds[];
  float* window = lds;                                  // [kSmWindow + 1][E]
  float* wl = lds + (kSmWindow + 1) * E + (CG == 1 ? 3 : 0);   // [STEPS][64][NB]
  float* bl = wl + STEPS * 64 * NB;                     // [32 NB]
  int* red = reinterpret_cast<int*>(bl + 32 * NB);
  const int lane = threadIdx.x & 63, h = lane >> 5;
  const int n0 = blockIdx.z * 32 * NB;
  for (int st = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6); st < STEPS; st += tl.waves) {
    const int g = st / CG, c = st % CG, k = h * HALF + g;
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const int n = n0 + 32 * a + (lane & 31);
      const bool on = c < Cg && k < K && n < Cp;
      const float w = Wm[on ? (n * Cg + c) * K + k : 0];
      wl[(st * 64 + lane) * NB + a] = on ? w : 0.0f;
    }
  }
  for (int e = threadIdx.x; e < 32 * NB; e += 64 * tl.waves)
    bl[e] = (bias != nullptr && n0 + e < Cp) ? bias[n0 + e] : 0.0f;
  const size_t HW = (size_t)H * W;
  const int b_begin = blockIdx.y * tl.batches, b_end = min(B, b_begin + tl.batches);
  constexpr bool kHoist = NG == 1 && !WEIGHTED;   // the taps fit in registers for all of them

  const LanePixel lp = lane_pixel(tl, blockIdx.x, OW, M, K, WEIGHTED ? P : 1, HALF);
  const int anchor =
      tile_anchor<INTERP>(map[lp.anchor_sample * 2], map[lp.anchor_sample * 2 + 1], H, W);
  LanePoints<WEIGHTED, kSmGroup> first;
  if constexpr (kHoist) first.read(map, wts, lp.m, lp.k_first, K, P, 0);
  LaneTaps<INTERP, kSmGroup> taps;
  const TileWindow win = tile_window<INTERP, WEIGHTED, kHoist>(
      first, map, wts, lp.m, lp.k_first, lp.samples, K, P, anchor, H, W, tl.waves, red, E * 4, taps);
  const bool all_rows = n0 + 32 * NB <= Cp;
  const int at_once = windows_at_once(win, b_end - b_begin);
  const int stride = window_stride(win);
  for (int b = b_begin, j = 0; b < b_end; ++b, ++j) {
    const float* img_b = img + (size_t)b * Cg * HW;
    if (b == b_begin || j == at_once) {
      j = 0;
      __syncthreads();   // the windows' last readers are through (first round: red, wl, bl)
      if (win.fits) stage_windows<CG, kPad>(win, img_b, min(at_once, b_end - b), HW, Cg, W, tl.waves, window);
      __syncthreads();
    }
    const float* window_b = window + j * stride * E;
    floatx16 acc[NB];
#pragma unroll
    for (int a = 0; a < NB; ++a)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        const f32x4 v = *reinterpret_cast<const f32x4*>(bl + 32 * a + 8 * q + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[a][4 * q + i] = v[i];
      }
#pragma unroll
    for (int gr = 0; gr < NG; ++gr) {
      float col[kSmGroup][CG];
#pragma unroll
      for (int g = 0; g < kSmGroup; ++g)
#pragma unroll
        for (int c = 0; c < CG; ++c) col[g][c] = 0.0f;
      if constexpr (kHoist) {
        add_columns<INTERP, CG, kSmGroup, kPad>(taps, win.fits, window_b, img_b, HW, Cg, col);
      } else {
        const int q = WEIGHTED ? P : 1, k0 = gr * kSmGroup;
        for (int p = 0; p < q; ++p) {
          LanePoints<WEIGHTED, kSmGroup> pt;
          pt.read(map, wts, lp.m, lp.k_first + k0, K, P, p);
          LaneSamples<INTERP, kSmGroup> s;
          decode<INTERP, WEIGHTED, kSmGroup>(pt, lp.samples - k0, win.anchor, H, W, s);
          place(s, win, W, E * 4, taps);
          add_columns<INTERP, CG, kSmGroup, kPad>(taps, win.fits, window_b, img_b, HW, Cg, col);
        }
      }
#pragma unroll
      for (int g = 0; g < kSmGroup; ++g)
#pragma unroll
        for (int c = 0; c < CG; ++c) {
          const float* w = wl + (((gr * kSmGroup + g) * CG + c) * 64 + lane) * NB;
#pragma unroll
          for (int a = 0; a < NB; ++a)
            acc[a] = __builtin_amdgcn_mfma_f32_32x32x2f32(w[a], col[g][c], acc[a], 0, 0, 0);
        }
    }
    if (lp.valid) {
      // row 32 a + 8 (v / 4) + v % 4 of the block is uniform, its 4 h part goes to the lane
      const __amdgpu_buffer_rsrc_t out = __builtin_amdgcn_make_buffer_rsrc(
          pix + ((size_t)b * Cp + n0) * M, 0, min(32 * NB, Cp - n0) * M * 4, kRawBuffer);
      const int lane_at = (4 * h * M + lp.m) * 4;
      const auto store = [&](int a, int v) {
        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(acc[a][v]), out, lane_at,
                                              (32 * a + 8 * (v >> 2) + (v & 3)) * M * 4, 0);
      };
      if (all_rows) {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int v = 0; v < 16; ++v) store(a, v);
      } else {
#pragma unroll
        for (int a = 0; a < NB; ++a)
#pragma unroll
          for (int v = 0; v < 16; ++v)
            if (n0 + 32 * a + 8 * (v >> 2) + (v & 3) + 4 * h < Cp) store(a, v);
      }
    }
  }
}

// grid (workgroups, batch parts, channel chunks of 32 NB); a workgroup walks the tiles
// blockIdx.x, blockIdx.x + gridDim.x, ...  The column values of a wave's 32 pixels go through an LDS
// tile of the wave's own, colT[(k, c)][pixel], because here the pixel is the reduction index;
// the pixel-side operand is read straight from memory, 16 bytes of a row per lane (a lane half
// takes four consecutive pixels, the order of the reduction being free).  The waves' sums leave
// the workgroup as one float atomic per element of gW.  gbias (optional): the sums of the
// pixel-side rows, from the same registers, one atomic per channel and wave.
//
// The layer above: 457 us when every (c, k) worked out its own taps, about 150 now (268 MB of pixel-side
// values read, 31 us of matrix instructions); waves wait 0.57 of their cycles for a tile's map, box and
// window.  With a window per wave 171 us.
// 32-column blocks of (k, c)
constexpr int small_columns(int NG, int CG) { return (2 * NG * kSmGroup * CG + 31) / 32; }
constexpr int kSmLd = 36;   // row stride of colT (floats): 16-byte reads of 8 rows cover the banks
template <int INTERP, bool WEIGHTED, int CG, int NG, int NB>
__global__ __launch_bounds__(kSmThreads, small_waves(NG, 1 + NB * small_columns(NG, CG))) void small_wgrad_kernel(
    const float* __restrict__ pix, const float* __restrict__ img, const float* __restrict__ map,
    const float* __restrict__ wts, float* __restrict__ gW, float* __restrict__ gbias, int Cg,
    int H, int W, int Cp, int M, int OW, int K, int P, int B, SmallTiling tl) {
  constexpr int E = SmallElem<CG>::kFloats, HALF = NG * kSmGroup;
  constexpr int CB = small_columns(NG, CG);
  extern __shared__ __align__(16) float lds[];
  float* window = lds;   // [kSmWindow + 1][E]
  float* colT = lds + (kSmWindow + 1) * E + (CG == 1 ? 3 : 0) +
                (threadIdx.x >> 6) * (32 * CB * kSmLd);   // [32 CB][kSmLd] per wave
  int* red = reinterpret_cast<int*>(lds + (kSmWindow + 1) * E + (CG == 1 ? 3 : 0) +
                                    tl.waves * (32 * CB * kSmLd));
  const int lane = threadIdx.x & 63, nl = lane & 31, h = lane >> 5;
  const int n0 = blockIdx.z * 32 * NB;
  const size_t HW = (size_t)H * W;
  const int b_begin = blockIdx.y * tl.batches, b_end = min(B, b_begin + tl.batches);
  constexpr bool kHoist = NG == 1 && !WEIGHTED;
  floatx16 acc[NB][CB];
  float row_sum[NB];
#pragma unroll
  for (int a = 0; a < NB; ++a) {
    row_sum[a] = 0.0f;
#pragma unroll
    for (int cb = 0; cb < CB; ++cb)
#pragma unroll
      for (int v = 0; v < 16; ++v) acc[a][cb][v] = 0.0f;
  }
  // the next tile's map entries are requested before the work on a tile
  const int tiles = tl.nx * tl.ny;
  LanePoints<WEIGHTED, kSmGroup> ahead;
  float ahead_x = 0.0f, ahead_y = 0.0f;
  const auto request_map = [&](const LanePixel& p) {
    ahead_x = map[p.anchor_sample * 2];
    ahead_y = map[p.anchor_sample * 2 + 1];
    if constexpr (kHoist) ahead.read(map, wts, p.m, p.k_first, K, P, 0);
  };
  LanePixel lp = lane_pixel(tl, blockIdx.x, OW, M, K, WEIGHTED ? P : 1, HALF);
  request_map(lp);
  for (int t = blockIdx.x; t < tiles; t += tl.workgroups) {
    __syncthreads();   // red
    const int anchor = tile_anchor<INTERP>(ahead_x, ahead_y, H, W);
    LaneTaps<INTERP, kSmGroup> taps;
    const TileWindow win = tile_window<INTERP, WEIGHTED, kHoist>(
        ahead, map, wts, lp.m, lp.k_first, lp.samples, K, P, anchor, H, W, tl.waves, red, E * 4,
        taps);
    LanePixel lp_next = lp;
    if (t + tl.workgroups < tiles) {
      lp_next = lane_pixel(tl, t + tl.workgroups, OW, M, K, WEIGHTED ? P : 1, HALF);
      request_map(lp_next);
    }
    const int at_once = windows_at_once(win, b_end - b_begin);
    const int stride = window_stride(win);
    // pixel-side values: lane (n, h) pixels 8 q + 4 h .. + 3 of row n, requested a batch element
    // ahead; pixels past the wave's are zero, rows past Cp repeat the last (their sums are
    // not written)
    f32x4 next[NB][4];
    const auto request = [&](int b) {
#pragma unroll
      for (int a = 0; a < NB; ++a) {
        const int n = n0 + 32 * a + nl;
        const float* row = pix + ((size_t)b * Cp + min(n, Cp - 1)) * M + lp.first;
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const int p = 8 * q + 4 * h;
          if (lp.count == kSmPix) {
            typedef f32x4 __attribute__((aligned(4))) f32x4u;
            next[a][q] = *reinterpret_cast<const f32x4u*>(row + p);
          } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) next[a][q][i] = p + i < lp.count ? row[p + i] : 0.0f;
          }
        }
      }
    };
    if (b_begin < b_end) request(b_begin);
    for (int b = b_begin, j = 0; b < b_end; ++b, ++j) {
      const float* img_b = img + (size_t)b * Cg * HW;
      if (b == b_begin || j == at_once) {
        j = 0;
        __syncthreads();   // the windows' last readers are through
        if (win.fits) stage_windows<CG, false>(win, img_b, min(at_once, b_end - b), HW, Cg, W, tl.waves, window);
        __syncthreads();
      }
      const float* window_b = window + j * stride * E;
#pragma unroll
      for (int gr = 0; gr < NG; ++gr) {
        float col[kSmGroup][CG];
#pragma unroll
        for (int g = 0; g < kSmGroup; ++g)
#pragma unroll
          for (int c = 0; c < CG; ++c) col[g][c] = 0.0f;
        if constexpr (kHoist) {
          add_columns<INTERP, CG, kSmGroup, false>(taps, win.fits, window_b, img_b, HW, Cg, col);
        } else {
          const int q = WEIGHTED ? P : 1, k0 = gr * kSmGroup;
          for (int p = 0; p < q; ++p) {
            LanePoints<WEIGHTED, kSmGroup> pt;
            pt.read(map, wts, lp.m, lp.k_first + k0, K, P, p);
            LaneSamples<INTERP, kSmGroup> s;
            decode<INTERP, WEIGHTED, kSmGroup>(pt, lp.samples - k0, win.anchor, H, W, s);
            place(s, win, W, E * 4, taps);
            add_columns<INTERP, CG, kSmGroup, false>(taps, win.fits, window_b, img_b, HW, Cg, col);
          }
        }
#pragma unroll
        for (int g = 0; g < kSmGroup; ++g)
#pragma unroll
          for (int c = 0; c < CG; ++c)
            colT[((h * HALF + gr * kSmGroup + g) * CG + c) * kSmLd + nl] = col[g][c];
      }
      f32x4 av[NB][4];
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int q = 0; q < 4; ++q) av[a][q] = next[a][q];
      if (b + 1 < b_end) request(b + 1);
      wave_exchange();
      float sum_b[NB] = {};   // (this batch element's sixteen pixels apart: half the error of one chain)
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        f32x4 bv[CB];
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
          bv[cb] = *reinterpret_cast<const f32x4*>(colT + (32 * cb + nl) * kSmLd + 8 * q + 4 * h);
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
          for (int a = 0; a < NB; ++a) {
            sum_b[a] += av[a][q][i];
#pragma unroll
            for (int cb = 0; cb < CB; ++cb)
              acc[a][cb] = __builtin_amdgcn_mfma_f32_32x32x2f32(av[a][q][i], bv[cb][i], acc[a][cb],
                                                                0, 0, 0);
          }
      }
#pragma unroll
      for (int a = 0; a < NB; ++a) row_sum[a] += sum_b[a];
      wave_exchange();   // (the next batch element's columns go where these were)
    }
    lp = lp_next;
  }
  // ---- the waves' sums one after the other into LDS (over the tiles' space), then one atomic per
  // element.  D[row][column]: register v of lane l holds row 8 (v / 4) + 4 (l / 32) + v % 4,
  // column l % 32.
  constexpr int COLS = 32 * CB;
  float* sum = lds;   // [32 NB][COLS]
  const int wave = threadIdx.x >> 6;
  for (int w = 0; w < tl.waves; ++w) {
    __syncthreads();
    if (wave == w) {
#pragma unroll
      for (int a = 0; a < NB; ++a)
#pragma unroll
        for (int cb = 0; cb < CB; ++cb)
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int e = (32 * a + 8 * (v >> 2) + 4 * h + (v & 3)) * COLS + 32 * cb + nl;
            sum[e] = w == 0 ? acc[a][cb][v] : sum[e] + acc[a][cb][v];
          }
    }
  }
  __syncthreads();
  for (int e = threadIdx.x; e < 32 * NB * COLS; e += 64 * tl.waves) {
    const int n = n0 + e / COLS, k = e % COLS / CG, c = e % COLS % CG;
    if (n < Cp && k < K && c < Cg) atomic_add_noret(gW + ((size_t)n * Cg + c) * K + k, sum[e]);
  }
  if (gbias != nullptr) {
    // (the waves' sums together: an atomic each, one after the other on the channel, lost twice the bits)
    __syncthreads();   // the readers of sum are through
#pragma unroll
    for (int a = 0; a < NB; ++a) {
      const float s = row_sum[a] + __shfl_xor(row_sum[a], 32);
      if (h == 0) sum[(wave * NB + a) * 32 + nl] = s;
    }
    __syncthreads();
    if (threadIdx.x < 32 * NB && n0 + (int)threadIdx.x < Cp) {
      float s = sum[threadIdx.x];
      for (int w = 1; w < tl.waves; ++w) s += sum[w * NB * 32 + threadIdx.x];
      atomic_add_noret(gbias + n0 + threadIdx.x, s);
    }
  }
}

}  // namespace

bool small_conv_supported(const ConvGeom& g) {
  return g.Cg >= 1 && g.Cg <= 4 && g.K >= 1 && g.K <= 25 && g.Cp >= 1 && g.Cp <= 128 &&
         g.B <= 65535 && (int64_t)g.Cg * g.H * g.W < ((int64_t)1 << 31) &&
         (int64_t)g.M * g.K * (g.P > 0 ? g.P : 1) * 2 < ((int64_t)1 << 31);
}

static int padded_blocks(int64_t n) {
  const int b = (int)ceil_div(n, 32);
  return b <= 2 ? b : 4;
}
bool small_wgrad_supported(const ConvGeom& g) {
  // accumulators of a wave: 16 registers per (row block, column block)
  return small_conv_supported(g) && padded_blocks(g.Cp) * padded_blocks((int64_t)g.Cg * g.K) <= 8;
}

// Four waves per workgroup (they share a window) unless that leaves CUs without one; then a wave
// each (64 x 128 pixels, one picture: 256 workgroups instead of 64).
static SmallTiling small_tiling(const ConvGeom& g) {
  const int OH = g.M / g.OW;
  SmallTiling t;
  t.waves = ceil_div(g.OW, kSmPix) * (int64_t)OH * g.B >= 4 * 256 ? 4 : 1;
  t.stacked = OH >= t.waves;
  t.nx = (int)ceil_div(g.OW, t.stacked ? kSmPix : kSmPix * t.waves);
  t.ny = t.stacked ? (int)ceil_div(OH, t.waves) : OH;
  t.batches = (int)g.B;
  t.workgroups = t.nx * t.ny;
  return t;
}

// Runs CALL with CGv, NGv, NBv bound to channels of a window element, sample groups per lane half
// and 32-row blocks of pixel-side channels.
#define SDK_SMALL_DISPATCH(CALL)                                                             \
  do {                                                                                       \
    if (g.K <= 2 * kSmGroup) {                                                               \
      constexpr int NGv = 1;                                                                 \
      if (g.Cp <= 32) {                                                                      \
        constexpr int NBv = 1;                                                               \
        if (g.Cg <= 1) { constexpr int CGv = 1; CALL; }                                      \
        else if (g.Cg == 2) { constexpr int CGv = 2; CALL; }                                 \
        else if (g.Cg == 3) { constexpr int CGv = 3; CALL; }                                 \
        else { constexpr int CGv = 4; CALL; }                                                \
      } else {                                                                               \
        constexpr int NBv = 2;                                                               \
        if (g.Cg <= 1) { constexpr int CGv = 1; CALL; }                                      \
        else if (g.Cg == 2) { constexpr int CGv = 2; CALL; }                                 \
        else if (g.Cg == 3) { constexpr int CGv = 3; CALL; }                                 \
        else { constexpr int CGv = 4; CALL; }                                                \
      }                                                                                      \
    } else {                                                                                 \
      constexpr int NGv = 3, NBv = 1;                                                        \
      if (g.Cg <= 1) { constexpr int CGv = 1; CALL; }                                        \
      else { constexpr int CGv = 4; CALL; }                                                  \
    }                                                                                        \
  } while (0)

static size_t small_window_floats(int CG) { return CG == 1 ? kSmWindow + 4 : (kSmWindow + 1) * 4; }

static int small_pixel_forward(const ConvGeom& g, const float* img, const float* map,
                               const float* wts, const float* Wm, const float* bias, float* pix,
                               hipStream_t stream) {
  // few pixels: small workgroups, so that they spread over the CUs
  const int threads = (int64_t)g.M * g.B < 256 * 256 ? 64 : kSmThreads;
  const dim3 grid((unsigned)ceil_div(g.M, threads), (unsigned)g.B);
#define SF(CGv, KMv)                                                                            \
  SDK_DISPATCH_INTERP(g.interp, g.P,                                                            \
                      (launch_lds((small_pixel_forward_kernel<INTERP, WEIGHTED, CGv, KMv>),           \
                                          grid, dim3(threads),                                  \
                                          sizeof(float) * (size_t)g.Cp * CGv * KMv, stream, img, map, wts, Wm, \
                                          bias, pix, g.Cg, g.H, g.W, g.Cp, g.M, g.K, g.P)))
  if (g.K <= 9) {
    if (g.Cg <= 1) SF(1, 9); else if (g.Cg <= 3) SF(3, 9); else SF(4, 9);
  } else {
    if (g.Cg <= 1) SF(1, 25); else if (g.Cg <= 3) SF(3, 25); else SF(4, 25);
  }
#undef SF
  SDK_LAUNCH_CHECK("small_forward");
  return SDK_OK;
}

int small_forward(const ConvGeom& g, const float* img, const float* map, const float* wts,
                  const float* Wm, const float* bias, float* pix, hipStream_t stream) {
  // The matrix unit multiplies 32 output rows whatever Cp is, and a wave's window takes its setup;
  // the vector unit does Cg * K multiply-adds per output.  K = 9, bilinear, 4 x 256 x 512: 3 -> 16
  // channels 28 us per pixel against 30, 3 -> 32 43 against 32, 1 -> 32 21 against 23, 4 -> 48 62
  // against 57.
  // (A workgroup of the matrix kernel stores through one descriptor: 64 rows of the output have to
  // lie within its 31-bit byte offsets.  Larger pictures take the kernel that addresses flatly.)
  constexpr int kDescriptorPixels = 1 << 22;
  if (g.Cg == 1 || g.Cp <= 16 || g.M > kDescriptorPixels)
    return small_pixel_forward(g, img, map, wts, Wm, bias, pix, stream);
  SmallTiling tl = small_tiling(g);
  const int64_t tiles = (int64_t)tl.nx * tl.ny;
  SDK_SMALL_DISPATCH({
    // a workgroup keeps its taps for as many batch elements as leave eight workgroups per CU
    tl.batches = (int)ceil_div(g.B, std::min<int64_t>(g.B, ceil_div(2048, tiles)));
    const int64_t parts = ceil_div(g.B, tl.batches);
    const dim3 grid((unsigned)tiles, (unsigned)parts, (unsigned)ceil_div(g.Cp, 32 * NBv));
    const size_t smem = sizeof(float) * (small_window_floats(CGv) +
                                         (size_t)NGv * kSmGroup * CGv * 64 * NBv + 32 * NBv + 16);
    SDK_DISPATCH_INTERP(g.interp, g.P,
                        (launch_lds((small_forward_kernel<INTERP, WEIGHTED, CGv, NGv, NBv>), grid,
                                    dim3(64 * tl.waves), smem, stream, img, map, wts, Wm, bias, pix,
                                    g.Cg, g.H, g.W, g.Cp, g.M, g.OW, g.K, g.P, (int)g.B, tl)));
  });
  SDK_LAUNCH_CHECK("small_forward");
  return SDK_OK;
}

int small_scatter(const ConvGeom& g, const float* pix, const float* map, const float* wts,
                  const float* Wm, float* img, hipStream_t stream) {
  const int threads = (int64_t)g.M * g.B < 256 * 256 ? 64 : kSmThreads;
  const dim3 grid((unsigned)ceil_div(g.M, threads), (unsigned)g.B);
#define SS(CGv, KMv)                                                                            \
  SDK_DISPATCH_INTERP(g.interp, g.P,                                                            \
                      (launch_lds((small_scatter_kernel<INTERP, WEIGHTED, CGv, KMv>),           \
                                          grid, dim3(threads),                                  \
                                          sizeof(float) * (size_t)g.Cp * CGv * KMv, stream, pix, map, wts, Wm, \
                                          img, g.Cg, g.H, g.W, g.Cp, g.M, g.K, g.P)))
  if (g.K <= 9) {
    if (g.Cg <= 1) SS(1, 9); else if (g.Cg <= 3) SS(3, 9); else SS(4, 9);
  } else {
    if (g.Cg <= 1) SS(1, 25); else if (g.Cg <= 3) SS(3, 25); else SS(4, 25);
  }
#undef SS
  SDK_LAUNCH_CHECK("small_scatter");
  return SDK_OK;
}

int small_wgrad(const ConvGeom& g, const float* pix, const float* map, const float* wts,
                const float* img, float* gW, hipStream_t stream, float* gbias) {
  SmallTiling tl = small_tiling(g);
  const int64_t tiles = (int64_t)tl.nx * tl.ny;
  SDK_SMALL_DISPATCH({
    constexpr int CB = small_columns(NGv, CGv);
    // Every workgroup ends with one atomic per element of gW, all onto the same few lines, about
    // 0.05 us per workgroup; a tile takes some 10 us of it.  Both meet near 8 sqrt(tiles): 3 -> 32,
    // K = 9, bilinear, 1 x 176 x 350 (484 tiles): 24 us with 192 workgroups, 28 with 484; 4 x 256 x 512
    // (4096) 51 with 384, 59 with 256, 57 with 768.  At most what is resident at a time.
    const int64_t want = std::min<int64_t>(
        768, std::max<int64_t>(64, (int64_t)(8.0 * std::sqrt((double)(tiles * g.B)))));
    const int64_t gx = std::min(tiles, want);
    tl.workgroups = (int)gx;
    tl.batches = (int)ceil_div(g.B, std::min<int64_t>(g.B, std::max<int64_t>(1, want / gx)));
    const int64_t parts = ceil_div(g.B, tl.batches);
    const dim3 grid((unsigned)gx, (unsigned)parts, (unsigned)ceil_div(g.Cp, 32 * NBv));
    const size_t floats = std::max(
        small_window_floats(CGv) + (size_t)tl.waves * 32 * CB * kSmLd + 16,
        (size_t)32 * NBv * 32 * CB);
    SDK_DISPATCH_INTERP(g.interp, g.P,
                        (launch_lds((small_wgrad_kernel<INTERP, WEIGHTED, CGv, NGv, NBv>), grid,
                                    dim3(64 * tl.waves), sizeof(float) * floats, stream, pix, img,
                                    map, wts, gW, gbias, g.Cg, g.H, g.W, g.Cp, g.M, g.OW, g.K, g.P,
                                    (int)g.B, tl)));
  });
  SDK_LAUNCH_CHECK("small_wgrad");
  return SDK_OK;
}

}  // namespace sdk
