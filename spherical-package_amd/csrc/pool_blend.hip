// Mapped max / average pooling of float32 maps whose samples are blended from four pixels
// (bilinear, bispherical; ext_modules/include/common/mapped_max_pool.h:13-57, :81-133,
// common/mapped_avg_pool.h:13-40, :70-105 over core/interpolation.h).
//
// The per-pixel kernels read K * 4 taps per pooled pixel and plane from global memory, one
// float per lane: bound by the address rate of the vector memory path (36 reads a result; 48 x 4
// planes of 190 x 378 on a 95 x 189 grid 81 us, 13 MB written).  Here a workgroup owns a tile of
// the pooled grid, R rows x P columns, and a range of planes, one thread per pooled pixel.
// The taps are resolved once: four 16-bit positions inside the box of the image they fall into,
// whose columns may run over the seam, and four weights per sample, in registers.
// Per pass the box of four planes goes to LDS interleaved, [element][plane], so that one
// 16-byte LDS read serves a tap of four planes; the next pass's first groups are read while this
// one is blended.  A box too large for four planes (at a pole it is as wide as the image) takes two or
// one per pass, past that its taps come from global memory (blend_apart); the choice is made per workgroup.
// Results are the per-pixel kernels' bit for bit: the same products, summed in the same order.
// (Measured, us, average / maximum, per-pixel kernels or whole rows of the image in LDS -> so: 4 x 48 planes of
// 190 x 378, stride 2, 51 / 54 -> 31 / 33; 8 x 64 of 256 x 512, stride 2, 120 / 132 -> 96 / 108; 4 x 32 of
// 512 x 1024, stride 2, 338 / 362 -> 116 / 133; 2 x 16 of 512 x 1024, stride 1, 170 / 200 -> 86 / 94; 64 of 24 x 48,
// stride 2, 18 -> 9.5.  Whole rows with the reads ahead,
// three workgroups a CU: 33, 104, 123 with one of 512 pixels, 134.  What bounds it: the wait for the next box where
// images are large, the taps of a tile, worked out twice, where planes are few.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>

#include "pool_band.hpp"
#include "sdk_host.hpp"
#include "sdk_taps.hpp"

namespace sdk {
namespace {

constexpr int kBlendThreads = 256;   // most pooled pixels of a tile
constexpr int kBlendColumns = 128;   // ... and of a row of it, where a pooled row has more than 256

template <bool AVG, int K>
struct BlendOp {
  float acc = AVG ? 0.0f : -FLT_MAX;
  int best = -1;
  __device__ __forceinline__ void take(float v, int k) {
    if constexpr (AVG) {
      acc += v;
    } else if (v > acc) {   // strict: the first maximum wins, NaN never wins
      acc = v;
      best = k;
    }
  }
  __device__ __forceinline__ void store(float* __restrict__ out, int64_t* __restrict__ idx,
                                        size_t o, int pix) const {
    __builtin_nontemporal_store(AVG ? acc / float(K) : acc, out + o);
    if constexpr (!AVG)
      __builtin_nontemporal_store(best < 0 ? (int64_t)-1 : (int64_t)(((size_t)pix * K + best) * 2),
                                  idx + o);
  }
};

typedef float vec4 __attribute__((ext_vector_type(4)));

// The part of the image a tile's taps fall into: `rows` rows of `cols` columns, from c0 on and, past
// the last column of the image, from its first on.  A row is read in groups of four neighbours (16 bytes
// from any element boundary) of the columns before the seam (at least four) and of those behind it (none or at
// least four); the last group of either overlaps the one before it.
struct BlendBox {
  int row0, rows, c0, cols;
  int before, groups_before, groups;   // columns and groups of a row before the seam, groups of a row
  __device__ __forceinline__ void set(int r0, int r1, int first, int n, int W) {
    row0 = r0;
    rows = r1 - r0 + 1;
    n = max(n, 8);
    if (n + 8 > W) {
      c0 = 0;
      cols = before = W;
    } else {
      c0 = first;
      before = min(n, W - c0);
      int behind = n - before;
      if (before < 4) {   // (first > W - 4)
        c0 -= 4 - before;
        before = 4;
      }
      if (behind > 0) behind = max(behind, 4);
      cols = before + behind;
    }
    groups_before = (before + 3) >> 2;
    groups = groups_before + ((cols - before + 3) >> 2);
  }
  // group i: where it lies in LDS and, in bytes from row0's first column, in the image
  __device__ __forceinline__ void group(int i, int W, unsigned& to, unsigned& from) const {
    const int row = i / groups, q = i - row * groups;
    const bool first = q < groups_before;
    const int at = first ? min(4 * q, before - 4) : min(4 * (q - groups_before), cols - before - 4);
    to = (unsigned)(row * cols + (first ? at : before + at));
    from = 4u * (unsigned)(row * W + (first ? c0 + at : at));
  }
};

// Planes past the range repeat the last.
template <int PG>
__device__ __forceinline__ void read_group(vec4 (&v)[PG], const float* __restrict__ in, int p,
                                           int p_end, size_t HW, unsigned from) {
#pragma unroll
  for (int g = 0; g < PG; ++g)
    __builtin_memcpy(&v[g], reinterpret_cast<const char*>(in + (size_t)min(p + g, p_end - 1) * HW) + from,
                     sizeof(vec4));
}
template <int PG, typename V>
__device__ __forceinline__ void place_group(V* box, const vec4 (&v)[PG], unsigned to) {
#pragma unroll
  for (int x = 0; x < 4; ++x) {
    V y;
#pragma unroll
    for (int g = 0; g < PG; ++g) y[g] = v[g][x];
    box[to + x] = y;
  }
}

// The first groups of a pass that a thread holds in registers: of the next pass while it blends.
// (Two: 4 x 64 results of stride 2 have 1.5 of them.)
constexpr int kBlendHeld = 2;

// pos[k][0] = positions of taps 0 (low half) and 1, pos[k][1] = of taps 2 and 3; the position
// behind the box is the zero element inactive taps read.
template <bool AVG, int K, int PG, typename Taps>
__device__ __forceinline__ void run_blend(const float* __restrict__ in, float* __restrict__ out,
                                          int64_t* __restrict__ idx, float* lds, Taps&& taps,
                                          int pix, bool on, int p_begin, int p_end, size_t HW,
                                          int W, int M, const BlendBox& b) {
  typedef float vecp __attribute__((ext_vector_type(PG)));
  vecp* box = reinterpret_cast<vecp*>(lds);
  const int t = threadIdx.x, nt = blockDim.x, total = b.rows * b.groups;
  in += (size_t)b.row0 * W;
  vec4 held[kBlendHeld][PG];
  unsigned to[kBlendHeld], from[kBlendHeld];
#pragma unroll
  for (int i = 0; i < kBlendHeld; ++i) b.group(min(t + i * nt, total - 1), W, to[i], from[i]);
  auto read_held = [&](int p) {
#pragma unroll
    for (int i = 0; i < kBlendHeld; ++i)
      if (t + i * nt < total) read_group(held[i], in, p, p_end, HW, from[i]);
  };
  read_held(p_begin);
  unsigned pos[K][2];
  float w[K][4];
  taps(pos, w);   // (worked out while the first planes are on their way)
  if (t == 0) box[b.rows * b.cols] = vecp(0.0f);
  for (int p = p_begin; p < p_end; p += PG) {
#pragma unroll
    for (int i = 0; i < kBlendHeld; ++i)
      if (t + i * nt < total) place_group(box, held[i], to[i]);
    constexpr int kMore = PG == 4 ? 2 : 4;
    for (int i0 = t + kBlendHeld * nt; i0 < total; i0 += kMore * nt) {
      vec4 v[kMore][PG];
      unsigned at[kMore];
#pragma unroll
      for (int i = 0; i < kMore; ++i) {
        unsigned from_i;
        b.group(min(i0 + i * nt, total - 1), W, at[i], from_i);
        read_group(v[i], in, p, p_end, HW, from_i);
      }
#pragma unroll
      for (int i = 0; i < kMore; ++i)
        if (i0 + i * nt < total) place_group(box, v[i], at[i]);
    }
    __syncthreads();
    if (p + PG < p_end) read_held(p + PG);
    __builtin_amdgcn_sched_barrier(0);
    if (on) {
      BlendOp<AVG, K> op[PG];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        // (opaque to the compiler, which otherwise unpacks all positions ahead of the loop over
        // the planes, into registers that are not there)
        unsigned p01 = pos[k][0], p23 = pos[k][1];
        asm volatile("" : "+v"(p01), "+v"(p23));
        const vecp v0 = box[p01 & 0xffffu], v1 = box[p01 >> 16];
        const vecp v2 = box[p23 & 0xffffu], v3 = box[p23 >> 16];
        const vecp v = w[k][0] * v0 + w[k][1] * v1 + w[k][2] * v2 + w[k][3] * v3;
#pragma unroll
        for (int g = 0; g < PG; ++g) op[g].take(v[g], k);
        // (done before the next: else what a plane takes is moved into its store's branch, and all 36
        // reads wait for it in 144 registers)
#pragma unroll
        for (int g = 0; g < PG; ++g) asm volatile("" : "+v"(op[g].acc));
      }
#pragma unroll
      for (int g = 0; g < PG; ++g)
        if (p + g < p_end) op[g].store(out, idx, (size_t)(p + g) * M + pix, pix);
    }
    __syncthreads();
  }
}

// A pooled pixel whose taps come from global memory, PC planes side by side, S samples of them in flight: a tap's
// two neighbours of a row in one read.  Bound by the lines that the caches hold: planes that are no larger than
// kBlendNear go four at a time, others alone.  (Uniformly random samples, average, us, an element a read and one
// plane / four planes at a time -> pairs, one / two / four planes: 64 planes of 128 x 256, stride 2, 53 / 44 -> 46 /
// 42 / 43; 4 x 48 of 190 x 378 370 / 300 -> 301 / 275 / 282; 8 x 64 of 256 x 512 1496 / 2207 -> 1473 / 2146 / 2248;
// 64 of 300 x 600 600 / 459 -> 308 / 363 / 474; 128 of 512 x 1024 4498 / 4416 -> 3796 / 4563 / 4570.)
constexpr size_t kBlendNear = 384 * 1024;
template <bool AVG, int INTERP, int K, int PC, int S>
__device__ __forceinline__ void blend_apart(const float* __restrict__ in, const float* __restrict__ map,
                                            float* __restrict__ out, int64_t* __restrict__ idx, int pix,
                                            int p_begin, int p_end, int H, int W, int M) {
  const float* coords = map + (size_t)pix * K * 2;
  for (int p = p_begin; p < p_end; p += PC) {
    const int np = min(PC, p_end - p);
    const float* base = in + (size_t)p * H * W;
    BlendOp<AVG, K> op[PC];
#pragma unroll S
    for (int k = 0; k < K; ++k) {
      float v[PC];
      if (W >= 2) gather_pairs<float, INTERP, PC>(base, (size_t)H * W, np, coords[2 * k], coords[2 * k + 1], H, W, v);
      else gather_sample<float, INTERP, false, PC>(base, (size_t)H * W, np, coords + 2 * k, nullptr, 0, H, W, v);
#pragma unroll
      for (int g = 0; g < PC; ++g) op[g].take(v[g], k);
    }
#pragma unroll
    for (int g = 0; g < PC; ++g)
      if (g < np) op[g].store(out, idx, (size_t)(p + g) * M + pix, pix);
  }
}

// An XCD takes an eighth of the tiles of all plane chunks in turn, so whole chunks or parts of one:
// the image elements neighbouring tiles share are read through one L2.  Tile rows from both poles
// towards the equator: the widest boxes first.
template <bool AVG, int INTERP, int K>
__global__ __launch_bounds__(kBlendThreads, 3) void pool_blend_kernel(
    const float* __restrict__ in, const float* __restrict__ map, float* __restrict__ out,
    int64_t* __restrict__ idx, int planes, int H, int W, int OH, int OW, int R, int P, int tiles_x,
    int tiles_y, int chunks, int lds_floats) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ int s_rows[2], s_cols[2], s_middle;
  const int t = threadIdx.x, M = OH * OW, tiles = tiles_x * tiles_y;
  const int unit = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  const int tile = unit % tiles, chunk = unit / tiles;
  if (chunk >= chunks) return;
  const int p_begin = (int)((int64_t)chunk * planes / chunks);
  const int p_end = (int)((int64_t)(chunk + 1) * planes / chunks);
  const int nth = tile / tiles_x, row = nth & 1 ? tiles_y - 1 - nth / 2 : nth / 2;
  const int oy = row * R + t / P, ox = (tile - nth * tiles_x) * P + t % P;
  const bool on = t < R * P && oy < OH && ox < OW;
  const int pix = min(oy, OH - 1) * OW + min(ox, OW - 1);
  const size_t HW = (size_t)H * W;
  const float2* coords = reinterpret_cast<const float2*>(map) + (size_t)pix * K;
  float2 at[K];   // (requested together: one at a time their way from memory is most of a small call)
#pragma unroll
  for (int k = 0; k < K; ++k) at[k] = coords[k];
  if (t == 0) {
    s_rows[0] = s_cols[0] = INT_MAX;
    s_rows[1] = s_cols[1] = -1;
    s_middle = (int)fminf(fmaxf(at[K / 2].x, 0.0f), (float)(W - 1));
  }
  __syncthreads();
  // columns are counted from half the image's width before the first pixel's
  int start = s_middle - W / 2;
  start += start < 0 ? W : 0;
  int rmin = INT_MAX, rmax = -1, cmin = INT_MAX, cmax = -1;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    PointTaps<float, INTERP> tp;
    tp.set(at[k].x, at[k].y, H, W);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (on && tp.off[i] >= 0) {
        const int c = tp.tx[i] - start + (tp.tx[i] < start ? W : 0);
        rmin = min(rmin, tp.ty[i]);
        rmax = max(rmax, tp.ty[i]);
        cmin = min(cmin, c);
        cmax = max(cmax, c);
      }
    __builtin_amdgcn_sched_barrier(0);
  }
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    rmin = min(rmin, __shfl_xor(rmin, d));
    rmax = max(rmax, __shfl_xor(rmax, d));
    cmin = min(cmin, __shfl_xor(cmin, d));
    cmax = max(cmax, __shfl_xor(cmax, d));
  }
  if ((t & 63) == 0 && rmax >= 0) {
    atomicMin(&s_rows[0], rmin);
    atomicMax(&s_rows[1], rmax);
    atomicMin(&s_cols[0], cmin);
    atomicMax(&s_cols[1], cmax);
  }
  __syncthreads();
  const bool none = s_rows[1] < 0;
  int first = none ? 0 : start + s_cols[0];
  first -= first >= W ? W : 0;
  BlendBox b;
  b.set(none ? 0 : s_rows[0], none ? 0 : s_rows[1], first, none ? 1 : s_cols[1] - s_cols[0] + 1, W);
  const int64_t elems = (int64_t)b.rows * b.cols;
  if (W >= 4 && elems < 65536 && elems + 1 <= lds_floats) {
    const int n = (int)elems;
    // (the taps worked out a second time, from coordinates that the compiler takes for others: kept from
    // the first they would not fit the registers)
    auto taps = [&](unsigned (&pos)[K][2], float (&w)[K][4]) {
#pragma unroll
      for (int k = 0; k < K; ++k) {
        PointTaps<float, INTERP> tp;
        asm volatile("" : "+v"(at[k].x), "+v"(at[k].y));
        tp.set(at[k].x, at[k].y, H, W);
        unsigned q[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int c = tp.tx[i] - b.c0 + (tp.tx[i] < b.c0 ? W : 0);
          q[i] = (unsigned)(tp.off[i] < 0 || !on ? n : (tp.ty[i] - b.row0) * b.cols + c);
          w[k][i] = tp.w[i];
        }
        pos[k][0] = q[0] | (q[1] << 16);
        pos[k][1] = q[2] | (q[3] << 16);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    if ((elems + 1) * 4 <= lds_floats)
      run_blend<AVG, K, 4>(in, out, idx, lds, taps, pix, on, p_begin, p_end, HW, W, M, b);
    else if ((elems + 1) * 2 <= lds_floats)
      run_blend<AVG, K, 2>(in, out, idx, lds, taps, pix, on, p_begin, p_end, HW, W, M, b);
    else
      run_blend<AVG, K, 1>(in, out, idx, lds, taps, pix, on, p_begin, p_end, HW, W, M, b);
  } else if (on) {
    if (HW * sizeof(float) <= kBlendNear)
      blend_apart<AVG, INTERP, K, 4, 1>(in, map, out, idx, pix, p_begin, p_end, H, W, M);
    else blend_apart<AVG, INTERP, K, 1, 3>(in, map, out, idx, pix, p_begin, p_end, H, W, M);
  }
}

constexpr int kBlendLdsBytes = 52 * 1024;

}  // namespace

bool pool_blend_launch(bool avg, const float* in, const float* map, float* out, int64_t* idx,
                       int64_t planes, int H, int W, int OH, int OW, int K, int interp,
                       hipStream_t stream) {
  if ((K != 4 && K != 9) || (interp != 1 && interp != 2)) return false;
  const int64_t pixels = (int64_t)OH * OW;
  if (pixels >= ((int64_t)1 << 30) || W >= kBlendLdsBytes / 4) return false;
  // Tiles of up to 256 pooled pixels: whole rows where they are no longer than that, else equal shares of up to
  // 128.  (us with 64, 128, 256 columns: 8 x 64 planes of 256 x 512, stride 2, 124, 114, 96; 4 x 48 of 190 x 378 37,
  // 35, 30; rows of 512: 4 x 32 of 512 x 1024 150, 117, 160; of 601, stride 1, 32 planes 44, 34, 50: low tiles have a
  // smaller box at the poles, square ones elsewhere.)
  const int P = OW <= kBlendThreads ? OW : (int)ceil_div(OW, ceil_div(OW, kBlendColumns));
  const int R = std::min(OH, kBlendThreads / P);
  const int tiles_x = (int)ceil_div(OW, P), tiles_y = (int)ceil_div(OH, R);
  const int threads = (int)(ceil_div((int64_t)R * P, 64) * 64);
  // Plane chunks: what a workgroup takes for the taps it resolves anew (about two passes of four
  // planes) and its passes, times the rounds of workgroups (three a CU by their LDS), at its least;
  // at least four planes each.
  const int64_t at_once = 768, tiles = (int64_t)tiles_x * tiles_y;
  int chunks = 1;
  int64_t least = INT64_MAX;
  for (int c = 1; c <= std::max<int64_t>(1, planes / 4) && c * tiles <= 8 * at_once; ++c) {
    const int64_t cost = ceil_div(c * tiles, at_once) * (ceil_div(ceil_div(planes, c), 4) + 2);
    if (cost < least) {
      least = cost;
      chunks = c;
    }
  }
  const unsigned grid = 8u * (unsigned)ceil_div(tiles * chunks, 8);
#define PB(AVGv, Iv, Kv)                                                                       \
  pool_blend_kernel<AVGv, Iv, Kv><<<dim3(grid), dim3(threads), kBlendLdsBytes, stream>>>(      \
      in, map, out, idx, (int)planes, H, W, OH, OW, R, P, tiles_x, tiles_y, chunks, kBlendLdsBytes / 4)
#define PBI(AVGv, Kv)                                       \
  do {                                                      \
    if (interp == 1) PB(AVGv, 1, Kv); else PB(AVGv, 2, Kv); \
  } while (0)
  if (K == 9) {
    if (avg) PBI(true, 9); else PBI(false, 9);
  } else {
    if (avg) PBI(true, 4); else PBI(false, 4);
  }
#undef PBI
#undef PB
  return true;
}

}  // namespace sdk
