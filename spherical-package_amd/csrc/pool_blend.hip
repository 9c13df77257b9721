// Mapped max / average pooling of float32 maps whose samples are blended from four pixels
// (bilinear, bispherical; ext_modules/include/common/mapped_max_pool.h:13-57, :81-133,
// common/mapped_avg_pool.h:13-40, :70-105 over core/interpolation.h).
//
// The per-pixel kernels read K * 4 taps per pooled pixel and plane from global memory, one
// float per lane: bound by the address rate of the vector memory path (36 reads a result; 48 x 4
// planes of 190 x 378 on a 95 x 189 grid 81 us, 13 MB written).  Here a workgroup owns R whole
// rows of the pooled grid and a range of planes, one thread per pooled pixel.  The taps are
// resolved once: four 16-bit positions inside the band of image rows they fall into (a few
// whole rows whatever the longitude, pool_band.hip) and four weights per sample, in registers.
// Per pass the band rows of four planes go to LDS interleaved, [element][plane], so that one
// 16-byte LDS read serves a tap of four planes.  A band too tall for four planes takes two or
// one per pass, past that its taps come from global memory; the choice is made per workgroup.
// Results are the per-pixel kernels' bit for bit: the same products, summed in the same order.
// (Measured, average / maximum: 4 x 48 planes of 190 x 378, stride 2, 80 -> 52 / 82 -> 55 us (58 / 61
// with the band read an element at a time);
// 8 x 64 planes of 256 x 512, stride 2, 335 -> 126 / 360 -> 141 us.  Two workgroups per CU of 256
// registers: at three the nine samples' positions and weights spill, 69 us.)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cfloat>
#include <climits>

#include "pool_band.hpp"
#include "sdk_host.hpp"
#include "sdk_taps.hpp"

namespace sdk {
namespace {

constexpr int kBlendThreads = 256;   // most pooled pixels of a band

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

// pos[k][0] = positions of taps 0 (low half) and 1, pos[k][1] = of taps 2 and 3; position
// band_elems is the zero element inactive taps read.
template <bool AVG, int K, int PG>
__device__ __forceinline__ void run_blend(const float* __restrict__ in, float* __restrict__ out,
                                          int64_t* __restrict__ idx, float* lds,
                                          const unsigned (&pos)[K][2], const float (&w)[K][4],
                                          int pix, bool on, int p_begin, int p_end, size_t HW,
                                          int M, int row_start, int band_elems) {
  typedef float vecp __attribute__((ext_vector_type(PG)));
  vecp* band = reinterpret_cast<vecp*>(lds);
  const int t = threadIdx.x, nt = blockDim.x;
  if (t == 0) band[band_elems] = vecp(0.0f);
  for (int p = p_begin; p < p_end; p += PG) {
    const float* src = in + (size_t)p * HW + row_start;
    // The band is one run of memory: four neighbours of PG planes a read (16 bytes from any element
    // boundary), AHEAD such groups in flight per thread; planes past the range repeat the last, the
    // last groups overlap (and store the same values).
    typedef float vec4 __attribute__((ext_vector_type(4)));
    constexpr int AHEAD = 2;
    if (band_elems >= 4) {
      for (int e0 = 4 * t; e0 < band_elems; e0 += AHEAD * 4 * nt) {
        vec4 v[AHEAD][PG];
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          const int e = min(e0 + i * 4 * nt, band_elems - 4);
#pragma unroll
          for (int g = 0; g < PG; ++g)
            __builtin_memcpy(&v[i][g], src + (size_t)min(g, p_end - 1 - p) * HW + e, sizeof(vec4));
        }
#pragma unroll
        for (int i = 0; i < AHEAD; ++i) {
          if (i > 0 && e0 + i * 4 * nt >= band_elems) break;
          const int e = min(e0 + i * 4 * nt, band_elems - 4);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            vecp y;
#pragma unroll
            for (int g = 0; g < PG; ++g) y[g] = v[i][g][x];
            band[e + x] = y;
          }
        }
      }
    } else {
      for (int e = t; e < band_elems; e += nt) {
        vecp y;
#pragma unroll
        for (int g = 0; g < PG; ++g) y[g] = src[(size_t)min(g, p_end - 1 - p) * HW + e];
        band[e] = y;
      }
    }
    __syncthreads();
    if (on) {
      BlendOp<AVG, K> op[PG];
#pragma unroll
      for (int k = 0; k < K; ++k) {
        // (opaque to the compiler, which otherwise unpacks all positions ahead of the loop over
        // the planes, into registers that are not there)
        unsigned p01 = pos[k][0], p23 = pos[k][1];
        asm volatile("" : "+v"(p01), "+v"(p23));
        const vecp v0 = band[p01 & 0xffffu], v1 = band[p01 >> 16];
        const vecp v2 = band[p23 & 0xffffu], v3 = band[p23 >> 16];
        const vecp v = w[k][0] * v0 + w[k][1] * v1 + w[k][2] * v2 + w[k][3] * v3;
#pragma unroll
        for (int g = 0; g < PG; ++g) op[g].take(v[g], k);
        if (k % 3 == 2) __builtin_amdgcn_sched_barrier(0);   // (reads of three samples at a time)
      }
#pragma unroll
      for (int g = 0; g < PG; ++g)
        if (p + g < p_end) op[g].store(out, idx, (size_t)(p + g) * M + pix, pix);
    }
    __syncthreads();
  }
}

// grid.x = 8 * nbands * ceil(chunks / 8), as in pool_band.hip: an XCD takes whole plane chunks,
// so that the rows neighbouring bands share are read through one L2.
template <bool AVG, int INTERP, int K>
__global__ __launch_bounds__(kBlendThreads, 2) void pool_blend_kernel(
    const float* __restrict__ in, const float* __restrict__ map, float* __restrict__ out,
    int64_t* __restrict__ idx, int planes, int H, int W, int OW, int M, int R, int nbands,
    int chunks, int lds_floats) {
  extern __shared__ __attribute__((aligned(16))) float lds[];
  __shared__ int s_rows[2];
  const int t = threadIdx.x;
  const int xcd = blockIdx.x & 7, within = blockIdx.x >> 3;
  const int band = within % nbands;
  const int chunk = (within / nbands) * 8 + xcd;
  if (chunk >= chunks) return;
  const int p_begin = (int)((int64_t)chunk * planes / chunks);
  const int p_end = (int)((int64_t)(chunk + 1) * planes / chunks);
  const int pix0 = band * R * OW;
  const int npix = min(R * OW, M - pix0);
  const bool on = t < npix;
  const int pix = pix0 + min(t, npix - 1);
  const size_t HW = (size_t)H * W;
  if (t == 0) {
    s_rows[0] = INT_MAX;
    s_rows[1] = -1;
  }
  __syncthreads();
  const float2* coords = reinterpret_cast<const float2*>(map) + (size_t)pix * K;
  int rmin = INT_MAX, rmax = -1;
#pragma unroll 1
  for (int k = 0; k < K; ++k) {
    PointTaps<float, INTERP> tp;
    tp.set(coords[k].x, coords[k].y, H, W);
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (tp.off[i] >= 0) {
        rmin = min(rmin, tp.ty[i]);
        rmax = max(rmax, tp.ty[i]);
      }
  }
  if (rmax >= 0) {
    atomicMin(&s_rows[0], rmin);
    atomicMax(&s_rows[1], rmax);
  }
  __syncthreads();
  const int row0 = s_rows[0], row1 = s_rows[1];
  const int64_t elems = row1 < 0 ? 0 : (int64_t)(row1 - row0 + 1) * W;
  const int row_start = row1 < 0 ? 0 : row0 * W;
  if (elems < 65536 && elems + 1 <= lds_floats) {
    const int n = (int)elems;
    // (the taps worked out a second time: kept from the first they would not fit the registers)
    unsigned pos[K][2];
    float w[K][4];
#pragma unroll
    for (int k = 0; k < K; ++k) {
      PointTaps<float, INTERP> tp;
      tp.set(coords[k].x, coords[k].y, H, W);
      unsigned q[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        q[i] = (unsigned)(tp.off[i] < 0 ? n : tp.off[i] - row_start);
        w[k][i] = tp.w[i];
      }
      pos[k][0] = q[0] | (q[1] << 16);
      pos[k][1] = q[2] | (q[3] << 16);
      __builtin_amdgcn_sched_barrier(0);
    }
    if ((elems + 1) * 4 <= lds_floats)
      run_blend<AVG, K, 4>(in, out, idx, lds, pos, w, pix, on, p_begin, p_end, HW, M, row_start, n);
    else if ((elems + 1) * 2 <= lds_floats)
      run_blend<AVG, K, 2>(in, out, idx, lds, pos, w, pix, on, p_begin, p_end, HW, M, row_start, n);
    else
      run_blend<AVG, K, 1>(in, out, idx, lds, pos, w, pix, on, p_begin, p_end, HW, M, row_start, n);
  } else if (on) {
    for (int p = p_begin; p < p_end; ++p) {
      BlendOp<AVG, K> op;
      for (int k = 0; k < K; ++k) {
        PointTaps<float, INTERP> tp;
        tp.set(coords[k].x, coords[k].y, H, W);
        op.take(tp.gather(in + (size_t)p * HW), k);
      }
      op.store(out, idx, (size_t)p * M + pix, pix);
    }
  }
}

constexpr int kBlendLdsBytes = 52 * 1024;
constexpr int64_t kBlendLeast = (int64_t)1 << 19;

}  // namespace

bool pool_blend_launch(bool avg, const float* in, const float* map, float* out, int64_t* idx,
                       int64_t planes, int H, int W, int OH, int OW, int K, int interp,
                       hipStream_t stream) {
  if ((K != 4 && K != 9) || (interp != 1 && interp != 2)) return false;
  // Below half a million results the launch is short either way and resolving the taps twice
  // does not pay (128 planes of 33 x 66, stride 1: 14 against 15 us).  A pooled row of more than
  // 256 pixels would stage its image rows once per piece (128 planes of 512 x 1024, stride 2: 339
  // per pixel against 357 us).
  if (OW > kBlendThreads || planes * OH * OW < kBlendLeast) return false;
  // rows of a band: at most 256 pooled pixels, as long as the image rows they are expected to
  // touch (R strides, a kernel's own height, one more for the blend) of four planes leave room
  // for three workgroups per CU
  const int sy = (int)ceil_div(H, OH);
  auto bytes = [&](int r) { return ((int64_t)(r * sy + 2 * sy + 2) * W + 1) * 16; };
  int R = 1;
  while (2 * R * OW <= kBlendThreads && 2 * R <= OH && bytes(2 * R) <= kBlendLdsBytes)
    R *= 2;
  const int64_t lds = std::min<int64_t>(bytes(R), kBlendLdsBytes);
  if ((int64_t)W + 1 > lds / 4) return false;
  const int nbands = (int)ceil_div(OH, R), M = OH * OW;
  const int threads = (int)(ceil_div((int64_t)R * OW, 64) * 64);
  // about four workgroups per CU, at least eight planes each (the taps are resolved anew in
  // every workgroup), chunks in eighths
  int chunks = (int)std::max<int64_t>(1, std::min<int64_t>(planes / 8, 1024 / nbands));
  chunks = std::max(8, chunks / 8 * 8);
  chunks = (int)std::min<int64_t>(chunks, planes);
  const unsigned grid = 8u * (unsigned)nbands * (unsigned)ceil_div(chunks, 8);
  const int floats = (int)(lds / 4);
#define PB(AVGv, Iv, Kv)                                                                        \
  pool_blend_kernel<AVGv, Iv, Kv><<<dim3(grid), dim3(threads), (size_t)lds, stream>>>(          \
      in, map, out, idx, (int)planes, H, W, OW, M, R, nbands, chunks, floats)
#define PBI(AVGv, Kv)                                   \
  do {                                                  \
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
