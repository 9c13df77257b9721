// Mapped convolution as columns and matrix products, for calls so small that the fused
// kernels cannot fill the GPU.
//
// The fused kernels (conv_window_gemm.hip, conv_window_wgrad.hip) own 128-pixel tiles and walk
// all samples and channels of a tile in one workgroup: at 6 x 25 x 50 output pixels that is a
// few dozen workgroups on 256 CUs, each a serial chain of hundreds of dependent LDS and memory
// steps, once per class of tiles.  The same work cut into an im2col, a matrix product and a
// col2im (the reference's own order, ext_modules/src/cpp/mapped_convolution_layer.cpp:8-60)
// has thousands of independent pieces per launch.  No tap plan is needed either: the map is read
// once per sample.
//
// Here: which calls take the route, the layout of its workspace, the col2im, and the products of
// columns that lie in memory: of samples of more than four points, and of wide layers of few columns.
// All others' columns exist only in
// LDS, or, a scatter's, as the products of a slice of the batch or of its channels that, where 32 channels
// of one element have no more, stays in the 256 MB memory-side cache until the col2im reads them
// (conv_columns_direct.hip).
// (Measured, on the fused kernels and so: 96 -> 160 channels, 6 x 50 x 100, stride 2, split,
// forward + backward 907 -> 122 us; 64 -> 64 channels on a map not seen before, 1 x 128 x 256,
// forward 368 -> 50 us, of which 265 were its plan.)
//
// Everything is channels-last and padded with zeros to a multiple of eight channels, so that
// every access of these kernels is an aligned 16-byte one:
//   rows   img[b][c][u] -> [b][u][c]            (channels_last_kernel)
//   col    [b][m][k][c], row length R = K * Cgp (columns_kernel)
//   W      [n][k][c] or [k][c][n]               (columns_weight_kernel)
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "conv_columns.hpp"
#include "conv_product.hpp"
#include "sdk_host.hpp"
#include "sdk_mfma.hpp"
#include "sdk_taps.hpp"

namespace sdk {
namespace {

constexpr int kClThreads = 256;
typedef float vec4 __attribute__((ext_vector_type(4)));

// dst[b][n][c] = src[b][c][n], c padded to Cp8 with zeros.  grid (tiles of 64 n, tiles of 32 c,
// batch): the tile goes through LDS, reads run along n, writes along c.
__global__ __launch_bounds__(kClThreads) void channels_last_kernel(
    const float* __restrict__ src, float* __restrict__ dst, int C, int Cp8, int N) {
  __shared__ float tile[32][65];
  const int n0 = blockIdx.x * 64, c0 = blockIdx.y * 32;
  channels_last_tile(src + (size_t)blockIdx.z * C * N, dst + (size_t)blockIdx.z * N * Cp8, C, Cp8, N, n0, c0, tile);
}

// REDUCTION_N = false: W[n][k][c]; true: W[k][c][n].  c and n padded to multiples of eight.
template <bool REDUCTION_N>
__global__ __launch_bounds__(kClThreads) void columns_weight_kernel(
    const float* __restrict__ Wm, float* __restrict__ dst, int Cg, int Cgp, int K, int Cp,
    int Cpp, int total) {
  const int e = blockIdx.x * kClThreads + threadIdx.x;
  if (e >= total) return;
  int n, k, c;
  if constexpr (REDUCTION_N) {
    n = e % Cpp;
    const int q = e / Cpp;
    c = q % Cgp;
    k = q / Cgp;
  } else {
    c = e % Cgp;
    const int q = e / Cgp;
    k = q % K;
    n = q / K;
  }
  dst[e] = (c < Cg && n < Cp) ? Wm[((size_t)n * Cg + c) * K + k] : 0.0f;
}

// col[b][m][k][:] = the blended image rows of sample (m, k).  A workgroup owns 64 consecutive
// samples of one batch element: their taps are worked out once into LDS (zero-weight and
// outside taps dropped), then a thread takes four channels of a sample.
// SLOTS: most taps of a sample the LDS lists hold (the points of a weighted sample times four).
constexpr int kClSamples = 64;
template <int INTERP, bool WEIGHTED, int SLOTS>
__global__ __launch_bounds__(kClThreads) void columns_kernel(
    const float* __restrict__ rows, const float* __restrict__ map, const float* __restrict__ wts,
    float* __restrict__ col, int samples, int P, int H, int W, int C4) {
  __shared__ int s_n[kClSamples];
  __shared__ int s_off[SLOTS][kClSamples];
  __shared__ float s_co[SLOTS][kClSamples];
  const int s0 = blockIdx.x * kClSamples;
  if (threadIdx.x < kClSamples) {
    const int s = s0 + threadIdx.x;
    int n = 0;
    if (s < samples) {
      PointTaps<float, INTERP> t;
      const int q = WEIGHTED ? P : 1;
      for (int p = 0; p < q; ++p) {
        const size_t at = (size_t)s * q + p;
        t.set(map[2 * at], map[2 * at + 1], H, W);
        const float wt = WEIGHTED ? wts[at] : 1.0f;
#pragma unroll
        for (int i = 0; i < PointTaps<float, INTERP>::N; ++i) {
          const float c = WEIGHTED ? t.w[i] * wt : t.w[i];
          if (t.off[i] >= 0 && c != 0.0f && n < SLOTS) {
            s_off[n][threadIdx.x] = t.off[i];
            s_co[n][threadIdx.x] = c;
            ++n;
          }
        }
      }
    }
    s_n[threadIdx.x] = n;
  }
  __syncthreads();
  const vec4* r = reinterpret_cast<const vec4*>(rows) + (size_t)blockIdx.y * H * W * C4;
  vec4* out = reinterpret_cast<vec4*>(col) + ((size_t)blockIdx.y * samples + s0) * C4;
  const int items = min(kClSamples, samples - s0) * C4;
  for (int it = threadIdx.x; it < items; it += kClThreads) {
    const int s = it / C4, c = it - s * C4;
    const int n = s_n[s];
    vec4 acc = {0.f, 0.f, 0.f, 0.f};
    for (int i0 = 0; i0 < n; i0 += 4) {
      vec4 v[4];
      float w[4];
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int j = min(i0 + i, n - 1);
        w[i] = s_co[j][s];
        v[i] = r[(size_t)s_off[j][s] * C4 + c];
      }
#pragma unroll
      for (int i = 0; i < 4; ++i)
        if (i0 + i < n) acc += w[i] * v[i];
    }
    out[it] = acc;
  }
}

// ---------------------------------------------------------------------------
// The products.  Four waves make a 64 x 64 tile of C, 32 x 32 each (KS = 2: two such groups
// share the reduction of one tile, alternate steps each, and add up at the end); the reduction
// goes through LDS in steps of 32, double-buffered, the values of the step after next requested
// from memory before the current step's MFMAs (a step is 0.1 to 0.4 us of matrix work, a read
// from beyond the L2 takes longer).  LDS rows hold 32 reduction elements and are 36 floats apart
// (16-byte reads of 32 consecutive rows then use all banks evenly); a lane reads eight
// consecutive reduction elements of its row, which are a bf16 operand once converted, or the
// operands of eight fp32 MFMAs (whose two reduction indices may be any pair, as long as both
// operands agree).
//   TN = false: C[i][n] = sum_r A[i][r] B[n][r] + bias[i]    (both operands run along r)
//   TN = true:  C[i][n] = sum_r A[r][i] B[r][n], r in the split's range (a thread transposes
//               4 x 4 blocks in registers on the way to LDS)
// Leading dimensions and the reduction length (TN: the rows' lengths) are multiples of eight.
// ---------------------------------------------------------------------------
constexpr int kGk = 32;
constexpr int kGld = 36;
// CONV: bf16 operands are formed on the way to LDS, once per workgroup: a wave that forms its own from
// float32 rows repeats what the neighbour of the same rows does, and six vector instructions an element
// weigh as much as the products.  A row then holds 64 bytes a piece (one, or the three of the split)
// and 16 of skew.  6 x 25 x 50 pixels, 96 -> 160, split, weight gradient 41.7 -> 39.0 us; 325 x 648, batch 2,
// 16 -> 29, bf16, map and forward 251 -> 232.  Split operands take three workgroups to a CU so instead of
// four: where the products are short (gemm below) and with two groups of waves they stay float32 rows.
constexpr int columns_row_bytes(int mm, bool conv) {
  return !conv ? kGld * 4 : (mm == kMmBf16 ? 64 : 192) + 16;
}
// A split of the weight gradient's reduction is hundreds of pixels; added up one after the other they
// lose twice the bits of the tile kernels' sums (6 x 25 x 50 pixels, 96 -> 160: 4.5e-7 of the float64
// norm against 2.1e-7), so two steps at a time are summed apart and then added: 1.7e-7, for 2 us of the
// layer's 174.

__device__ __forceinline__ void split_bf16x4(const vec4& f, uint2 (&piece)[3]) {
  unsigned u[3][4];
#pragma unroll
  for (int i = 0; i < 4; ++i) split_bf16(f[i], u[0][i], u[1][i], u[2][i]);
#pragma unroll
  for (int p = 0; p < 3; ++p)
    piece[p] = make_uint2((u[p][0] >> 16) | u[p][1], (u[p][2] >> 16) | u[p][3]);
}

struct GemmArgs {
  const float *A, *B;
  float* C;
  const float* bias;
  int rows_a, rows_b;       // tiles past them read the last row and store nothing
  int red;                  // reduction length
  int lda, ldb;
  size_t ldc;
  size_t batch_b, batch_c;  // strides of a batch element (TN: batch_c of the split)
  int split;                // TN: reduction elements of one split
  int spread;               // TN: splits and tiles dealt to the XCDs together
  int tiles_a, tiles_b;
};

template <int MM, bool TN, int KS, bool CONV>
__global__ __launch_bounds__(KS * kClThreads) void columns_gemm_kernel(GemmArgs g) {
  constexpr int BM = 64, BN = 64;
  constexpr int LA = BM / 32, LB = BN / 32;   // 16-byte pieces per thread and step
  static_assert(CONV ? MM != kMmF32 : MM != kMmBf16, "bf16 operands are formed early, float32 never");
  constexpr int RB = columns_row_bytes(MM, CONV);
  __shared__ __attribute__((aligned(16))) char lds[KS][2][(BM + BN) * RB];
  __shared__ float s_bias[BM];
  // consecutive slots of one XCD share the tile of the larger operand, or (spread) the rows of one
  // split (workgroup ids go round-robin over the 8 XCDs)
  const int total = g.tiles_a * g.tiles_b;
  int slot = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3), z = blockIdx.y;
  if (TN && g.spread) {
    z = slot / total;
    if (z * g.split >= g.red) return;
    slot -= z * total;
  } else {
    if (slot >= total) return;
  }
  const int ta = slot % g.tiles_a, tb = slot / g.tiles_a;
  const int i0 = ta * BM, n0 = tb * BN;
  const int group = KS == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x / kClThreads);
  const int tid = threadIdx.x % kClThreads, lane = tid & 63, wave = tid >> 6;
  const int j = lane & 31, h = lane >> 5;
  const int wr = (wave >> 1) * 32, wc = (wave & 1) * 32;
  char* As[2] = {lds[group][0], lds[group][1]};
  char* Bs[2] = {lds[group][0] + BM * RB, lds[group][1] + BM * RB};
  const float* B = TN ? g.B : g.B + (size_t)z * g.batch_b;
  float* C = g.C + (size_t)z * g.batch_c;
  const int r_begin = TN ? z * g.split : 0;
  const int r_end = TN ? min(r_begin + g.split, g.red) : g.red;

  const int kb = tid & 7, rb = tid >> 3;   // reduction quad, row (TN: quad of columns)
  vec4 ra[2][LA], rbv[2][LB];   // two steps in flight
  const vec4 zero = {0.f, 0.f, 0.f, 0.f};
  auto fetch = [&](int r0, vec4 (&ga)[LA], vec4 (&gb)[LB]) {
    // (every read is made, from a clamped address, and what lies past the end becomes zero on
    // the way to LDS: a test around a read costs a branch and a wait for it)
    if constexpr (!TN) {
      const int r = min(r0 + 4 * kb, g.red - 4);
#pragma unroll
      for (int i = 0; i < LA; ++i)
        ga[i] = *reinterpret_cast<const vec4*>(g.A + (size_t)min(i0 + rb + 32 * i, g.rows_a - 1) * g.lda + r);
#pragma unroll
      for (int i = 0; i < LB; ++i)
        gb[i] = *reinterpret_cast<const vec4*>(B + (size_t)min(n0 + rb + 32 * i, g.rows_b - 1) * g.ldb + r);
    } else {
      // blocks of four reduction rows x four columns: threads 0..127 take A's, the others B's
      const bool is_a = tid < 128;
      const int ld = is_a ? g.lda : g.ldb;
      const float* src = (is_a ? g.A : B) + min((is_a ? i0 : n0) + 4 * (rb & 15), ld - 4);
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const vec4 v = *reinterpret_cast<const vec4*>(src + (size_t)min(r0 + 4 * kb + e, g.red - 1) * ld);
        if (e < 2) ga[e] = v;
        else gb[e - 2] = v;
      }
    }
  };
  // four reduction elements, quad kb of a row
  auto put = [&](char* row, const vec4& v) {
    if constexpr (!CONV) {
      *reinterpret_cast<vec4*>(row + 16 * kb) = v;
    } else if constexpr (MM == kMmBf16) {
      *reinterpret_cast<uint2*>(row + 8 * kb) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    } else {
      uint2 piece[3];
      split_bf16x4(v, piece);
#pragma unroll
      for (int p = 0; p < 3; ++p) *reinterpret_cast<uint2*>(row + 64 * p + 8 * kb) = piece[p];
    }
  };
  auto stash = [&](int buf, int r0, const vec4 (&ga)[LA], const vec4 (&gb)[LB]) {
    if constexpr (!TN) {
      const bool on = r0 + 4 * kb < r_end;
#pragma unroll
      for (int i = 0; i < LA; ++i)
        put(As[buf] + (rb + 32 * i) * RB, on ? ga[i] : zero);
#pragma unroll
      for (int i = 0; i < LB; ++i)
        put(Bs[buf] + (rb + 32 * i) * RB, on ? gb[i] : zero);
    } else {
      char* dst = (tid < 128 ? As[buf] : Bs[buf]) + 4 * (rb & 15) * RB;
      const int r = r0 + 4 * kb;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const vec4 v = {r < r_end ? ga[0][e] : 0.0f, r + 1 < r_end ? ga[1][e] : 0.0f,
                        r + 2 < r_end ? gb[0][e] : 0.0f, r + 3 < r_end ? gb[1][e] : 0.0f};
        put(dst + e * RB, v);
      }
    }
  };

  if (threadIdx.x < BM)
    s_bias[threadIdx.x] = !TN && g.bias != nullptr ? g.bias[min(i0 + (int)threadIdx.x, g.rows_a - 1)] : 0.0f;

  const floatx16 none = {};
  floatx16 acc = none, all = none;   // (TN: all = the sums of two steps each, acc those under way)

  auto load8 = [&](const char* p, float (&f)[8]) {
    const vec4 lo = *reinterpret_cast<const vec4*>(p), hi = *reinterpret_cast<const vec4*>(p + 16);
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      f[e] = lo[e];
      f[4 + e] = hi[e];
    }
  };

  auto multiply = [&](int buf) {
    if (TN && buf == 0) acc = none;
#pragma unroll
    for (int s = 0; s < kGk / 16; ++s) {
      if constexpr (CONV) {
        auto piece = [&](const char* row, int p) {
          return __builtin_bit_cast(Bf16Frag, *reinterpret_cast<const uint4*>(row + 64 * p));
        };
        const char* pa = As[buf] + (wr + j) * RB + 32 * s + 16 * h;
        const char* pb = Bs[buf] + (wc + j) * RB + 32 * s + 16 * h;
        if constexpr (MM == kMmBf16) {
          acc = mfma_bf16(piece(pa, 0), piece(pb, 0), acc);
        } else {
          const Bf16Split a = {piece(pa, 0), piece(pa, 1), piece(pa, 2)};
          const Bf16Split b = {piece(pb, 0), piece(pb, 1), piece(pb, 2)};
          acc = mfma_split(a, b, acc);
        }
      } else {
        float fa[8], fb[8];
        load8(As[buf] + (wr + j) * RB + 64 * s + 32 * h, fa);
        load8(Bs[buf] + (wc + j) * RB + 64 * s + 32 * h, fb);
        if constexpr (MM == kMmF32) {
#pragma unroll
          for (int e = 0; e < 8; ++e)
            acc = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[e], acc, 0, 0, 0);
        } else {
          acc = mfma_split(split_bf16x8(fa), split_bf16x8(fb), acc);
        }
      }
    }
  };

  // step t: registers t & 1 hold its values until they go to LDS buffer t & 1, one step ahead
  // of the MFMAs; step t + 2 is requested right after.  With KS groups, group q's step t is the
  // reduction's step KS t + q.
  constexpr int kStep = KS * kGk;
  const int steps = (r_end - r_begin + kStep - 1) / kStep;
  const int r_first = r_begin + group * kGk;
  fetch(r_first, ra[0], rbv[0]);
  fetch(r_first + kStep, ra[1], rbv[1]);
  stash(0, r_first, ra[0], rbv[0]);
  __syncthreads();
  // (the scheduling barriers keep the requests in front of the MFMAs and the waits for older
  // ones behind them; left alone the compiler sinks the requests to their uses)
  for (int t = 0; t < steps; t += 2) {
    const int r0 = r_first + t * kStep;
    fetch(r0 + 2 * kStep, ra[0], rbv[0]);
    __builtin_amdgcn_sched_barrier(0);
    multiply(0);
    __builtin_amdgcn_sched_barrier(0);
    stash(1, r0 + kStep, ra[1], rbv[1]);
    __syncthreads();
    fetch(r0 + 3 * kStep, ra[1], rbv[1]);
    __builtin_amdgcn_sched_barrier(0);
    multiply(1);   // (a step past the end multiplies zeros)
    __builtin_amdgcn_sched_barrier(0);
    stash(0, r0 + 2 * kStep, ra[0], rbv[0]);
    if constexpr (TN) all += acc;
    __syncthreads();
  }
  if constexpr (TN) acc = all;
  if constexpr (KS == 2) {
    // the second group's sums join the first's through LDS, [register][thread]
    static_assert(2 * (BM + BN) * RB >= 16 * kClThreads * (int)sizeof(float), "sums fit a group's rows");
    float* sums = reinterpret_cast<float*>(lds[1][0]);
    if (group == 1) {
#pragma unroll
      for (int v = 0; v < 16; ++v) sums[v * kClThreads + tid] = acc[v];
    }
    __syncthreads();
    if (group == 1) return;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] += sums[v * kClThreads + tid];
  }
  const int n = n0 + wc + j;
#pragma unroll
  for (int v = 0; v < 16; ++v) {
    const int i = wr + 8 * (v >> 2) + 4 * h + (v & 3);
    if (i0 + i < g.rows_a && n < g.rows_b) C[(size_t)(i0 + i) * g.ldc + n] = acc[v] + s_bias[i];
  }
}

// gW[i][c][k] = sum over the splits of partial[split][i][k][c].
__global__ __launch_bounds__(kClThreads) void columns_wgrad_sum_kernel(
    const float* __restrict__ partial, float* __restrict__ gW, int splits, size_t split_stride,
    int Cg, int Cgp, int K, int total) {
  const int e = blockIdx.x * kClThreads + threadIdx.x;   // (i, k, c), c fastest
  if (e >= total) return;
  const int c = e % Cgp, q = e / Cgp, k = q % K, i = q / K;
  if (c >= Cg) return;
  float sum = 0.f;
  for (int s = 0; s < splits; s += 8) {
    float v[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = partial[(size_t)min(s + x, splits - 1) * split_stride + e];
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = s + x < splits ? v[x] : 0.0f;
    sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  gW[((size_t)i * Cg + c) * K + k] = sum;
}

// img[b][c][u] = bias[c] + sum over the entries of u's list of coefficient * col[b][sample][c].
// A workgroup owns 256 / (L S) image elements x 4 L channels of one batch element, L S lanes an element:
// L lanes read an entry's products as one run, S such groups share the list, eight entries of it in
// flight, and the sums leave through LDS as runs along the image.  L is what the channels fill: with 16
// lanes of which two have channels (8 -> 56, 6 x 100 x 200, 5 x 5) 154 us, with L = 2 and S = 4 84; 64 channels
// 24 us with S = 1, 22 with S = 2; 96 channels 17 us in two chunks of 64, 15 in three of 32.  grid (blocks of
// elements, channel chunks, batch).
// A list of more than kClLong entries (a map that sends many samples to one image element, invalid ones
// for instance) is the whole workgroup's: eight entries in turn for each group of L lanes, whose
// sums are added in their order.  (64 channels, 1 x 128 x 256, a tenth of 295 thousand samples on
// one spot, backward: 365 us with 16 lanes, 219 with 8; 117 without the spot.)
constexpr int kClLong = 256;
template <int L, int S>
__global__ __launch_bounds__(kClThreads, 6) void columns_col2im_kernel(
    const float* __restrict__ col, const int* __restrict__ offset, const int* __restrict__ src,
    const float* __restrict__ co, const float* __restrict__ bias, float* __restrict__ img, int Cg,
    int C4, int HW, int samples) {
  constexpr int T = kClThreads / (L * S);
  __shared__ float tile[4 * L][T + 1];
  __shared__ vec4 parts[T][L * S];
  const int ql = threadIdx.x % (L * S), q = ql % L, share = ql / L, t = threadIdx.x / (L * S);
  const int u0 = blockIdx.x * T, c0 = blockIdx.y * (4 * L);
  const vec4* col_b = reinterpret_cast<const vec4*>(col) + (size_t)blockIdx.z * samples * C4 +
                      min(c0 / 4 + q, C4 - 1);
  vec4 acc = {0.f, 0.f, 0.f, 0.f};
  constexpr int kShort = 8 / S, kLong = 8;   // entries of a lane in flight
  // acc += this lane's shares (U entries of each S * U) of the entries from beg on, S * U and then `step`
  // further each turn, before end (> 0); those of the next turn are named before this one's products are here
  auto add = [&](auto count, int beg, int end, int step) {
    constexpr int U = decltype(count)::value;
    int s[U];
    float w[U];
    auto name = [&](int e) {
#pragma unroll
      for (int i = 0; i < U; ++i) {
        const int at = min(e + i, end - 1);
        w[i] = co[at];
        s[i] = src[at];
      }
    };
    beg += share * U;
    if (beg < end) name(beg);
    for (int e = beg; e < end; e += step) {
      vec4 v[U];
      float here[U];
#pragma unroll
      for (int i = 0; i < U; ++i) {
        v[i] = col_b[(size_t)s[i] * C4];
        here[i] = w[i];
      }
      if (e + step < end) name(e + step);
#pragma unroll
      for (int i = 0; i < U; ++i)
        if (e + i < end) acc += here[i] * v[i];
    }
  };
  const int u = min(u0 + t, HW - 1);
  const int beg = offset[u], end = offset[u + 1];
  if (end - beg <= kClLong) add(std::integral_constant<int, kShort>(), beg, end, 8);
  if (__syncthreads_or(end - beg > kClLong)) {
    const int u_last = min(u0 + T, HW);
    for (int x = u0; x < u_last; ++x) {
      const int b = offset[x], e = offset[x + 1];
      if (e - b <= kClLong) continue;
      const vec4 own = acc;
      acc = vec4{0.f, 0.f, 0.f, 0.f};
      add(std::integral_constant<int, kLong>(), b + kLong * S * t, e, kLong * S * T);
      parts[t][ql] = acc;
      acc = own;
      __syncthreads();
      if (t == x - u0) {
        acc = parts[0][ql];
        for (int p = 1; p < T; ++p) acc += parts[p][ql];
      }
      __syncthreads();
    }
  }
#pragma unroll
  for (int x = 0; x < 4; ++x) {
#pragma unroll
    for (int d = L; d < L * S; d *= 2) acc[x] += __shfl_xor(acc[x], d, 64);
    tile[4 * q + x][t] = acc[x];   // (equal in the lanes that share a place)
  }
  __syncthreads();
  float* img_b = img + (size_t)blockIdx.z * Cg * HW;
#pragma unroll
  for (int i = 0; i < 4 / S; ++i) {
    const int item = threadIdx.x + kClThreads * i, c = item / T, n = item % T;
    if (c0 + c < Cg && u0 + n < HW)
      img_b[(size_t)(c0 + c) * HW + u0 + n] = tile[c][n] + (bias != nullptr ? bias[c0 + c] : 0.0f);
  }
}

// ---------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------
size_t up256(size_t v) { return (v + 255) & ~(size_t)255; }

// What a call's contractions take at a time.
struct Slices {
  bool both;
  int64_t scatter, wgrad;   // elements of the batch
  int channels;
};

struct ColumnsLayout {
  size_t pix_rows, pix_cols, img_rows, col, weights, partial, strip_sums, lists, total;
  int splits, split_len;
  Slices slices;
};

size_t column_values(const ConvGeom& g) { return (size_t)g.B * g.M * g.K * pad8(g.Cg); }

// The products of a scatter go through in slices of so many batch elements that a slice is still in the 256 MB
// memory-side cache when it is read back (4 x 128 x 256, 64 -> 64, backward: 474 us in one piece of 288 MB, 442 in
// two, 421 in four), at least one; an element that alone has more than that cache in chunks of so many channels, at
// least 32, a run of 128 bytes (backward, float32 / bf16, us, whole and so: 793 MB, 104 -> 88, 200 x 400, 5 x 5 1973 /
// 1363 and 1799 / 1138; 381 MB, 200 -> 160, 100 x 200 1636 / 801 and 1592 / 688; but 200 MB, 8 x 128 x 256, 64 -> 256,
// whose pixels are as large, 6143 / 2624 and 6404 / 2713).
// Both forms of the pixels' operands are laid out in one launch, side by side, where they take less than 256 MB; beyond
// that each contraction lays out its own, one after the other in the same place, of elements of up to 256 MB (both always
// and so, float32: 8 x 256 x 512, 64 -> 64, 5 x 5 1938 and 626 MB of workspace, backward 9857 and 10035 us; 8 x 128 x
// 256, 64 -> 256 1286 and 586, 6100 and 6331; apart from 128 MB on 16 -> 194, 3 x 302 x 605, stride 2 487 and 520 us).
// The line gives time for memory: few channels into many lose most beyond it (16 -> 256 there, 280 MB 526 and 574 us;
// split 16 -> 194, 412 MB 491 and 508); 512 MB would take back those, and add up to 300 MB to such calls' workspace.
constexpr size_t kSliceBytes = (size_t)128 << 20, kCacheBytes = (size_t)256 << 20;
constexpr size_t kOperandBytes = (size_t)256 << 20;
Slices slices_of(const ConvGeom& g, int mm) {
  const size_t samples = sizeof(float) * g.M * g.K;
  const size_t rows = columns_pixel_row_bytes(g, mm, 1), cols = columns_pixel_column_bytes(g, mm, 1);
  auto elements = [&](size_t most, size_t one) { return std::max<int64_t>(1, std::min<int64_t>(g.B, most / one)); };
  Slices s;
  s.both = g.B * (rows + cols) < kOperandBytes;
  s.wgrad = s.both ? g.B : elements(kOperandBytes, rows);
  s.channels = pad8(g.Cg);
  if (samples * s.channels > kCacheBytes && s.channels > 32) {
    const int64_t most = std::max<int64_t>(1, kSliceBytes / (32 * samples));   // chunks of 32, shared out evenly
    s.channels = std::min(s.channels, (int)(32 * ceil_div(s.channels, 32 * ceil_div(s.channels, 32 * most))));
    s.scatter = 1;
  } else {
    s.scatter = elements(kSliceBytes, samples * s.channels);
  }
  if (!s.both) s.scatter = std::min(s.scatter, elements(kOperandBytes, cols));
  return s;
}

// Of a forward, or of both gradients.
ColumnsLayout columns_layout(const ConvGeom& g, int mm, bool backward) {
  const int Cgp = pad8(g.Cg), Cpp = pad8(g.Cp);
  ColumnsLayout l{};
  size_t at = 0;
  auto take = [&](size_t bytes) {
    const size_t here = at;
    at += up256(bytes);
    return here;
  };
  const size_t image = sizeof(float) * ((size_t)g.B * g.H * g.W + 1) * Cgp;   // (and a row of zeros)
  // The image first, always: the gather and the weight gradient of a transposed layer's backward lay out the same one,
  // and a second copy beside the first pushes both out of the memory-side cache (84 MB, icosphere level 7, 128
  // channels: weight gradient 34 us in one place, 51 in two).
  if (!backward && columns_direct_gather(g, mm)) {
    l.img_rows = take(image);
    l.weights = take(columns_weight_bytes(g, mm));
    l.partial = take(columns_forward_sum_bytes(g, mm));
  } else if (backward && columns_direct_backward(g, mm)) {
    const Slices& t = l.slices = slices_of(g, mm);
    l.img_rows = take(image);
    l.pix_rows = take(columns_pixel_row_bytes(g, mm, t.wgrad));
    // (not in the products' place: 256 x 4 x 6 pixels, 64 -> 128, bf16, backward 52 us, 57 so)
    l.partial = take(columns_partial_bytes(g, mm, t.wgrad));
    const size_t end = at;
    if (!t.both) at = 0;
    l.pix_cols = take(columns_pixel_column_bytes(g, mm, t.both ? g.B : t.scatter));
    l.col = take(sizeof(float) * t.scatter * g.M * g.K * t.channels);
    at = std::max(at, end);
    l.weights = take(columns_weight_bytes(g, mm));
    l.strip_sums = take(columns_strip_bytes(g));
  } else {
    l.img_rows = take(image);
    l.col = take(sizeof(float) * column_values(g));
    l.weights = take(sizeof(float) * g.K * Cgp * Cpp);
    l.pix_rows = take(sizeof(float) * g.B * g.M * Cpp);
    // the weight gradient's reduction (all pixels of the batch) in splits: about two
    // workgroups per CU, at least 64 pixels each
    const int64_t tiles = ceil_div(g.Cp, 64) * ceil_div((int64_t)g.K * Cgp, 64);
    const int64_t pixels = g.B * (int64_t)g.M;
    int64_t splits = std::max<int64_t>(1, std::min<int64_t>(ceil_div(512, tiles), ceil_div(pixels, 64)));
    l.split_len = (int)(ceil_div(ceil_div(pixels, splits), kGk) * kGk);
    l.splits = (int)ceil_div(pixels, l.split_len);
    l.partial = take(sizeof(float) * l.splits * g.Cp * g.K * Cgp);
  }
  l.lists = at;
  l.total = at + (backward ? up256(col2im_lists_bytes(g.H, g.W, g.M, g.K, g.P, g.interp)) : 0);
  return l;
}

ColumnsScratch columns_scratch(const ColumnsLayout& l, char* ws) {
  return ColumnsScratch{reinterpret_cast<float*>(ws + l.img_rows), ws + l.weights, ws + l.pix_rows, ws + l.pix_cols,
                        reinterpret_cast<float*>(ws + l.strip_sums), reinterpret_cast<float*>(ws + l.col),
                        reinterpret_cast<float*>(ws + l.partial)};
}

int to_rows(const float* src, float* dst, int64_t B, int C, int64_t N, hipStream_t stream) {
  const dim3 grid((unsigned)ceil_div(N, 64), (unsigned)ceil_div(pad8(C), 32), (unsigned)B);
  launch(channels_last_kernel, grid, dim3(kClThreads), stream, src, dst, C, pad8(C), (int)N);
  SDK_LAUNCH_CHECK("mapped_conv(channels last)");
  return SDK_OK;
}

int make_columns(const ConvGeom& g, const float* rows, const float* map, const float* wts,
                 float* col, hipStream_t stream) {
  const int samples = g.M * g.K;
  const dim3 grid((unsigned)ceil_div(samples, kClSamples), (unsigned)g.B);
  const int C4 = pad8(g.Cg) / 4;
  SDK_DISPATCH_INTERP(g.interp, g.P,
                      (launch((columns_kernel<INTERP, WEIGHTED, WEIGHTED ? 32 : 4>), grid,
                              dim3(kClThreads), stream, rows, map, wts, col, samples, g.P, g.H,
                              g.W, C4)));
  SDK_LAUNCH_CHECK("mapped_conv(columns)");
  return SDK_OK;
}

template <bool TN>
int gemm(int mm, GemmArgs a, int64_t batches, hipStream_t stream) {
  a.tiles_a = (int)ceil_div(a.rows_a, 64);
  a.tiles_b = (int)ceil_div(a.rows_b, 64);
  const int64_t total = (int64_t)a.tiles_a * a.tiles_b;
  // Tiles of a weight gradient that leave more than an eighth of the XCDs' shares empty are dealt together
  // with the splits: one tile in 450 splits is not one XCD's.  (32 x 32 in runs of 256 of 115200 pixels, split,
  // the product alone 74 -> 13.5 us, 8 x 720 in runs of 672 40.3 -> 38.2; with 40 tiles, 200 x 600 in runs
  // of 256, 16.6 -> 20.2, so not there.)
  const int64_t padded = (total + 7) / 8 * 8;
  a.spread = TN && 8 * total < 7 * padded;
  const dim3 grid((unsigned)(a.spread ? (total * batches + 7) / 8 * 8 : padded),
                  (unsigned)(a.spread ? 1 : batches));
  // Two groups of waves per tile, each with every other step of a reduction that is long enough to share, where the
  // tiles alone leave the SIMDs with a wave or two.  (Whole forward of eight points a sample, float32 / bf16 / split,
  // one group and two: 1 x 20 x 40, 256 -> 200 125 / 96 / 121 and 123 / 92 / 118 us; 2 x 24 x 48, 128 -> 96, nearest
  // 54 / 40 / 52 and 54 / 38 / 50; of many more tiles no faster: five points, 1 x 128 x 256, 64 -> 64 99 / 86 / 94 and
  // 99 / 87 / 99; but the chains of the sums are half as long.)
  const bool shared = !TN && total * batches <= (mm == kMmF32 ? 256 : 1024) && a.red >= 4 * kGk;
  // Split operands are formed early by the weight gradient, where a reduction is longer than two steps, and by a
  // forward of so few tiles that all are at work at once either way.  (us late and early: backward of one sample,
  // 40 -> 232, 2 x 147 x 290 159 and 150, 64 -> 232 172 and 164; forward 40 -> 232 51 and 54, 24 -> 83, 3 x 156 x 312
  // 46 and 50, 8 -> 64, 4 x 181 x 363 43 and 45; eight points, 6 x 50 x 100, stride 2, 96 -> 160, backward 185 and 181.)
  const bool early = TN || a.red > 2 * kGk || (a.rows_a <= a.rows_b && total * batches <= 768);
#define CG2(MMv, KSv, CONVv) \
  launch((columns_gemm_kernel<MMv, TN, KSv, CONVv>), grid, dim3(KSv * kClThreads), stream, a)
  if constexpr (!TN) {
    if (shared) {
      if (mm == kMmBf16) CG2(kMmBf16, 2, true);
      else if (mm == kMmSplit) CG2(kMmSplit, 2, false);
      else CG2(kMmF32, 2, false);
    }
  }
  if (!shared) {
    if (mm == kMmBf16) CG2(kMmBf16, 1, true);
    else if (mm == kMmF32) CG2(kMmF32, 1, false);
    else if (early) CG2(kMmSplit, 1, true);
    else CG2(kMmSplit, 1, false);
  }
#undef CG2
  SDK_LAUNCH_CHECK("mapped_conv(columns product)");
  return SDK_OK;
}

// Calls whose column matrix has at most this many bytes take the route (a scatter holds a slice of it, the others
// none of it).  On a kept plan, 3 x 3 kernels, us of the tile kernels and of these, float32 / bf16 / split, forward
// and backward, and the forward alone:
//   112 MB  4 x 160 x 320, 16 -> 16   350 / 231 / 294 and 213 / 181 / 221    72 /  46 /  59 and  59 /  44 /  60
//   122 MB  6 x 96 x 192, 32 -> 32    304 / 210 / 266 and 217 / 168 / 216    46 /  34 /  41 and  59 /  42 /  58
//   122 MB  8 x 96 x 192, 24 -> 24    274 / 194 / 238 and 246 / 196 / 243    54 /  37 /  46 and  60 /  44 /  54
//   126 MB  4 x 120 x 240, 32 -> 32   271 / 194 / 238 and 219 / 173 / 216    55 /  38 /  48 and  59 /  44 /  58
//   131 MB  2 x 100 x 200, 96 -> 160  990 / 377 / 690 and 618 / 254 / 472   259 /  81 / 173 and 181 /  60 / 136
//   142 MB  4 x 90 x 180, 64 -> 64    371 / 236 / 304 and 300 / 190 / 288    92 /  49 /  70 and  71 /  45 /  69
//   175 MB  4 x 200 x 400, 16 -> 16   444 / 276 / 367 and 384 / 306 / 403
//   288 MB  4 x 128 x 256, 64 -> 64   513 / 284 / 400 and 558 / 344 / 530
// nearest taps
//    72 MB  2 x 128 x 256, 32 -> 32   177 / 138 / 162 and 107 /  78 / 106    37 /  27 /  33 and  25 /  18 /  23
//   108 MB  4 x 64 x 128, 96 -> 96    513 / 246 / 387 and 284 / 119 / 219   147 /  58 / 103 and  78 /  30 /  64
//   122 MB  8 x 96 x 192, 24 -> 24    215 / 155 / 187 and 176 / 121 / 180    48 /  33 /  41 and  50 /  28 /  41
//   144 MB  2 x 256 x 512, 12 -> 24   289 / 192 / 240 and 231 / 153 / 239    70 /  42 /  54 and  56 /  33 /  50
//   288 MB  4 x 128 x 256, 64 -> 64   460 / 247 / 356 and 480 / 253 / 415
// (A forward of 24 or 32 channels that is called again and again on one map is faster by the tile kernels from 100 MB
// on; the first call on a map, which builds their plan for 200 to 300 us, is not, nor is a training step.)
// Above ten samples the tile kernels' weight gradient is another, 5 x 5:
//   400 MB  2 x 128 x 256, 64 -> 64  1815 / 1403 / 1657 and 737 / 475 / 694   492 / 335 / 430 and 164 / 92 / 159
//   693 MB  8 x 169 x 336, 16 -> 56  4043 / 2935 / 3529 and 1676 / 1169 / 1600   734 / 371 / 544 and 317 / 190 / 308
//   793 MB  1 x 200 x 400, 104 -> 88  4320 / 2396 / 3274 and 2358 / 1367 / 1945   1417 / 597 / 982 and 554 / 222 / 412
//   800 MB  4 x 128 x 256, 64 -> 64, nearest  1616 / 926 / 1301 and 1188 / 616 / 996
//           309 / 106 / 224 and 325 / 92 / 215
//   1.6 GB  8 x 128 x 256, 64 -> 256  11929 / 7004 / 9174 and 8576 / 3450 / 6460
//           2137 / 742 / 1457 and 2235 / 709 / 1615
//   3.2 GB  8 x 256 x 512, 32 -> 32  6085 / 4988 / 5805 and 5166 / 4197 / 5132   912 / 555 / 755 and 877 / 568 / 846
//   6.4 GB  8 x 256 x 512, 64 -> 64  13310 / 8850 / 11446 and 12557 / 8334 / 11489
//           2399 / 1039 / 1796 and 2429 / 1226 / 2176
// No training step up there is slower by columns; forwards alone are even from about 1.5 GB on and behind, where split
// or bf16, by up to a fifth at the end.  What ends the route are the 1 GB below.
// Weighted samples stop at the line their calls had when the columns went through memory, for those whose
// samples have more than four taps.
// Fewer than seven samples leave the tile kernels' scatter little to sum twice, and pixels and image are most of the
// traffic: the lines their calls had when the columns went through memory.  us of the tile kernels -> by columns,
// float32 / bf16 / split:
//                                                 forward                  backward
//   nearest, one, 4 x 159 x 316, 64 -> 128    65/ 43/ 57 ->  73/ 51/ 65    173/138/161 -> 271/201/293
//   nearest, four, 8 x 120 x 240, 32 -> 64    59/ 36/ 48 ->  68/ 36/ 51    161/115/136 -> 200/136/224
//   nearest, four, 4 x 159 x 316, 16 -> 128   87/ 41/ 64 ->  60/ 35/ 51    237/151/194 -> 225/149/245
//   bilinear, one, 8 x 200 x 400, 48 -> 64   122/103/127 -> 165/153/187    316/282/308 -> 538/457/578
//   bilinear, four, 8 x 120 x 240, 32 -> 64   68/ 43/ 59 ->  72/ 51/ 74    203/149/176 -> 224/162/247
// (the third, few channels into many, is the one kind that float32 loses by it.)
constexpr size_t kColumnsBytes = (size_t)150 << 20, kColumnsWeightedBytes = (size_t)100 << 20;
constexpr size_t kColumnsFewBytes = (size_t)100 << 20, kColumnsFewNearestBytes = (size_t)36 << 20;
constexpr int kTileSamples = 10, kFewSamples = 7;
// ... and the tensors laid out for them (32-bit byte offsets into the image's rows)
constexpr size_t kColumnsTensorBytes = (size_t)1 << 30, kColumnsElementBytes = (size_t)1 << 30;
bool columns_fit(const ConvGeom& g) {
  const size_t image = sizeof(float) * g.B * g.H * g.W * pad8(g.Cg), pixels = sizeof(float) * g.B * g.M * pad8(g.Cp);
  const size_t columns = sizeof(float) * column_values(g);
  if (g.K > kTileSamples && columns_direct(g))
    return columns / g.B <= kColumnsElementBytes && image <= kColumnsTensorBytes && pixels <= kColumnsTensorBytes;
  const size_t few = g.interp == 0 ? kColumnsFewNearestBytes : kColumnsFewBytes;
  const size_t limit = g.P != 0 ? kColumnsWeightedBytes : (g.K < kFewSamples ? few : kColumnsBytes);
  return columns <= limit && image <= 2 * limit && pixels <= 2 * limit;
}

thread_local bool t_columns = true;

}  // namespace

bool columns_map(const ConvGeom& g) {
  // (the lists of the inverted map: 32 bytes a sample of four taps)
  const int64_t most = (int64_t)1 << (!columns_direct(g) || g.K < kFewSamples ? 20 : (g.K > kTileSamples ? 24 : 21));
  return g.M >= 1 && g.K >= 1 && (int64_t)g.M * g.K <= most && pts(g.P) <= 8 &&
         col2im_lists_bytes(g.H, g.W, g.M, g.K, g.P, g.interp) != 0;
}

bool columns_route(const ConvGeom& g) {
  return t_columns && g.B >= 1 && g.B <= 65535 && g.Cg >= 5 && columns_map(g) && columns_fit(g) &&
         (size_t)pad8(g.Cp) * g.K * pad8(g.Cg) < ((size_t)1 << 31);
}

// (a wave adds up a channel's strips)
bool columns_sums_bias(const ConvGeom& g, int mm) {
  return columns_direct_backward(g, mm) && g.B * ceil_div(g.M, 64) <= 4096;
}

// One size for every arithmetic and direction.  Where split operands, the largest, lie side by side, their backward's is
// it, but for the sums, of which other shapes of tiles, or a forward, may have more.  (Six layouts a query are 300 ns a
// query more, two or three queries a call.)
size_t columns_workspace_bytes(const ConvGeom& g) {
  if (!columns_route(g)) return 0;
  if (g.K > 1 && columns_direct(g)) {
    const ColumnsLayout l = columns_layout(g, kMmSplit, true);
    if (l.slices.both) {
      const size_t split = columns_partial_bytes(g, kMmSplit, g.B), f32 = columns_partial_bytes(g, kMmF32, g.B);
      return l.total - up256(split) + up256(std::max({split, f32, columns_forward_sum_bytes(g, kMmSplit)}));
    }
  }
  size_t most = 0;
  for (int mm : {kMmF32, kMmBf16, kMmSplit})
    for (bool backward : {false, true}) most = std::max(most, columns_layout(g, mm, backward).total);
  return most;
}

int columns_gather_gemm(const ConvGeom& g, int mm, const float* img, const float* map,
                        const float* wts, const float* Wm, const float* bias, float* pix,
                        void* workspace, hipStream_t stream) {
  const ColumnsLayout l = columns_layout(g, mm, false);
  char* ws = static_cast<char*>(workspace);
  float* rows = reinterpret_cast<float*>(ws + l.img_rows);
  float* col = reinterpret_cast<float*>(ws + l.col);
  float* w = reinterpret_cast<float*>(ws + l.weights);
  if (columns_direct_gather(g, mm))
    return columns_direct_forward(g, mm, img, map, wts, Wm, bias, pix, columns_scratch(l, ws), stream);
  const int Cgp = pad8(g.Cg), R = g.K * Cgp;
  int rc = to_rows(img, rows, g.B, g.Cg, (int64_t)g.H * g.W, stream);
  if (rc) return rc;
  rc = make_columns(g, rows, map, wts, col, stream);
  if (rc) return rc;
  const int total = g.Cp * R;
  launch(columns_weight_kernel<false>, dim3((unsigned)ceil_div(total, kClThreads)),
         dim3(kClThreads), stream, Wm, w, g.Cg, Cgp, g.K, g.Cp, g.Cp, total);
  SDK_LAUNCH_CHECK("mapped_conv(columns weights)");
  GemmArgs a{};
  a.A = w;
  a.B = col;
  a.C = pix;
  a.bias = bias;
  a.rows_a = g.Cp;
  a.rows_b = g.M;
  a.red = R;
  a.lda = a.ldb = R;
  a.ldc = (size_t)g.M;
  a.batch_b = (size_t)g.M * R;
  a.batch_c = (size_t)g.Cp * g.M;
  return gemm<false>(mm, a, g.B, stream);
}

int columns_gemm_scatter(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* Wm, const float* bias, float* img,
                         void* workspace, hipStream_t stream, const void* lists,
                         const float* wgrad_img, bool bias_sum) {
  const ColumnsLayout l = columns_layout(g, mm, true);
  char* ws = static_cast<char*>(workspace);
  float* rows = reinterpret_cast<float*>(ws + l.pix_rows);
  float* col = reinterpret_cast<float*>(ws + l.col);
  float* w = reinterpret_cast<float*>(ws + l.weights);
  const int Cgp = pad8(g.Cg), Cpp = pad8(g.Cp), R = g.K * Cgp;
  int rc = SDK_OK;
  if (lists == nullptr) {
    rc = col2im_lists_build(map, wts, ws + l.lists, g.H, g.W, g.M, g.K, g.P, g.interp, stream);
    if (rc) return rc;
    lists = ws + l.lists;
  }
  const Col2imView v = col2im_lists_view(lists, g.H, g.W, g.M, g.K, g.P, g.interp);
  const int HW = g.H * g.W;
  // channels c0 .. of so many batch elements, of one where they are not all
  auto col2im = [&](int64_t first, int64_t elements, int c0, int padded) -> int {
    float* out = img + ((size_t)first * g.Cg + c0) * HW;
    const float* add = bias != nullptr ? bias + c0 : nullptr;
    const int C4 = padded / 4, channels = std::min(padded, g.Cg - c0);
    // as many lanes an element as its channels fill
#define CI(Lv, Sv)                                                                                            \
  launch((columns_col2im_kernel<Lv, Sv>),                                                                     \
         dim3((unsigned)ceil_div(HW, kClThreads / (Lv * Sv)), (unsigned)ceil_div(C4, Lv), (unsigned)elements), \
         dim3(kClThreads), stream, (const float*)col, v.offset, v.src, v.co, add, out, channels, C4, HW, g.M * g.K)
    if (C4 <= 2) CI(2, 4);
    else if (C4 <= 4) CI(4, 4);
    else CI(8, 2);   // (sixteen lanes: 22 us instead of 23 for 64 channels, a long list half as fast)
#undef CI
    SDK_LAUNCH_CHECK("mapped_conv(columns col2im)");
    return SDK_OK;
  };
  if (columns_direct_backward(g, mm)) {
    const ColumnsScratch s = columns_scratch(l, ws);
    const Slices& t = l.slices;
    const bool rows_too = t.both && wgrad_img != nullptr;
    for (int64_t first = 0; first < g.B; first += t.scatter) {
      const int64_t elements = std::min<int64_t>(t.scatter, g.B - first);
      if (first == 0 || !t.both)
        rc = columns_direct_prepare(g, mm, pix, first, t.both ? g.B : elements, rows_too, true, rows_too && bias_sum,
                                    first == 0 ? Wm : nullptr, t.channels, rows_too ? wgrad_img : nullptr, s, stream);
      for (int c0 = 0; c0 < Cgp && rc == SDK_OK; c0 += t.channels) {
        const int channels = std::min(t.channels, Cgp - c0);
        rc = columns_direct_product(g, mm, t.both ? first : 0, elements, c0, channels, s, stream);
        if (rc == SDK_OK) rc = col2im(first, elements, c0, channels);
      }
      if (rc) return rc;
    }
    return SDK_OK;
  }
  rc = to_rows(pix, rows, g.B, g.Cp, g.M, stream);
  if (rc) return rc;
  const int total = R * Cpp;
  launch(columns_weight_kernel<true>, dim3((unsigned)ceil_div(total, kClThreads)),
         dim3(kClThreads), stream, Wm, w, g.Cg, Cgp, g.K, g.Cp, Cpp, total);
  SDK_LAUNCH_CHECK("mapped_conv(columns weights)");
  // all pixels of the batch are the rows of one product
  GemmArgs a{};
  a.A = rows;
  a.B = w;
  a.C = col;
  a.rows_a = (int)(g.B * g.M);
  a.rows_b = R;
  a.red = Cpp;
  a.lda = a.ldb = Cpp;
  a.ldc = (size_t)R;
  rc = gemm<false>(mm, a, 1, stream);
  if (rc) return rc;
  return col2im(0, g.B, 0, Cgp);
}

int columns_gather_wgrad(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* img, float* gW, void* workspace,
                         hipStream_t stream, bool prepared, float* gb) {
  const ColumnsLayout l = columns_layout(g, mm, true);
  char* ws = static_cast<char*>(workspace);
  if (columns_direct_backward(g, mm))
    return columns_direct_wgrad(g, mm, pix, map, wts, img, gW, l.slices.wgrad, columns_scratch(l, ws),
                                prepared && l.slices.both, gb, stream);
  float* prows = reinterpret_cast<float*>(ws + l.pix_rows);
  float* irows = reinterpret_cast<float*>(ws + l.img_rows);
  float* col = reinterpret_cast<float*>(ws + l.col);
  float* partial = reinterpret_cast<float*>(ws + l.partial);
  const int Cgp = pad8(g.Cg), Cpp = pad8(g.Cp), R = g.K * Cgp;
  int rc = SDK_OK;
  if (!prepared) rc = to_rows(pix, prows, g.B, g.Cp, g.M, stream);
  if (rc) return rc;
  rc = to_rows(img, irows, g.B, g.Cg, (int64_t)g.H * g.W, stream);
  if (rc) return rc;
  rc = make_columns(g, irows, map, wts, col, stream);
  if (rc) return rc;
  GemmArgs a{};
  a.A = prows;
  a.B = col;
  a.C = partial;
  a.rows_a = g.Cp;
  a.rows_b = R;
  a.red = (int)(g.B * g.M);
  a.lda = Cpp;
  a.ldb = R;
  a.ldc = (size_t)R;
  a.batch_c = (size_t)g.Cp * R;
  a.split = l.split_len;
  rc = gemm<true>(mm, a, l.splits, stream);
  if (rc) return rc;
  const int total = g.Cp * R;
  launch(columns_wgrad_sum_kernel, dim3((unsigned)ceil_div(total, kClThreads)), dim3(kClThreads),
         stream, (const float*)partial, gW, l.splits, a.batch_c, g.Cg, Cgp, g.K, total);
  SDK_LAUNCH_CHECK("mapped_conv(columns sums)");
  return SDK_OK;
}

}  // namespace sdk

extern "C" int sdk_mapped_conv_columns_enable(int32_t enabled) {
  const int before = sdk::t_columns ? 1 : 0;
  sdk::t_columns = enabled != 0;
  return before;
}
