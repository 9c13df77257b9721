// Mapped convolution forward of small calls without a column matrix in memory:
//
//   pix[b][n][m] = bias[n] + sum over (k, c) of W[n][c][k] * column(b, m, k, c)
//
// where column(b, m, k, :) is the blend of the image rows sample (m, k) falls between
// (ext_modules/src/cpp/mapped_convolution_layer.cpp:8-60 writes it out first).  The image is
// channels-last (conv_columns.hip), so a tap is one run of channels; the columns of a tile of
// pixels are blended on the way to LDS, 32 reduction elements at a time, and multiplied from there.
//
// Whole forward, us, with the columns written to memory and read back -> so: 64 -> 64, 1 x 128 x 256, float32
// 60 -> 47; 96 -> 160, 6 x 50 x 100, stride 2, split 52 -> 37; 104 -> 37, 2 x 41 x 83, float32 46 -> 23; 200 -> 37,
// 3 x 45 x 91, split 82 -> 47; 256 -> 256, 5 x 5, 2 x 24 x 48, stride 2, split 149 -> 45; 24 -> 32, 2 x 115 x 231,
// float32 50 -> 27.  What bounds it: in float32 the MFMAs (half of the kernel at 64 -> 64) and the vector
// instructions of the blend, which do not overlap them; in the others the blend, and the reads of weights and
// taps by too few waves.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "conv_columns.hpp"
#include "sdk_host.hpp"
#include "sdk_taps.hpp"

namespace sdk {
namespace {

// G groups of RA waves make a tile of 32 RA output channels x 32 pixels of one batch element;
// the groups take steps of 32 reduction elements (k, c) in turn and add up at the end, a wave owns
// 32 channels x all pixels of the tile.  Per step a thread blends up to four channels of NI
// samples (NT taps each, offsets and coefficients from a table in LDS) and leaves them in LDS in
// the form the MFMAs read; the weights come from memory as the operands they are
// (columns_operand_kernel).  The reads of a step are made before the MFMAs of the step before it.
//
// The taps of `cap` samples of every pixel of the tile fit the table at a time; the reduction is
// walked in runs of steps whose samples do.  Unused slots and steps past the end point at a row
// of zeros behind the image, with coefficient zero.  (A sample of more than four taps, possible in
// weighted maps, takes several entries of the table.)
constexpr int kDirectStep = 32, kDirectPixels = 32;
constexpr int row_bytes(int mm) { return mm == kMmF32 ? 144 : (mm == kMmBf16 ? 80 : 208); }

struct DirectArgs {
  const float* rows;        // [B][H * W][Cgp], then a row of zeros
  const float *map, *wts;
  const char* operands;
  const float* bias;
  float* out;
  int B, M, K, P, H, W, interp;
  int Cgp, Cp, steps;       // steps: of the whole reduction
  int tiles_a, tiles_m;
  int cap;
  int split_steps;          // steps of one split; more than one split: sums without bias to `partial`
  float* partial;
};

template <int MM, int RA, int G, int NT>
__global__ __launch_bounds__(64 * RA * G, 2) void columns_forward_kernel(DirectArgs g) {
  constexpr int BN = kDirectPixels, GT = 64 * RA, NI = (8 * BN + GT - 1) / GT, RB = row_bytes(MM);
  constexpr int kThreads = GT * G;
  // steps on their way: one hides behind the float32 MFMAs; two of four samples a thread would not fit the registers
  constexpr int DEEP = MM == kMmF32 || RA == 1 ? 1 : 2;
  constexpr int kFrag = MM == kMmF32 ? 2 : (MM == kMmBf16 ? 1 : 3);   // 16-byte operands of 16 reduction elements
  typedef float vec4 __attribute__((ext_vector_type(4)));
  typedef int ivec4 __attribute__((ext_vector_type(4)));
  extern __shared__ __attribute__((aligned(16))) char lds[];
  __shared__ float s_bias[32 * RA];
  __shared__ int s_most;
  // [group][buffer][pixel] rows, then offsets and coefficients [entry][pixel][NT], entry `cap` = zeros
  int* s_off = reinterpret_cast<int*>(lds + G * 2 * BN * RB);
  float* s_co = reinterpret_cast<float*>(s_off + (g.cap + 1) * BN * NT);

  const int total = g.tiles_a * g.tiles_m * g.B;
  const int slot = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);   // an eighth of the tiles per XCD
  if (slot >= total) return;
  const int ta = slot % g.tiles_a, tm = slot / g.tiles_a % g.tiles_m, b = slot / (g.tiles_a * g.tiles_m);
  const int m0 = tm * BN;
  const int group = __builtin_amdgcn_readfirstlane(threadIdx.x / GT);
  const int tid = threadIdx.x % GT, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  const int HW = g.H * g.W;
  const char* rows_b = reinterpret_cast<const char*>(g.rows + (size_t)b * HW * g.Cgp);
  const int zero_at = (g.B - b) * HW * g.Cgp * 4;

  for (int i = threadIdx.x; i < 32 * RA; i += kThreads)
    s_bias[i] = g.bias != nullptr ? g.bias[min(32 * RA * ta + i, g.Cp - 1)] : 0.0f;
  for (int i = threadIdx.x; i < BN * NT; i += kThreads) {
    s_off[g.cap * BN * NT + i] = zero_at;
    s_co[g.cap * BN * NT + i] = 0.0f;
  }

  // the taps of a weighted sample (m, k): put(i, offset, coefficient) for each that counts; their number
  auto taps = [&](int m, int k, auto&& put) {
    int n = 0;
    auto points = [&](auto tag) {
      constexpr int INTERP = decltype(tag)::value;
      float2 xy[4];
      float wt[4];
#pragma unroll
      for (int p = 0; p < 4; ++p) {   // (all points are requested together; columns_direct: at most four)
        const size_t at = ((size_t)m * g.K + k) * g.P + min(p, g.P - 1);
        __builtin_memcpy(&xy[p], g.map + 2 * at, 8);   // (a map is aligned to its floats)
        wt[p] = g.wts[at];
      }
#pragma unroll
      for (int p = 0; p < 4; ++p) {
        if (p >= g.P) break;
        PointTaps<float, INTERP> t;
        t.set(xy[p].x, xy[p].y, g.H, g.W);
#pragma unroll
        for (int i = 0; i < PointTaps<float, INTERP>::N; ++i) {
          const float c = t.w[i] * wt[p];
          if (t.off[i] >= 0 && c != 0.0f) put(n++, t.off[i], c);
        }
      }
    };
    if (g.interp == 1) points(std::integral_constant<int, 1>());
    else if (g.interp == 2) points(std::integral_constant<int, 2>());
    else points(std::integral_constant<int, 0>());
    return n;
  };
  // entries a sample takes: one, unless a weighted sample of this tile has more than NT taps
  int each = 1;
  if (NT == 4 && g.P != 0) {
    if (threadIdx.x == 0) s_most = 0;
    __syncthreads();
    int most = 0;
    for (int i = threadIdx.x; i < BN * g.K; i += kThreads)
      if (m0 + i / g.K < g.M) most = max(most, taps(m0 + i / g.K, i % g.K, [](int, int, float) {}));
    if (most > NT) atomicMax(&s_most, most);
    __syncthreads();
    each = max(1, (s_most + NT - 1) / NT);
  }
  const int samples = min(g.K, g.cap / each);   // of a run

  // (one group: even and odd turns are summed apart, as two groups' are; the sums of 864 products of the 96 -> 160
  // layer are 3.2e-7 off in the norm so, 4.5e-7 in one chain)
  floatx16 sum[G == 1 ? 2 : 1] = {};

  const int quad = tid & 7, px0 = tid >> 3;
  constexpr int kRowStep = GT / 8;   // pixels between a thread's samples
  const char* frag = g.operands + ((size_t)(ta * RA + wave) * g.steps * 2 * kFrag * 64 + lane) * 16;
  const int tile0 = group * 2 * BN * RB;   // (of lds: the group's two buffers)

  vec4 v[DEEP][NI][NT];   // samples on their way, and their entry and channel
  int at_e[DEEP], at_c[DEEP];
  uint4 a_next[2 * kFrag];
  int t0 = blockIdx.y * g.split_steps;
  const int t_end = min(t0 + g.split_steps, g.steps);
  while (t0 < t_end) {
    // ---- a run: steps t0 .. t1 - 1, samples k0 .. k0 + samples - 1
    const int k0 = t0 * kDirectStep / g.Cgp;
    const int t1 = min(t_end, k0 + samples >= g.K ? g.steps : max(t0 + 1, (k0 + samples) * g.Cgp / kDirectStep));
    __syncthreads();   // the run before is done with the table
    const int held = min(samples, g.K - k0);
    if (g.P == 0) {
      // (four samples at a time: their coordinates are requested together)
      for (int i0 = threadIdx.x; i0 < BN * held; i0 += 4 * kThreads) {
        float2 at[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = min(i0 + u * kThreads, BN * held - 1);
          // (a map is aligned to its floats)
          __builtin_memcpy(&at[u], g.map + 2 * ((size_t)min(m0 + i % BN, g.M - 1) * g.K + k0 + i / BN), 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + u * kThreads;
          if (i >= BN * held) break;
          const bool inside = m0 + i % BN < g.M;
          auto write = [&](auto tag) {
            constexpr int INTERP = decltype(tag)::value;
            PointTaps<float, INTERP> t;
            t.set(at[u].x, at[u].y, g.H, g.W);
            if constexpr (NT == 1) {
              s_off[i] = inside && t.off[0] >= 0 ? t.off[0] * g.Cgp * 4 : zero_at;
            } else {
              ivec4 off;
              vec4 co;
#pragma unroll
              for (int x = 0; x < 4; ++x) {
                const bool on = inside && t.off[x] >= 0;   // (a weight of zero has no offset)
                off[x] = on ? t.off[x] * g.Cgp * 4 : zero_at;
                co[x] = on ? t.w[x] : 0.0f;
              }
              *reinterpret_cast<ivec4*>(s_off + 4 * i) = off;
              *reinterpret_cast<vec4*>(s_co + 4 * i) = co;
            }
          };
          if constexpr (NT == 1) write(std::integral_constant<int, 0>());
          else if (g.interp == 1) write(std::integral_constant<int, 1>());
          else write(std::integral_constant<int, 2>());
        }
      }
    } else if constexpr (NT == 4) {
      for (int i = threadIdx.x; i < BN * held; i += kThreads) {
        const int px = i % BN, k = i / BN;
        int* off = s_off + (k * each * BN + px) * NT;
        float* co = s_co + (k * each * BN + px) * NT;
        int n = 0;
        if (m0 + px < g.M)
          n = taps(m0 + px, k0 + k, [&](int at, int o, float c) {
            const int x = (at / NT) * BN * NT + at % NT;
            off[x] = o * g.Cgp * 4;
            co[x] = c;
          });
        for (; n < NT * each; ++n) {
          const int x = (n / NT) * BN * NT + n % NT;
          off[x] = zero_at;
          co[x] = 0.0f;
        }
      }
    }
    __syncthreads();

    // this thread's samples: reduction element 32 t + 4 quad = (k, c), 32 G further each turn
    int t = t0 + group;
    int k = (t * kDirectStep + 4 * quad) / g.Cgp, c = (t * kDirectStep + 4 * quad) - k * g.Cgp;
    k -= k0;
    const int dk = kDirectStep * G / g.Cgp, dc = kDirectStep * G - dk * g.Cgp;
    auto fetch = [&](int st) {
      at_e[st] = t < t1 && k < held ? k * each : g.cap;
      at_c[st] = at_e[st] == g.cap ? 0 : 4 * c;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int px = NI * GT == 8 * BN ? px0 + i * kRowStep : min(px0 + i * kRowStep, BN - 1);
        if constexpr (NT == 4) {
          const ivec4 o = *reinterpret_cast<const ivec4*>(s_off + (at_e[st] * BN + px) * 4);
#pragma unroll
          for (int x = 0; x < 4; ++x)
            v[st][i][x] = *reinterpret_cast<const vec4*>(rows_b + (unsigned)(o[x] + at_c[st]));
        } else {
          v[st][i][0] = *reinterpret_cast<const vec4*>(rows_b + (unsigned)(s_off[at_e[st] * BN + px] + at_c[st]));
        }
      }
    };
    auto fetch_operands = [&](int step) {
      const char* f = frag + (size_t)min(step, g.steps - 1) * (2 * kFrag * 64 * 16);
#pragma unroll
      for (int i = 0; i < 2 * kFrag; ++i) a_next[i] = *reinterpret_cast<const uint4*>(f + i * 1024);
    };
    auto stash = [&](int st, int buf) {
      char* dst = lds + tile0 + buf * BN * RB;
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int px = px0 + i * kRowStep;
        if (NI * GT != 8 * BN && px >= BN) break;
        vec4 s;
        if constexpr (NT == 4) {
          const vec4 w = *reinterpret_cast<const vec4*>(s_co + (at_e[st] * BN + px) * 4);
#pragma unroll
          for (int x = 0; x < 4; ++x) {
            s[x] = w[0] * v[st][i][0][x];
            s[x] = __builtin_fmaf(w[1], v[st][i][1][x], s[x]);
            s[x] = __builtin_fmaf(w[2], v[st][i][2][x], s[x]);
            s[x] = __builtin_fmaf(w[3], v[st][i][3][x], s[x]);
          }
          for (int q = 1; q < each; ++q)
#pragma unroll
            for (int y = 0; y < 4; ++y) {
              const int at = (min(at_e[st] + q, g.cap) * BN + px) * 4 + y;
              const float w = s_co[at];
              const vec4 r = *reinterpret_cast<const vec4*>(rows_b + (unsigned)(s_off[at] + at_c[st]));
#pragma unroll
              for (int x = 0; x < 4; ++x) s[x] = __builtin_fmaf(w, r[x], s[x]);
            }
        } else {
          s = v[st][i][0];
        }
        char* row = dst + px * RB;
        if constexpr (MM == kMmF32) {
          *reinterpret_cast<vec4*>(row + 16 * quad) = s;
        } else if constexpr (MM == kMmBf16) {
          *reinterpret_cast<uint2*>(row + 8 * quad) = make_uint2(pack_bf16x2(s[0], s[1]), pack_bf16x2(s[2], s[3]));
        } else {
          unsigned u[3][4];
#pragma unroll
          for (int x = 0; x < 4; ++x) split_bf16(s[x], u[0][x], u[1][x], u[2][x]);
#pragma unroll
          for (int p = 0; p < 3; ++p)
            *reinterpret_cast<uint2*>(row + 64 * p + 8 * quad) =
                make_uint2((u[p][0] >> 16) | u[p][1], (u[p][2] >> 16) | u[p][3]);
        }
      }
    };
    auto advance = [&]() {
      t += G;
      k += dk;
      c += dc;
      if (c >= g.Cgp) {
        c -= g.Cgp;
        ++k;
      }
    };

    const int turns = (t1 - t0 + G - 1) / G;
    fetch_operands(t);
    fetch(0);
    if constexpr (DEEP == 2) {
      advance();
      fetch(1);
    }
    stash(0, 0);
    auto turn_of = [&](int turn, auto parity) {
      constexpr int kBuf = decltype(parity)::value, kNext = DEEP == 2 ? kBuf : 0;
      uint4 a[2 * kFrag];
#pragma unroll
      for (int i = 0; i < 2 * kFrag; ++i) a[i] = a_next[i];
      const int now = t0 + group + turn * G;
      advance();
      __syncthreads();
      fetch_operands(now + G);
      fetch(kNext);
      __builtin_amdgcn_sched_barrier(0);
      const char* src = lds + tile0 + kBuf * BN * RB;
      floatx16& acc = sum[G == 1 ? kBuf : 0];
      if (now < t1) {   // (the last turn of a run may have no step left for this group)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const char* row = src + j * RB;
          if constexpr (MM == kMmF32) {
            const vec4 lo = *reinterpret_cast<const vec4*>(row + 64 * s + 32 * h);
            const vec4 hi = *reinterpret_cast<const vec4*>(row + 64 * s + 32 * h + 16);
            const vec4 al = __builtin_bit_cast(vec4, a[2 * s]), ah = __builtin_bit_cast(vec4, a[2 * s + 1]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(al[e], lo[e], acc, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ah[e], hi[e], acc, 0, 0, 0);
          } else {
            auto weights = [&](int q) { return __builtin_bit_cast(Bf16Frag, a[kFrag * s + q]); };
            auto columns = [&](int q) {
              return __builtin_bit_cast(Bf16Frag, *reinterpret_cast<const uint4*>(row + 64 * q + 32 * s + 16 * h));
            };
            if constexpr (MM == kMmBf16) {
              acc = mfma_bf16(weights(0), columns(0), acc);
            } else {
              const Bf16Split x = {weights(0), weights(1), weights(2)}, y = {columns(0), columns(1), columns(2)};
              acc = mfma_split(x, y, acc);
            }
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
      if (turn + 1 < turns) stash(DEEP == 2 ? 1 - kBuf : 0, 1 - kBuf);
    };
    for (int turn = 0; turn < turns; turn += 2) {
      turn_of(turn, std::integral_constant<int, 0>());
      if (turn + 1 < turns) turn_of(turn + 1, std::integral_constant<int, 1>());
    }
    t0 = t1;
  }

  floatx16 acc = sum[0];
  if constexpr (G == 1) {
#pragma unroll
    for (int x = 0; x < 16; ++x) acc[x] += sum[1][x];
  } else {
    // the groups' sums join the first's through LDS, [group][register][thread]
    float* sums = reinterpret_cast<float*>(lds);
    __syncthreads();
    if (group > 0) {
#pragma unroll
      for (int x = 0; x < 16; ++x) sums[((group - 1) * 16 + x) * GT + tid] = acc[x];
    }
    __syncthreads();
    if (group > 0) return;
#pragma unroll
    for (int q = 0; q < G - 1; ++q)
#pragma unroll
      for (int x = 0; x < 16; ++x) acc[x] += sums[(q * 16 + x) * GT + tid];
  }
  const bool whole = g.partial == nullptr;
  float* out = (whole ? g.out : g.partial + (size_t)blockIdx.y * g.B * g.Cp * g.M) + (size_t)b * g.Cp * g.M;
  const int m = m0 + j;
#pragma unroll
  for (int x = 0; x < 16; ++x) {
    const int i = 32 * wave + 8 * (x >> 2) + 4 * h + (x & 3), n = 32 * RA * ta + i;
    if (n < g.Cp && m < g.M) out[(size_t)n * g.M + m] = whole ? acc[x] + s_bias[i] : acc[x];
  }
}

// out[b][n][m] = bias[n] + sum over the splits of partial[split][b][n][m].
__global__ __launch_bounds__(256) void columns_forward_sum_kernel(const float* __restrict__ partial,
                                                                  const float* __restrict__ bias,
                                                                  float* __restrict__ out, int splits, int Cp, int M,
                                                                  int total) {
  const int e = blockIdx.x * 256 + threadIdx.x;
  if (e >= total) return;
  float sum = bias != nullptr ? bias[e / M % Cp] : 0.0f;
  for (int s = 0; s < splits; s += 4) {
    float v[4];
#pragma unroll
    for (int x = 0; x < 4; ++x) v[x] = partial[(size_t)min(s + x, splits - 1) * total + e];
#pragma unroll
    for (int x = 0; x < 4; ++x) sum += s + x < splits ? v[x] : 0.0f;
  }
  out[e] = sum;
}

// W[n][c][k] as the A operands of the forward: [block of 32 n][step of 32 (k, c)][half step s]
// [piece][lane][16 bytes], lane l holding rows l % 32 and reduction elements 16 s + 8 (l / 32) + 0 .. 7
// (fp32: two pieces of four floats; bf16: one; split: the three pieces).
// The first `image_blocks` blocks lay the image out channels-last instead; one more writes the row of zeros.
struct PrepareArgs {
  const float* img;
  float* rows;
  const float* Wm;
  uint4* operands;
  int B, Cg, Cgp, HW, K, Cp, steps, total;
  int strips, chunks, image_blocks;   // 64 pixels, 32 channels
};

template <int MM>
__global__ __launch_bounds__(256) void columns_prepare_kernel(PrepareArgs g) {
  __shared__ float tile[32][65];
  int block = blockIdx.x;
  if (block < g.image_blocks) {
    const int strip = block % g.strips, chunk = block / g.strips % g.chunks, b = block / (g.strips * g.chunks);
    channels_last_tile(g.img + (size_t)b * g.Cg * g.HW, g.rows + (size_t)b * g.HW * g.Cgp, g.Cg, g.Cgp, g.HW,
                       64 * strip, 32 * chunk, tile);
    return;
  }
  block -= g.image_blocks;
  if (block == 0) {
    for (int i = threadIdx.x; i < g.Cgp; i += 256) g.rows[(size_t)g.B * g.HW * g.Cgp + i] = 0.0f;
    return;
  }
  const int e = (block - 1) * 256 + threadIdx.x;   // (block of rows, step, s, lane)
  if (e >= g.total) return;
  const int lane = e & 63, s = (e >> 6) & 1, q = e >> 7;
  const int n = q / g.steps * 32 + (lane & 31), r0 = (q % g.steps) * kDirectStep + 16 * s + 8 * (lane >> 5);
  const int k = r0 / g.Cgp, c = r0 - k * g.Cgp;   // (eight elements from a multiple of eight: one sample)
  const float* w = g.Wm + ((size_t)min(n, g.Cp - 1) * g.Cg) * g.K + min(k, g.K - 1);
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const float value = w[(size_t)min(c + i, g.Cg - 1) * g.K];
    f[i] = n < g.Cp && k < g.K && c + i < g.Cg ? value : 0.0f;
  }
  constexpr int kFrag = MM == kMmF32 ? 2 : (MM == kMmBf16 ? 1 : 3);
  uint4* out = g.operands + (size_t)(e >> 6) * kFrag * 64 + lane;
  if constexpr (MM == kMmF32) {
    out[0] = make_uint4(__float_as_uint(f[0]), __float_as_uint(f[1]), __float_as_uint(f[2]), __float_as_uint(f[3]));
    out[64] = make_uint4(__float_as_uint(f[4]), __float_as_uint(f[5]), __float_as_uint(f[6]), __float_as_uint(f[7]));
  } else if constexpr (MM == kMmBf16) {
    out[0] = __builtin_bit_cast(uint4, pack_bf16x8(f));
  } else {
    const Bf16Split p = split_bf16x8(f);
    out[0] = __builtin_bit_cast(uint4, p.hi);
    out[64] = __builtin_bit_cast(uint4, p.mid);
    out[128] = __builtin_bit_cast(uint4, p.lo);
  }
}

// Shape of a call.  Measured, us of the whole forward, on either side of each line:
//   blocks of 32 channels share a tile (the columns are blended once for all of them) up to five: 160 channels
//     of 6 x 25 x 50 pixels, split, 50 as 96 + 64, 37 as one tile; 256 channels of 60 x 120, nearest, bf16, 31 as
//     one tile of eight, 22 as two of four;
//   groups where the tiles leave SIMDs without a wave: 216 tiles of two blocks (104 -> 37 channels, 2 x 41 x 83)
//     39, 26 and 24 with 1, 2, 4; 384 of two (200 -> 37, 3 x 45 x 91, split) 60 and 47; 638 of three (8 -> 96,
//     101 x 202) 18.5 and 21.5; 1024 of two (64 -> 64, 128 x 256, bf16) 36, 41 and 55;
//   splits (another launch, and their sums through memory) where even that leaves CUs idle over a long
//     reduction: 72 tiles of four, 200 steps (256 -> 256, 5 x 5, 2 x 12 x 24, split) 126 and 48.
// Tiles of 64 pixels halve the weight operands read, not the time (64 -> 64, 128 x 256, float32, 46 and 46; 104 -> 37
// above 38 and 24).
struct DirectShape {
  int ra, groups, tiles_a, tiles_m, steps, splits, split_steps;
};
DirectShape direct_shape(const ConvGeom& g) {
  DirectShape t;
  const int64_t blocks = ceil_div(g.Cp, 32);
  t.tiles_a = (int)ceil_div(blocks, 5);
  t.ra = (int)ceil_div(blocks, t.tiles_a);
  t.tiles_m = (int)ceil_div(g.M, kDirectPixels);
  t.steps = (int)ceil_div((int64_t)g.K * pad8(g.Cg), kDirectStep);
  const int64_t tiles = (int64_t)t.tiles_a * t.tiles_m * g.B, waves = tiles * t.ra;
  int64_t splits = 1;
  if (tiles < 192 && t.steps >= 32) splits = std::min<int64_t>(384 / tiles, t.steps / 8);
  // (the sums take the place of the column matrix in the workspace)
  splits = std::max<int64_t>(1, std::min<int64_t>(splits, (int64_t)g.K * pad8(g.Cg) / g.Cp));
  t.split_steps = (int)ceil_div(t.steps, splits);
  t.splits = (int)ceil_div(t.steps, t.split_steps);
  t.groups = waves >= 1024 || t.splits > 1 ? 1 : (waves >= 512 ? 2 : 4);
  if (t.ra == 4) t.groups = std::min(t.groups, 2);
  if (t.ra == 5) t.groups = 1;
  return t;
}

}  // namespace

// (Maps with more points a sample would need a larger table of taps.)
bool columns_direct(const ConvGeom& g) { return pts(g.P) <= 4; }

size_t columns_operand_bytes(const ConvGeom& g) {
  const DirectShape t = direct_shape(g);
  return (size_t)t.tiles_a * t.ra * t.steps * 2 * 64 * 16 * 3;
}

int columns_direct_forward(const ConvGeom& g, int mm, const float* img, const float* map, const float* wts,
                           const float* Wm, const float* bias, float* pix, float* rows, void* operands,
                           float* partial, hipStream_t stream) {
  const DirectShape t = direct_shape(g);
  const int Cgp = pad8(g.Cg), HW = g.H * g.W;
  PrepareArgs p{};
  p.img = img;
  p.rows = rows;
  p.Wm = Wm;
  p.operands = static_cast<uint4*>(operands);
  p.B = (int)g.B;
  p.Cg = g.Cg;
  p.Cgp = Cgp;
  p.HW = HW;
  p.K = g.K;
  p.Cp = g.Cp;
  p.steps = t.steps;
  p.total = t.tiles_a * t.ra * t.steps * 2 * 64;
  p.strips = (int)ceil_div(HW, 64);
  p.chunks = (int)ceil_div(Cgp, 32);
  p.image_blocks = p.strips * p.chunks * (int)g.B;
  const dim3 pgrid((unsigned)(p.image_blocks + 1 + ceil_div(p.total, 256)));
  if (mm == kMmBf16) launch(columns_prepare_kernel<kMmBf16>, pgrid, dim3(256), stream, p);
  else if (mm == kMmSplit) launch(columns_prepare_kernel<kMmSplit>, pgrid, dim3(256), stream, p);
  else launch(columns_prepare_kernel<kMmF32>, pgrid, dim3(256), stream, p);
  SDK_LAUNCH_CHECK("mapped_conv(columns layouts)");

  DirectArgs a{};
  a.rows = rows;
  a.map = map;
  a.wts = wts;
  a.operands = static_cast<const char*>(operands);
  a.bias = bias;
  a.out = pix;
  a.B = (int)g.B;
  a.M = g.M;
  a.K = g.K;
  a.P = g.P;
  a.H = g.H;
  a.W = g.W;
  a.interp = g.interp;
  a.Cgp = Cgp;
  a.Cp = g.Cp;
  a.steps = t.steps;
  a.tiles_a = t.tiles_a;
  a.tiles_m = t.tiles_m;
  a.split_steps = t.split_steps;
  a.partial = t.splits > 1 ? partial : nullptr;
  const bool blended = g.interp == 1 || g.interp == 2, single = !blended && g.P == 0;
  // nine samples of a pixel in the table at a time; the five a step of 32 elements may touch, if each has
  // four taps a point
  a.cap = std::min(g.K, 9);
  if (g.P != 0) a.cap = std::max(a.cap, 5 * (int)ceil_div((int64_t)g.P * (blended ? 4 : 1), 4));
  const size_t tiles = (size_t)t.groups * 2 * kDirectPixels * row_bytes(mm) +
                       (size_t)(a.cap + 1) * kDirectPixels * (single ? 1 : 4) * 8;
  const size_t sums = (size_t)(t.groups - 1) * 16 * 64 * t.ra * 4;
  const size_t smem = std::max(tiles, sums);
  const dim3 grid((unsigned)(((int64_t)t.tiles_a * t.tiles_m * g.B + 7) / 8 * 8), (unsigned)t.splits);
  const dim3 block((unsigned)(64 * t.ra * t.groups));
#define CF3(MMv, RAv, Gv, NTv) columns_forward_kernel<MMv, RAv, Gv, NTv><<<grid, block, smem, stream>>>(a)
#define CF2(MMv, RAv, Gv)              \
  do {                                 \
    if (single) CF3(MMv, RAv, Gv, 1);  \
    else CF3(MMv, RAv, Gv, 4);         \
  } while (0)
#define CFG(MMv, RAv)                          \
  do {                                         \
    if (t.groups == 1) CF2(MMv, RAv, 1);       \
    else if (t.groups == 2) CF2(MMv, RAv, 2);  \
    else CF2(MMv, RAv, (RAv < 4 ? 4 : 2));     \
  } while (0)
#define CF1(MMv)                       \
  do {                                 \
    if (t.ra == 1) CFG(MMv, 1);        \
    else if (t.ra == 2) CFG(MMv, 2);   \
    else if (t.ra == 3) CFG(MMv, 3);   \
    else if (t.ra == 4) CFG(MMv, 4);   \
    else CF2(MMv, 5, 1);               \
  } while (0)
  if (mm == kMmBf16) CF1(kMmBf16);
  else if (mm == kMmSplit) CF1(kMmSplit);
  else CF1(kMmF32);
#undef CF1
#undef CFG
#undef CF2
#undef CF3
  SDK_LAUNCH_CHECK("mapped_conv(columns forward)");
  if (t.splits > 1) {
    const int total = (int)(g.B * g.Cp * g.M);
    launch(columns_forward_sum_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), stream,
           (const float*)partial, bias, pix, t.splits, g.Cp, g.M, total);
    SDK_LAUNCH_CHECK("mapped_conv(columns forward sums)");
  }
  return SDK_OK;
}

}  // namespace sdk
