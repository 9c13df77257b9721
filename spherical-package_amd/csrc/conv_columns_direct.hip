// Mapped convolution of small calls without a column matrix in front of the products:
//
//   forward          pix[b][n][m] = bias[n] + sum over (k, c) of W[n][c][k] * column(b, m, k, c)
//   weight gradient  gW[n][c][k] = sum over (b, m) of pix[b][n][m] * column(b, m, k, c)
//
// where column(b, m, k, :) is the blend of the image rows sample (m, k) falls between
// (ext_modules/src/cpp/mapped_convolution_layer.cpp:8-60 writes it out first).  The image is
// channels-last (conv_columns.hip), so a tap is one run of channels; the columns of a tile are
// blended on the way to LDS, 32 pixels x 32 (k, c) at a time, and multiplied from there.  And the
// first half of a scatter, whose columns are its products:
//
//   col[b][m][(k, c)] = sum over n of pix[b][n][m] * W[n][c][k]
//
// Every other operand is laid out beforehand in the form the MFMAs read, rounded or split there once, by one launch
// a call (columns_prepare_kernel), which also sums the pixels for the bias gradient.
//
// Whole forward, us, with the columns written to memory and read back -> so: 64 -> 64, 1 x 128 x 256, float32
// 60 -> 47; 96 -> 160, 6 x 50 x 100, stride 2, split 52 -> 37; 104 -> 37, 2 x 41 x 83, float32 46 -> 23; 200 -> 37,
// 3 x 45 x 91, split 82 -> 47; 256 -> 256, 5 x 5, 2 x 24 x 48, stride 2, split 149 -> 45; 24 -> 32, 2 x 115 x 231,
// float32 50 -> 27.  Forward and backward of the same:
// 206 -> 156, 170 -> 124, 130 -> 87, 251 -> 171, 264 -> 125, 177 -> 114.
// A tile's 32 pixels are of one batch element, so a grid of fewer is padded; it is still the faster way: backward,
// float32, 4096 x 2 x 2 pixels, 16 -> 16 908 -> 104, 1024 x 2 x 4, 64 -> 64 468 -> 108, 4096 of one pixel, 64 -> 256,
// nine samples 1704 -> 1152, one sample 1663 -> 259.
// What bounds it: in float32 the MFMAs (half of the forward at 64 -> 64) and the vector
// instructions of the blend, which do not overlap them; in the others the blend, and the reads of operands and
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
// (columns_prepare_kernel).  The reads of a step are made before the MFMAs of the step before it.
//
// The taps of `cap` samples of every pixel of the tile fit the table at a time; the reduction is
// walked in runs of steps whose samples do.  Unused slots and steps past the end point at a row
// of zeros behind the image, with coefficient zero.  (A sample of more than four taps, possible in
// weighted maps, takes several entries of the table.)
typedef float floatx4 __attribute__((ext_vector_type(4)));
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
  int tiles_a, tiles_n;     // tiles_n: of pixels of a batch element; weight gradient: of columns (k, c)
  int splits, strips;       // strips: steps of 32 pixels of a batch element
  int cap;
  int split_steps;          // steps of one split; more than one split: sums without bias to `partial`
  float* partial;
};

template <bool WGRAD, int MM, int RA, int G, int NT>
__global__ __launch_bounds__(64 * RA * G, (RA > 1 && (MM != kMmSplit || (RA > 3 && !WGRAD)) ? 3 : 2)) void columns_direct_kernel(DirectArgs g) {
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

  // an eighth of the tiles, neighbours in the picture, per XCD (ids go round-robin over them); the column tiles
  // of a run of pixels together
  const int total = g.tiles_a * g.tiles_n * (WGRAD ? g.splits : g.B);
  const int slot = (blockIdx.x & 7) * (gridDim.x >> 3) + (blockIdx.x >> 3);
  if (slot >= total) return;
  const int ta = slot % g.tiles_a, tn = slot / g.tiles_a % g.tiles_n, tz = slot / (g.tiles_a * g.tiles_n);
  const int b = WGRAD ? 0 : tz, split = WGRAD ? tz : blockIdx.y;
  const int m0 = tn * BN;                                  // forward: first pixel
  const int r0 = tn * 32, R = g.K * g.Cgp;                 // weight gradient: first column
  const int kf = r0 / g.Cgp, nk = WGRAD ? min(g.K - 1, (r0 + 31) / g.Cgp) - kf + 1 : 1;   // ... and its samples
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

  // pixel m (past the last: not one) and sample k of table entry e (taps e of the run that starts at step t0,
  // sample k0) at pixel px of its 32, and the image rows before its batch element's
  struct Place {
    int m, k, base;
  };
  auto place = [&](int t0, int k0, int e, int px) {
    if constexpr (WGRAD) {
      const int t = t0 + e / nk, z = t / g.strips;
      return Place{(t - z * g.strips) * 32 + px, kf + e % nk, z * HW};
    } else {
      return Place{m0 + px, k0 + e, 0};
    }
  };
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
  const int t_begin = split * g.split_steps, t_end = min(t_begin + g.split_steps, g.steps);
  // entries a sample takes: one, until a run finds a weighted sample of more taps
  int each = 1;
  if (NT == 4 && g.P != 0 && threadIdx.x == 0) s_most = 0;

  // Forward: the even and the odd turns of a single group are summed apart, as two groups' are (864 products a
  // sum, 96 -> 160: 3.2e-7 off float64 in the norm so, 4.5e-7 in one chain).  Weight gradient: its reduction is
  // hundreds of pixels, so one turn at a time (split operands: two) is summed apart and then added, sum[1] the sums.
  // Distance from float64, 1e-7 of the norm, with 1, 2, 4 turns and all of a split in a chain: 96 -> 160, 7500 pixels,
  // float32 1.6, 1.7, 2.2, 5.5, split 1.9, 1.8, 2.0, 4.9; 8 -> 8, 86 thousand pixels, float32 1.6, 1.9, 2.3, 2.3,
  // split 4.0, 3.2, 3.2, 3.2.  Wide layers of few splits have longer chains of turns, and the tile kernels longer ones
  // yet (their distance in brackets): 5 x 5, 200 -> 160, 100 x 200, one split of 625 turns, float32 4.6 (6.4), split
  // 3.7 (6.0); 256 -> 160, 128 x 256, 1024 turns, 5.9 (8.2), 4.6 (8.1); 32 -> 32, 8 x 256 x 512, 3.8 (6.8), 9.4 (19).
  constexpr int kAlone = MM == kMmSplit ? 2 : 1;
  constexpr bool kTwo = WGRAD || G == 1;
  int done = 0;
  floatx16 sum[kTwo ? 2 : 1] = {};

  const int quad = tid & 7, px0 = tid >> 3;
  constexpr int kRowStep = GT / 8;   // pixels between a thread's samples
  const char* frag = g.operands + ((size_t)(ta * RA + wave) * g.steps * 2 * kFrag * 64 + lane) * 16;
  const int tile0 = group * 2 * BN * RB;   // (of lds: the group's two buffers)

  vec4 v[DEEP][NI][NT];   // samples on their way, and their entry and channel
  int at_e[DEEP], at_c[DEEP];
  uint4 a_next[2 * kFrag];
  int t0 = t_begin;
  while (t0 < t_end) {
    // ---- a run: steps t0 .. t1 - 1, samples k0 .. k0 + samples - 1
    const int samples = g.cap / each;
    const int k0 = WGRAD ? 0 : t0 * kDirectStep / g.Cgp;
    const int run = max(1, samples / nk);   // (whole turns where there are any)
    const int t1 = WGRAD ? min(t_end, t0 + (run > G ? run - run % G : run))
                         : min(t_end, k0 + samples >= g.K ? g.steps : max(t0 + 1, (k0 + samples) * g.Cgp / kDirectStep));
    __syncthreads();   // the run before is done with the table
    const int held = WGRAD ? min(samples, (t1 - t0) * nk) : min(samples, g.K - k0);
    if (g.P == 0) {
      // (four samples at a time: their coordinates are requested together)
      for (int i0 = threadIdx.x; i0 < BN * held; i0 += 4 * kThreads) {
        float2 at[4];
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = min(i0 + u * kThreads, BN * held - 1);
          const Place p = place(t0, k0, i / BN, i % BN);
          // (a map is aligned to its floats)
          __builtin_memcpy(&at[u], g.map + 2 * ((size_t)min(p.m, g.M - 1) * g.K + p.k), 8);
        }
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int i = i0 + u * kThreads;
          if (i >= BN * held) break;
          const Place p = place(t0, k0, i / BN, i % BN);
          const bool inside = p.m < g.M;
          auto write = [&](auto tag) {
            constexpr int INTERP = decltype(tag)::value;
            PointTaps<float, INTERP> t;
            t.set(at[u].x, at[u].y, g.H, g.W);
            if constexpr (NT == 1) {
              s_off[i] = inside && t.off[0] >= 0 ? (p.base + t.off[0]) * g.Cgp * 4 : zero_at;
            } else {
              ivec4 off;
              vec4 co;
#pragma unroll
              for (int x = 0; x < 4; ++x) {
                const bool on = inside && t.off[x] >= 0;   // (a weight of zero has no offset)
                off[x] = on ? (p.base + t.off[x]) * g.Cgp * 4 : zero_at;
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
      int most = 0;
      for (int i = threadIdx.x; i < BN * held; i += kThreads) {
        const int px = i % BN, e = i / BN;
        int* off = s_off + (e * each * BN + px) * NT;
        float* co = s_co + (e * each * BN + px) * NT;
        int n = 0;
        const Place p = place(t0, k0, e, px);
        if (p.m < g.M)
          n = taps(p.m, p.k, [&](int at, int o, float c) {
            if (at >= NT * each) return;
            const int x = (at / NT) * BN * NT + at % NT;
            off[x] = (p.base + o) * g.Cgp * 4;
            co[x] = c;
          });
        most = max(most, n);
        for (; n < NT * each; ++n) {
          const int x = (n / NT) * BN * NT + n % NT;
          off[x] = zero_at;
          co[x] = 0.0f;
        }
      }
      if (most > NT * each) atomicMax(&s_most, most);
    }
    __syncthreads();
    if (NT == 4 && g.P != 0) {
      const int needed = (s_most + NT - 1) / NT;
      if (needed > each) {   // (the same for every thread: the run again, shorter and with room for all taps)
        each = needed;
        continue;
      }
    }

    // this thread's samples.  Forward: reduction element 32 t + 4 quad = (k, c), 32 G further each turn; weight
    // gradient: column r0 + 4 quad = (kf + k, c) of the pixels 32 t ..
    int t = t0 + group;
    const int at0 = WGRAD ? r0 + 4 * quad : t * kDirectStep + 4 * quad;
    int k = at0 / g.Cgp, c = at0 - k * g.Cgp;
    k -= WGRAD ? kf : k0;
    const int dk = kDirectStep * G / g.Cgp, dc = kDirectStep * G - dk * g.Cgp;
    auto fetch = [&](int st) {
      const int e = WGRAD ? (t - t0) * nk + k : k;
      at_e[st] = t < t1 && (WGRAD ? at0 < R : true) && e < held ? e * each : g.cap;
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
      vec4 blend[NI];
      auto place_of = [&](int i) { return NI * GT == 8 * BN ? px0 + i * kRowStep : min(px0 + i * kRowStep, BN - 1); };
      if constexpr (NT == 4) {
        auto add = [&](int e, bool first) {
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const vec4 w = *reinterpret_cast<const vec4*>(s_co + (e * BN + place_of(i)) * 4);
#pragma unroll
            for (int x = 0; x < 4; ++x) {
              float f = first ? w[0] * v[st][i][0][x] : __builtin_fmaf(w[0], v[st][i][0][x], blend[i][x]);
              f = __builtin_fmaf(w[1], v[st][i][1][x], f);
              f = __builtin_fmaf(w[2], v[st][i][2][x], f);
              blend[i][x] = __builtin_fmaf(w[3], v[st][i][3][x], f);
            }
          }
        };
        add(at_e[st], true);
        for (int q = 1; q < each; ++q) {   // (more taps than four: read here, those of all samples together)
          const int e = min(at_e[st] + q, g.cap);
#pragma unroll
          for (int i = 0; i < NI; ++i) {
            const ivec4 o = *reinterpret_cast<const ivec4*>(s_off + (e * BN + place_of(i)) * 4);
#pragma unroll
            for (int x = 0; x < 4; ++x)
              v[st][i][x] = *reinterpret_cast<const vec4*>(rows_b + (unsigned)(o[x] + at_c[st]));
          }
          __builtin_amdgcn_sched_barrier(0);
          add(e, false);
        }
      } else {
#pragma unroll
        for (int i = 0; i < NI; ++i) blend[i] = v[st][i][0];
      }
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        const int px = px0 + i * kRowStep;
        if (NI * GT != 8 * BN && px >= BN) break;
        const vec4 s = blend[i];
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
      if constexpr (!WGRAD) {
        k += dk;
        c += dc;
        if (c >= g.Cgp) {
          c -= g.Cgp;
          ++k;
        }
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
      floatx16& acc = sum[kTwo && !WGRAD ? kBuf : 0];
      if (WGRAD && done++ % kAlone == 0) {
        sum[kTwo ? 1 : 0] += acc;
        acc = floatx16{};
      }
      if (now < t1) {   // (the last turn of a run may have no step left for this group)
#pragma unroll
        for (int s = 0; s < 2; ++s) {
          const char* row = src + j * RB;
          if constexpr (MM == kMmF32) {
            vec4 lo, hi;
            if constexpr (WGRAD) {   // column j of pixels 16 s + 8 h ..
#pragma unroll
              for (int e = 0; e < 4; ++e) {
                lo[e] = *reinterpret_cast<const float*>(src + (16 * s + 8 * h + e) * RB + 4 * j);
                hi[e] = *reinterpret_cast<const float*>(src + (16 * s + 8 * h + 4 + e) * RB + 4 * j);
              }
            } else {
              lo = *reinterpret_cast<const vec4*>(row + 64 * s + 32 * h);
              hi = *reinterpret_cast<const vec4*>(row + 64 * s + 32 * h + 16);
            }
            const vec4 al = __builtin_bit_cast(vec4, a[2 * s]), ah = __builtin_bit_cast(vec4, a[2 * s + 1]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(al[e], lo[e], acc, 0, 0, 0);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(ah[e], hi[e], acc, 0, 0, 0);
          } else {
            auto weights = [&](int q) { return __builtin_bit_cast(Bf16Frag, a[kFrag * s + q]); };
            auto columns = [&](int q) {
              if constexpr (WGRAD) {
                const char* at = src + (16 * s + 8 * h + ((lane & 15) >> 2)) * RB + 64 * q + 32 * ((lane >> 4) & 1) +
                                 8 * (lane & 3);
                return tr_frag(at, at + 4 * RB);
              } else {
                return __builtin_bit_cast(Bf16Frag, *reinterpret_cast<const uint4*>(row + 64 * q + 32 * s + 16 * h));
              }
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
  if constexpr (kTwo) acc += sum[1];
  if constexpr (G > 1) {
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
  if constexpr (WGRAD) {
    float* out = g.partial + (size_t)split * g.Cp * R;
#pragma unroll
    for (int x = 0; x < 16; ++x) {
      const int n = 32 * RA * ta + 32 * wave + 8 * (x >> 2) + 4 * h + (x & 3);
      if (n < g.Cp && r0 + j < R) out[(size_t)n * R + r0 + j] = acc[x];
    }
    return;
  }
  const bool whole = g.partial == nullptr;
  float* out = (whole ? g.out : g.partial + (size_t)split * g.B * g.Cp * g.M) + (size_t)b * g.Cp * g.M;
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

// gW[n][c][k] = (or, `add`, +=) sum over the splits of partial[split][n][k][c]; the last blocks, four channels each,
// sum the bias gradient gb[n] = sum of strip_sums[n][strip].
__global__ __launch_bounds__(256) void columns_gradient_sum_kernel(const float* __restrict__ partial,
                                                                   float* __restrict__ gW, int splits, int Cg, int Cgp,
                                                                   int K, int Cp, int total, int weight_blocks,
                                                                   const float* __restrict__ strip_sums,
                                                                   float* __restrict__ gb, int strips, int add) {
  if ((int)blockIdx.x >= weight_blocks) {
    const int n = ((int)blockIdx.x - weight_blocks) * 4 + (threadIdx.x >> 6), lane = threadIdx.x & 63;
    if (n >= Cp) return;
    double sum = 0.0;   // (up to 64 strips a lane: in float32 1.8e-7 off float64 with 4096 strips, so 0.7e-7)
    for (int s = lane; s < strips; s += 256) {
      float v[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) v[x] = strip_sums[(size_t)n * strips + min(s + 64 * x, strips - 1)];
#pragma unroll
      for (int x = 0; x < 4; ++x) sum += s + 64 * x < strips ? v[x] : 0.0f;
    }
    for (int off = 32; off > 0; off >>= 1) sum += __shfl_down(sum, off, 64);
    if (lane == 0) gb[n] = (float)sum;
    return;
  }
  const int e = blockIdx.x * 256 + threadIdx.x;   // (n, k, c), c fastest
  if (e >= total) return;
  const int c = e % Cgp, q = e / Cgp, k = q % K, n = q / K;
  if (c >= Cg) return;
  float sum = 0.f;
  for (int s = 0; s < splits; s += 8) {
    float v[8];
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = partial[(size_t)min(s + x, splits - 1) * total + e];
#pragma unroll
    for (int x = 0; x < 8; ++x) v[x] = s + x < splits ? v[x] : 0.0f;
    sum += ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
  }
  float* out = gW + ((size_t)n * Cg + c) * K + k;
  *out = add ? *out + sum : sum;
}

// col[b][m][r] = sum over n of pix[b][n][m] * W[n][r], r = (k, c): a wave makes 32 pixels x 64 columns from operands
// read as they lie (L2 and vector cache; nothing goes through LDS, no wave waits for another), those of 16 channels
// n requested before the MFMAs of the 16 before them.  LONG: 64 channels at a time are summed apart.
struct ProductArgs {
  const char *pixels, *weights;   // operands: [block of 32 pixels][n / 16], [block of 32 columns][n / 16]
  float* col;
  int M, R, strips, tiles_r, tiles, steps;   // strips, steps: blocks of an element, steps of a block
};
template <int MM, bool LONG>
__global__ __launch_bounds__(256, 2) void columns_product_kernel(ProductArgs g) {
  constexpr int kFrag = MM == kMmF32 ? 2 : (MM == kMmBf16 ? 1 : 3);
  // an eighth of the tiles per XCD; its waves take them in turn, the column tiles of a block of pixels together
  const int share = (g.tiles + 7) / 8, first = (blockIdx.x & 7) * share, last = min(first + share, g.tiles);
  const int waves = (gridDim.x >> 3) * 4;
  int tile = first + (blockIdx.x >> 3) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (tile >= last) return;
  const int lane = threadIdx.x & 63, j = lane & 31, h = lane >> 5;
  const size_t block = (size_t)g.steps * kFrag * 1024;
  uint4 a[kFrag], w[2][kFrag];
  auto fetch = [&](int tile, int s) {
    const int tr = tile % g.tiles_r, tm = tile / g.tiles_r;
    const char* pa = g.pixels + (size_t)tm * block + s * (kFrag * 1024) + lane * 16;
    // (past the last block of columns: that one again, nothing of it is stored)
    const char* pb = g.weights + (size_t)(2 * tr) * block + s * (kFrag * 1024) + lane * 16;
    const size_t next = min(2 * tr + 1, (g.R - 1) / 32) == 2 * tr ? 0 : block;
#pragma unroll
    for (int p = 0; p < kFrag; ++p) {
      a[p] = *reinterpret_cast<const uint4*>(pa + p * 1024);
      w[0][p] = *reinterpret_cast<const uint4*>(pb + p * 1024);
      w[1][p] = *reinterpret_cast<const uint4*>(pb + next + p * 1024);
    }
  };
  fetch(tile, 0);
  while (tile < last) {
    const int next = tile + waves;
    floatx16 all[2] = {}, acc[2] = {};
    for (int s = 0; s < g.steps; ++s) {
      if (LONG && (s & 3) == 0) {
#pragma unroll
        for (int x = 0; x < 2; ++x) {
          all[x] += acc[x];
          acc[x] = floatx16{};
        }
      }
      uint4 ah[kFrag], wh[2][kFrag];
#pragma unroll
      for (int p = 0; p < kFrag; ++p) {
        ah[p] = a[p];
#pragma unroll
        for (int x = 0; x < 2; ++x) wh[x][p] = w[x][p];
      }
      // (behind the last step the next tile's first; behind the last tile this one's again)
      const bool more = s + 1 < g.steps;
      fetch(more || next >= last ? tile : next, more ? s + 1 : 0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        auto piece = [](const uint4& v) { return __builtin_bit_cast(Bf16Frag, v); };
        if constexpr (MM == kMmF32) {
#pragma unroll
          for (int p = 0; p < 2; ++p) {
            const floatx4 u = __builtin_bit_cast(floatx4, ah[p]), v = __builtin_bit_cast(floatx4, wh[x][p]);
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[x] = __builtin_amdgcn_mfma_f32_32x32x2f32(u[e], v[e], acc[x], 0, 0, 0);
          }
        } else if constexpr (MM == kMmBf16) {
          acc[x] = mfma_bf16(piece(ah[0]), piece(wh[x][0]), acc[x]);
        } else {
          const Bf16Split u = {piece(ah[0]), piece(ah[1]), piece(ah[2])};
          const Bf16Split v = {piece(wh[x][0]), piece(wh[x][1]), piece(wh[x][2])};
          acc[x] = mfma_split(u, v, acc[x]);
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    const int tr = tile % g.tiles_r, tm = tile / g.tiles_r;
    const int b = tm / g.strips, strip = tm - b * g.strips;
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      if (LONG) acc[x] += all[x];
      const int r = 64 * tr + 32 * x + j;
      float* out = g.col + ((size_t)b * g.M + 32 * strip + 4 * h) * g.R + r;
      if (r < g.R) {
        if (32 * strip + 32 <= g.M) {
#pragma unroll
          for (int v = 0; v < 16; ++v) out[(size_t)(8 * (v >> 2) + (v & 3)) * g.R] = acc[x][v];
        } else {
#pragma unroll
          for (int v = 0; v < 16; ++v) {
            const int dm = 8 * (v >> 2) + (v & 3);
            if (32 * strip + 4 * h + dm < g.M) out[(size_t)dm * g.R] = acc[x][v];
          }
        }
      }
    }
    tile = next;
  }
}

// ---------------------------------------------------------------------------
// What a call lays out before its products, in one launch.
//   image   [b][u][c], and a row of zeros behind the last
//   weights as operands: of the forward [block of 32 n][step of 32 (k, c)][s], of the product, one chunk of channels
//           after the other, [block of 32 (k, c)][step of 16 n]
//   pixels  as operands: of the weight gradient [block of 32 n][step of 32 pixels][s], of the product
//           [block of 32 pixels][step of 16 n], and their sums over each 64 pixels of a channel
// An operand of 16 reduction elements is [piece][lane][16 bytes], lane l holding row (or column) l % 32 and elements
// 8 (l / 32) + 0 .. 7 (fp32: two pieces of four floats; bf16: one; split: the three pieces).
// ---------------------------------------------------------------------------
struct PrepareArgs {
  const float *img, *Wm, *pix;
  float* rows;
  uint4 *weights, *pix_rows, *pix_cols;   // pix_rows: of the weight gradient; pix_cols: of the product
  float* strip_sums;
  int B, Cg, Cgp, HW, K, Cp, M;
  int pix_B, pix_first;                   // elements of the batch whose pixels are laid out, and the first
  int steps;                              // of the weights' blocks
  int product_weights;                    // channels of a chunk of the product's weights; 0: the forward's
  int img_strips, img_chunks, img_blocks;      // 64 pixels, 32 channels
  int pix_strips, pix_chunks, pix_blocks;
  int total;                              // operands of the weights times 64 lanes
};

template <int MM>
__device__ __forceinline__ void put_operand(uint4* dst, size_t operand, int lane, const float (&f)[8]) {
  constexpr int kFrag = MM == kMmF32 ? 2 : (MM == kMmBf16 ? 1 : 3);
  uint4* out = dst + operand * kFrag * 64 + lane;
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

template <int MM>
__global__ __launch_bounds__(256) void columns_prepare_kernel(PrepareArgs g) {
  __shared__ float tile[32][65];
  __shared__ float part[32][9];
  int block = blockIdx.x;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int j = lane & 31, h = lane >> 5;
  if (block < g.img_blocks) {
    const int strip = block % g.img_strips, q = block / g.img_strips, chunk = q % g.img_chunks, b = q / g.img_chunks;
    channels_last_tile(g.img + (size_t)b * g.Cg * g.HW, g.rows + (size_t)b * g.HW * g.Cgp, g.Cg, g.Cgp, g.HW,
                       64 * strip, 32 * chunk, tile);
    return;
  }
  block -= g.img_blocks;
  if (block < g.pix_blocks) {
    // 32 channels of 64 pixels
    const int strip = block % g.pix_strips, q = block / g.pix_strips, chunk = q % g.pix_chunks, b = q / g.pix_chunks;
    const float* src = g.pix + (size_t)(g.pix_first + b) * g.Cp * g.M;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const int n = 32 * chunk + wave + 4 * i, m = 64 * strip + lane;
      const float v = src[(size_t)min(n, g.Cp - 1) * g.M + min(m, g.M - 1)];
      tile[wave + 4 * i][lane] = n < g.Cp && m < g.M ? v : 0.0f;
    }
    __syncthreads();
    const int steps = (g.M + 31) / 32;             // of a batch element
    float f[8];
    {   // channels x pixels: step wave / 2 of the two, half wave % 2
      const int step = 2 * strip + (wave >> 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = tile[j][16 * wave + 8 * h + i];
      if (g.pix_rows != nullptr && step < steps)
        put_operand<MM>(g.pix_rows, (((size_t)chunk * g.pix_B + b) * steps + step) * 2 + (wave & 1), lane, f);
      if (g.strip_sums != nullptr)
        part[j][2 * wave + h] = ((f[0] + f[1]) + (f[2] + f[3])) + ((f[4] + f[5]) + (f[6] + f[7]));
    }
    if (g.pix_cols != nullptr) {   // pixels x channels: block wave / 2 of the two, half wave % 2 of the channels
      const int at = 2 * strip + (wave >> 1);
#pragma unroll
      for (int i = 0; i < 8; ++i) f[i] = tile[16 * (wave & 1) + 8 * h + i][32 * (wave >> 1) + j];
      const int of = (g.Cp + 15) / 16, n16 = 2 * chunk + (wave & 1);
      if (at < steps && n16 < of) put_operand<MM>(g.pix_cols, ((size_t)b * steps + at) * of + n16, lane, f);
    }
    if (g.strip_sums != nullptr) {
      __syncthreads();
      const int n = 32 * chunk + (int)threadIdx.x;
      if (threadIdx.x < 32 && n < g.Cp) {
        const float* p = part[threadIdx.x];
        g.strip_sums[((size_t)n * g.B + g.pix_first + b) * g.pix_strips + strip] =
            ((p[0] + p[1]) + (p[2] + p[3])) + ((p[4] + p[5]) + (p[6] + p[7]));
      }
    }
    return;
  }
  block -= g.pix_blocks;
  if (block == 0) {
    if (g.rows != nullptr)
      for (int i = threadIdx.x; i < g.Cgp; i += 256) g.rows[(size_t)g.B * g.HW * g.Cgp + i] = 0.0f;
    return;
  }
  const int e = (block - 1) * 256 + threadIdx.x;   // (operand, lane)
  if (e >= g.total) return;
  float f[8];
  if (g.product_weights) {
    const int s = e / 64 % g.steps, r = e / 64 / g.steps * 32 + j, n0 = 16 * s + 8 * h;
    const int chunk = min(r / (g.K * g.product_weights), (g.Cgp - 1) / g.product_weights);
    const int c0 = chunk * g.product_weights, width = min(g.product_weights, g.Cgp - c0);
    const int k = (r - g.K * c0) / width, c = c0 + (r - g.K * c0) - k * width;
    const float* w = g.Wm + (size_t)min(c, g.Cg - 1) * g.K + min(k, g.K - 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float value = w[(size_t)min(n0 + i, g.Cp - 1) * g.Cg * g.K];
      f[i] = n0 + i < g.Cp && k < g.K && c < g.Cg ? value : 0.0f;
    }
  } else {
    const int s = (e >> 6) & 1, q = e >> 7;
    const int n = q / g.steps * 32 + j, r = (q % g.steps) * kDirectStep + 16 * s + 8 * h;
    const int k = r / g.Cgp, c = r - k * g.Cgp;   // (eight elements from a multiple of eight: one sample)
    const float* w = g.Wm + ((size_t)min(n, g.Cp - 1) * g.Cg) * g.K + min(k, g.K - 1);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
      const float value = w[(size_t)min(c + i, g.Cg - 1) * g.K];
      f[i] = n < g.Cp && k < g.K && c + i < g.Cg ? value : 0.0f;
    }
  }
  put_operand<MM>(g.weights, (size_t)(e >> 6), lane, f);
}

// Shape of a call.  Measured, us of the whole forward, on either side of each line:
//   blocks of 32 channels share a tile (the columns are blended once for all of them), up to five: 160 channels
//     of 6 x 25 x 50 pixels, split, 50 as 96 + 64, 37 as one tile; 256 channels of 60 x 120, nearest, bf16, 31 as
//     one tile of eight, 22 as two of four.  More are tiles of four, the last perhaps of padding: three or five waves
//     share four SIMDs badly.  Forward alone, us, float32 / bf16 / split, as equal tiles of three or five and so:
//     19 -> 176 channels, 188 x 376 106 / 56 / 102 and 109 / 50 / 80 (float32 as three of two 90; 176 -> 176,
//     4 x 24 x 49 78, 75 and 52 so); 32 -> 264, 3 x 62 x 125 87 / 40 / 74 and 72 / 33 / 53; 32 -> 291, 136 x 272
//     126 / 57 / 118 and 106 / 45 / 77.  Nine, a third of them padding so, stay two of five and four where the products
//     are long and not split: 72 -> 264, 62 x 125 54 / 23 / 49 and 55 / 25 / 42; 75 -> 280, 7 x 32 x 65, bf16 27 and 30.
//     Five blocks whose columns
//     are quickly multiplied are two tiles of four where they are split: 48 -> 160, 2 x 54 x 108 36 and 30, 24 -> 160,
//     7 x 60 x 121 75 and 62; 96 -> 160 above 33 and 33, 216 -> 152, 2 x 56 x 112 112 and 123;
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
DirectShape direct_shape(const ConvGeom& g, int mm) {
  DirectShape t;
  const int64_t blocks = ceil_div(g.Cp, 32);
  t.tiles_m = (int)ceil_div(g.M, kDirectPixels);
  t.steps = (int)ceil_div((int64_t)g.K * pad8(g.Cg), kDirectStep);
  if (blocks <= 4 || (blocks == 5 && (mm != kMmSplit || t.steps >= 24))) t.ra = (int)blocks;
  else if (blocks == 9 && mm != kMmSplit && t.steps >= 20) t.ra = 5;
  else t.ra = blocks == 6 && mm == kMmF32 ? 2 : 4;
  t.tiles_a = (int)ceil_div(blocks, t.ra);
  // (splits by the columns' tiles of up to five blocks: the sums' chains do not grow with the tiles of four)
  const int64_t waves = (int64_t)t.tiles_a * t.tiles_m * g.B * t.ra, tiles = ceil_div(blocks, 5) * t.tiles_m * g.B;
  int64_t splits = 1;
  if (tiles < 192 && t.steps >= 32) splits = std::min<int64_t>(384 / tiles, t.steps / 8);
  splits = std::max<int64_t>(1, splits);
  t.split_steps = (int)ceil_div(t.steps, splits);
  t.splits = (int)ceil_div(t.steps, t.split_steps);
  t.groups = waves >= 1024 || t.splits > 1 ? 1 : (waves >= 512 ? 2 : 4);
  if (t.ra == 4) t.groups = std::min(t.groups, 2);
  if (t.ra == 5) t.groups = 1;
  return t;
}

// The weight gradient's: tiles of 32 columns (k, c) and of at most five blocks of 32 channels, the pixels in
// splits of at least four turns.  Its kernel alone, us, with 1024, 2048 and 4096 waves: 160 rows (one tile of five
// blocks: one workgroup a CU; 1536, where some CUs have two, 54), 6 x 25 x 50, 96 -> 160, split 31, 35, 42; 64 rows,
// 128 x 256, 64 -> 64, float32 68, 61, 47; 37 rows, 3 x 45 x 91, split 67, 65, 51; 128 rows, 4 x 40 x 80, split 55,
// 45, 42; 32 rows, 2 x 115 x 231, 24 -> 32, float32 42, 26, 31.  One tile of five blocks for each of 129 to 255 column
// tiles is one split, and leaves CUs idle: 5 x 5, 256 -> 160, 48 x 96 (200), backward, float32 / bf16 / split, 405 / 177
// / 297 (tile kernels 1182 / 600 / 861); 512 -> 160, 3 x 3, 2 x 40 x 80 (144) 468 / 189 / 327 (549 / 264 / 422).
// More than five blocks are tiles of four, the last perhaps of padding; nine and ten of bf16 operands two of five where
// there are few columns and so several splits, float32 ones of a sample (32 -> 280, 3 x 88 x 177 103 and 112).  Whole
// backward, float32 / bf16 / split, as equal tiles of three or five and of four: 176 -> 176, 4 x 24 x 49 141 / 86 / 113
// and 127 / 69 / 105; 128 -> 184, 3 x 45 x 91 226 / 121 / 173 and 206 / 92 / 163; 32 -> 291, 136 x 272 265 / 113 / 212
// and 251 / 107 / 222; 56 -> 264, 49 x 99 85 / 49 / 63 and 85 / 51 / 69; 211 -> 272, 5 x 5, 2 x 19 x 36 245 / 122 / 185
// and 180 / 99 / 148.
struct WgradShape {
  int ra, groups, tiles_a, tiles_r, strips, steps, most, splits, split_steps, samples;   // samples: most of a tile
};
WgradShape wgrad_shape(const ConvGeom& g, int mm, int64_t elements) {   // (most: splits of so many or fewer)
  WgradShape t;
  const int64_t blocks = ceil_div(g.Cp, 32);
  t.tiles_r = (int)ceil_div((int64_t)g.K * pad8(g.Cg), 32);
  if (blocks <= 5) t.ra = (int)blocks;
  else t.ra = (blocks == 9 || blocks == 10) && t.tiles_r <= (mm == kMmF32 ? 2 : 64) ? 5 : 4;
  t.tiles_a = (int)ceil_div(blocks, t.ra);
  t.groups = t.ra == 1 ? 4 : (t.ra <= 3 ? 2 : 1);
  t.strips = (int)ceil_div(g.M, 32);
  t.samples = pad8(g.Cg) % 32 == 0 ? 1 : std::min(g.K, pad8(g.Cg) == 8 ? 4 : 2);
  t.steps = (int)(elements * t.strips);
  const int64_t waves = (int64_t)t.tiles_a * t.tiles_r * t.ra * t.groups;
  const int64_t wanted = t.ra == 5 ? 256 / ((int64_t)t.tiles_a * t.tiles_r) : ceil_div(t.ra == 1 ? 2048 : 4096, waves);
  const int64_t splits = std::max<int64_t>(1, std::min<int64_t>(wanted, t.steps / (4 * t.groups)));
  t.most = (int)splits;
  t.split_steps = (int)ceil_div(t.steps, splits);
  t.splits = (int)ceil_div(t.steps, t.split_steps);
  return t;
}

// 16-byte pieces of an operand
int operand_pieces(int mm) { return mm == kMmF32 ? 2 : (mm == kMmBf16 ? 1 : 3); }
// 64-pixel strips of the pixel-side tensor
int64_t pixel_strips(const ConvGeom& g) { return ceil_div(g.M, 64); }

PrepareArgs prepare_args(const ConvGeom& g) {
  PrepareArgs p{};
  p.B = (int)g.B;
  p.Cg = g.Cg;
  p.Cgp = pad8(g.Cg);
  p.HW = g.H * g.W;
  p.K = g.K;
  p.Cp = g.Cp;
  p.M = g.M;
  return p;
}
void prepare_image(PrepareArgs& p, const float* img, float* rows) {
  p.img = img;
  p.rows = rows;
  p.img_strips = (int)ceil_div(p.HW, 64);
  p.img_chunks = (int)ceil_div(p.Cgp, 32);
  p.img_blocks = p.img_strips * p.img_chunks * p.B;
}
void prepare_weights(PrepareArgs& p, const float* Wm, void* weights, int product, int blocks, int steps) {
  p.Wm = Wm;
  p.weights = static_cast<uint4*>(weights);
  p.product_weights = product;
  p.steps = steps;
  p.total = blocks * steps * (product ? 64 : 128);
}
void prepare_pixels(PrepareArgs& p, const float* pix, int64_t first, int64_t elements, void* rows, void* cols,
                    float* strip_sums) {
  p.pix = pix;
  p.pix_first = (int)first;
  p.pix_B = (int)elements;
  p.pix_rows = static_cast<uint4*>(rows);
  p.pix_cols = static_cast<uint4*>(cols);
  p.strip_sums = strip_sums;
  p.pix_strips = (int)ceil_div(p.M, 64);
  p.pix_chunks = (int)ceil_div(p.Cp, 32);
  p.pix_blocks = p.pix_strips * p.pix_chunks * p.pix_B;
}
int prepare(int mm, const PrepareArgs& p, hipStream_t stream) {
  const dim3 grid((unsigned)(p.img_blocks + p.pix_blocks + 1 + ceil_div(p.total, 256)));
  if (mm == kMmBf16) launch(columns_prepare_kernel<kMmBf16>, grid, dim3(256), stream, p);
  else if (mm == kMmSplit) launch(columns_prepare_kernel<kMmSplit>, grid, dim3(256), stream, p);
  else launch(columns_prepare_kernel<kMmF32>, grid, dim3(256), stream, p);
  SDK_LAUNCH_CHECK("mapped_conv(columns layouts)");
  return SDK_OK;
}

// The kernel of a shape.
template <bool WGRAD>
int direct(const ConvGeom& g, int mm, DirectArgs a, int ra, int groups, int samples, dim3 grid,
           hipStream_t stream) {
  const bool blended = g.interp == 1 || g.interp == 2, single = !blended && g.P == 0;
  // samples of a pixel in the table at a time: nine in the forward, those of a split of the weight gradient up to 40
  // (a run's start costs a wait for the map and one for the image); at least those a step of 32 elements may
  // touch, if each has four taps a point
  const size_t rows = (size_t)groups * 2 * kDirectPixels * row_bytes(mm);
  const size_t entry = (size_t)kDirectPixels * (single ? 1 : 4) * 8;
  const int fit = (int)((80 * 1024 - 1024 - rows) / entry) - 1;   // half a CU's LDS
  a.cap = std::min(WGRAD ? std::min(40, std::max(4, a.split_steps * samples)) : std::min(g.K, 9), std::max(fit, 9));
  if (g.P != 0) a.cap = std::max(a.cap, (WGRAD ? 4 : 5) * (int)ceil_div((int64_t)g.P * (blended ? 4 : 1), 4));
  const size_t tiles = rows + (a.cap + 1) * entry;
  const size_t sums = (size_t)(groups - 1) * 16 * 64 * ra * 4;
  const size_t smem = std::max(tiles, sums);
  const dim3 block((unsigned)(64 * ra * groups));
  hipError_t reserved = hipSuccess;
#define CF3(MMv, RAv, Gv, NTv)                                                                                \
  do {                                                                                                        \
    const auto kernel = columns_direct_kernel<WGRAD, MMv, RAv, Gv, NTv>;                                      \
    if (smem > 65536)                                                                                         \
      reserved = hipFuncSetAttribute(reinterpret_cast<const void*>(kernel),                                   \
                                     hipFuncAttributeMaxDynamicSharedMemorySize, (int)smem);                  \
    if (reserved == hipSuccess) kernel<<<grid, block, smem, stream>>>(a);                                     \
  } while (0)
#define CF2(MMv, RAv, Gv)              \
  do {                                 \
    if (single) CF3(MMv, RAv, Gv, 1);  \
    else CF3(MMv, RAv, Gv, 4);         \
  } while (0)
#define CFG(MMv, RAv)                                                                       \
  do {                                                                                      \
    if constexpr (WGRAD) CF2(MMv, RAv, (RAv == 1 ? 4 : (RAv <= 3 ? 2 : 1)));                \
    else if (groups == 1) CF2(MMv, RAv, 1);                                                 \
    else if (groups == 2) CF2(MMv, RAv, 2);                                                 \
    else CF2(MMv, RAv, (RAv < 4 ? 4 : 2));                                                  \
  } while (0)
#define CF1(MMv)                      \
  do {                                \
    if (ra == 1) CFG(MMv, 1);         \
    else if (ra == 2) CFG(MMv, 2);    \
    else if (ra == 3) CFG(MMv, 3);    \
    else if (ra == 4) CFG(MMv, 4);    \
    else CF2(MMv, 5, 1);              \
  } while (0)
  if (mm == kMmBf16) CF1(kMmBf16);
  else if (mm == kMmSplit) CF1(kMmSplit);
  else CF1(kMmF32);
#undef CF1
#undef CFG
#undef CF2
#undef CF3
  if (reserved != hipSuccess)
    return fail(SDK_ERR_DEVICE, "mapped_conv(columns direct): cannot reserve %zu bytes of LDS: %s", smem,
                hipGetErrorString(reserved));
  SDK_LAUNCH_CHECK("mapped_conv(columns direct)");
  return SDK_OK;
}

DirectArgs direct_args(const ConvGeom& g, const float* rows, const float* map, const float* wts, const void* operands) {
  DirectArgs a{};
  a.rows = rows;
  a.map = map;
  a.wts = wts;
  a.operands = static_cast<const char*>(operands);
  a.B = (int)g.B;
  a.M = g.M;
  a.K = g.K;
  a.P = g.P;
  a.H = g.H;
  a.W = g.W;
  a.interp = g.interp;
  a.Cgp = pad8(g.Cg);
  a.Cp = g.Cp;
  a.strips = (int)ceil_div(g.M, 32);
  return a;
}

}  // namespace

// Samples of several points.  The line is drawn for points on pixels, a tap each: the four nearest pixels with weights
// of their own, and vertices.  Between pixels a blended point has four, of which the first of a sample are read ahead and
// the others turn by turn; the host cannot tell the two.  us of the columns in memory and of these, float32 / bf16 /
// split, forward and backward:
//   1 x 128 x 256, 64 -> 64   four pixels 217 / 180 / 206 and 174 / 124 / 166   two points between 241 / 204 / 235 and
//                             219 / 176 / 222   four between 313 / 276 / 300 and 303 / 262 / 315   six, split, 361 and
//                             484   eight 470 and 648
//   2 x 48 x 96, 96 -> 96     four pixels 176 / 127 / 154 and 150 / 106 / 138   two between 193 / 145 / 172 and
//                             191 / 159 / 186   four between 234 / 186 / 213 and 252 / 227 / 255
// Over 180 drawn calls each, median: forward 0.72 / 0.70 / 0.71 on pixels, 0.90 / 0.98 / 0.92 with two points between,
// 1.00 / 1.12 / 1.07 with four; backward 0.77 / 0.70 / 0.78, 0.85 / 0.79 / 0.86, 0.89 / 0.87 / 0.94.  (The worst are
// forwards of eight channels: twice the time with four points between pixels.)
bool columns_direct(const ConvGeom& g) { return pts(g.P) <= 4; }

// One sample of few channels at many pixels of a wide layer: a tile of the forward is over after a step or two, and
// the pixels, laid out twice at four or six bytes a value, are most of the backward.  us, columns in memory and so,
// float32 / bf16 / split:
//   forward   8 -> 64   50 / 32 / 42 and 42 / 40 / 53      48 -> 64   78 / 64 / 72 and 64 / 57 / 73    4 x 181 x 363
//             8 -> 128  46 / 28 / 39 and 38 / 30 / 39      32 -> 128  55 / 39 / 48 and 42 / 35 / 44    2 x 181 x 363
//             8 -> 232  52 / 29 / 42 and 44 / 34 / 44      40 -> 232  60 / 38 / 51 and 60 / 41 / 56    2 x 147 x 290
//   backward 16 -> 64  189 / 165 / 178 and 197 / 159 / 230  96 -> 64  376 / 342 / 359 and 365 / 298 / 388
//            24 -> 128 152 / 130 / 144 and 170 / 119 / 182  64 -> 232 170 / 146 / 163 and 190 / 121 / 207
// With a quarter of the pixels (17 MB) all of these are the faster ones.
static bool one_sample_of_wide_pixels(const ConvGeom& g, int most_channels, size_t pixel_bytes) {
  return g.K == 1 && pad8(g.Cg) <= most_channels && g.Cp >= 64 && sizeof(float) * g.B * g.M * g.Cp >= pixel_bytes;
}
bool columns_direct_gather(const ConvGeom& g, int mm) {
  // (whole tiles of four waves, one a SIMD: 32 -> 128, split, 48 and 44; single taps: 16 -> 243, 4 x 159 x 316, nearest,
  // bf16 / split 56 / 85 and 51 / 72)
  const bool four = ceil_div(g.Cp, 32) % 4 == 0, single = g.interp == 0 && g.P == 0;
  const int most = mm == kMmF32 || single ? 0 : (mm == kMmSplit ? (four ? 8 : 48) : std::min(48, (g.Cp - 1) / 4));
  return columns_direct(g) && !one_sample_of_wide_pixels(g, most, (size_t)32 << 20);
}
bool columns_direct_backward(const ConvGeom& g, int mm) {
  const int most = mm == kMmF32 ? 64 : (mm == kMmSplit ? 96 : 0);
  return columns_direct(g) && !one_sample_of_wide_pixels(g, most, (size_t)54 << 20);
}

size_t columns_weight_bytes(const ConvGeom& g, int mm) {
  const DirectShape t = direct_shape(g, mm);
  const int64_t forward = (int64_t)t.tiles_a * t.ra * t.steps * 2;
  const int64_t product = ceil_div((int64_t)g.K * pad8(g.Cg), 32) * ceil_div(g.Cp, 16);
  return (size_t)std::max(forward, product) * 64 * 16 * operand_pieces(mm);
}
size_t columns_forward_sum_bytes(const ConvGeom& g, int mm) {
  const DirectShape t = direct_shape(g, mm);
  return t.splits > 1 ? sizeof(float) * t.splits * g.B * g.Cp * g.M : 0;
}
size_t columns_pixel_row_bytes(const ConvGeom& g, int mm, int64_t elements) {
  const WgradShape t = wgrad_shape(g, mm, elements);
  return (size_t)t.tiles_a * t.ra * t.steps * 2 * 64 * 16 * operand_pieces(mm);
}
size_t columns_pixel_column_bytes(const ConvGeom& g, int mm, int64_t elements) {
  return (size_t)(elements * ceil_div(g.M, 32) * ceil_div(g.Cp, 16)) * 64 * 16 * operand_pieces(mm);
}
size_t columns_partial_bytes(const ConvGeom& g, int mm, int64_t elements) {
  return (size_t)wgrad_shape(g, mm, elements).most * g.Cp * g.K * pad8(g.Cg) * sizeof(float);
}
size_t columns_strip_bytes(const ConvGeom& g) { return (size_t)g.B * pixel_strips(g) * g.Cp * sizeof(float); }

int columns_direct_forward(const ConvGeom& g, int mm, const float* img, const float* map, const float* wts,
                           const float* Wm, const float* bias, float* pix, const ColumnsScratch& s,
                           hipStream_t stream) {
  const DirectShape t = direct_shape(g, mm);
  PrepareArgs p = prepare_args(g);
  prepare_image(p, img, s.img_rows);
  prepare_weights(p, Wm, s.weights, 0, t.tiles_a * t.ra, t.steps);
  int rc = prepare(mm, p, stream);
  if (rc) return rc;
  DirectArgs a = direct_args(g, s.img_rows, map, wts, s.weights);
  a.bias = bias;
  a.out = pix;
  a.steps = t.steps;
  a.tiles_a = t.tiles_a;
  a.tiles_n = t.tiles_m;
  a.splits = t.splits;
  a.split_steps = t.split_steps;
  a.partial = t.splits > 1 ? s.partial : nullptr;
  const dim3 grid((unsigned)(((int64_t)t.tiles_a * t.tiles_m * g.B + 7) / 8 * 8), (unsigned)t.splits);
  rc = direct<false>(g, mm, a, t.ra, t.groups, 1, grid, stream);
  if (rc) return rc;
  if (t.splits > 1) {
    const int total = (int)(g.B * g.Cp * g.M);
    launch(columns_forward_sum_kernel, dim3((unsigned)ceil_div(total, 256)), dim3(256), stream,
           (const float*)s.partial, bias, pix, t.splits, g.Cp, g.M, total);
    SDK_LAUNCH_CHECK("mapped_conv(columns forward sums)");
  }
  return SDK_OK;
}

int columns_direct_prepare(const ConvGeom& g, int mm, const float* pix, int64_t first, int64_t elements, bool rows,
                           bool cols, bool strip_sums, const float* Wm, int channels, const float* img,
                           const ColumnsScratch& s, hipStream_t stream) {
  PrepareArgs p = prepare_args(g);
  if (img != nullptr) prepare_image(p, img, s.img_rows);
  if (Wm != nullptr)
    prepare_weights(p, Wm, s.weights, channels, (int)ceil_div((int64_t)g.K * pad8(g.Cg), 32), (int)ceil_div(g.Cp, 16));
  prepare_pixels(p, pix, first, elements, rows ? s.pix_rows : nullptr, cols ? s.pix_cols : nullptr,
                 strip_sums ? s.strip_sums : nullptr);
  return prepare(mm, p, stream);
}

int columns_direct_product(const ConvGeom& g, int mm, int64_t first, int64_t elements, int c0, int channels,
                           const ColumnsScratch& s, hipStream_t stream) {
  const int R = g.K * channels;
  const int pieces = operand_pieces(mm), steps = (int)ceil_div(g.Cp, 16);
  ProductArgs a{};
  a.weights = static_cast<const char*>(s.weights) + (size_t)c0 * g.K / 32 * steps * pieces * 1024;
  a.col = s.col;
  a.M = g.M;
  a.R = R;
  a.strips = (int)ceil_div(g.M, 32);
  a.tiles_r = (int)ceil_div(R, 64);
  const int64_t tiles = elements * a.strips * a.tiles_r;
  a.tiles = (int)tiles;
  a.steps = steps;
  a.pixels = static_cast<const char*>(s.pix_cols) + (size_t)first * a.strips * steps * pieces * 1024;
  // float32: one wave a SIMD.  With two or more, their loads and MFMAs take turns: 64 -> 64, 128 x 256, 33 us with
  // one, 53 with four (21 without the MFMAs, 30 without the loads); MFMAs alone run at
  // 150 TFLOP/s with any number of waves, 16 of them beside six 16-byte loads at 130 with one and 70 with two.  bf16 operands want
  // the waves: 256 -> 128, 60 x 120, bf16, 27 us with two a SIMD, 22 with four.
  const int groups = mm == kMmF32 ? 32 : 128;
  const dim3 grid((unsigned)(8 * std::min<int64_t>(ceil_div(tiles, 32), groups)));
#define CP(MMv)                                                                                     \
  do {                                                                                              \
    if (a.steps > 4) launch(columns_product_kernel<MMv, true>, grid, dim3(256), stream, a);         \
    else launch(columns_product_kernel<MMv, false>, grid, dim3(256), stream, a);                    \
  } while (0)
  if (mm == kMmBf16) CP(kMmBf16);
  else if (mm == kMmSplit) CP(kMmSplit);
  else CP(kMmF32);
#undef CP
  SDK_LAUNCH_CHECK("mapped_conv(columns product)");
  return SDK_OK;
}

int columns_direct_wgrad(const ConvGeom& g, int mm, const float* pix, const float* map, const float* wts,
                         const float* img, float* gW, int64_t slice, const ColumnsScratch& s, bool prepared, float* gb,
                         hipStream_t stream) {
  const int Cgp = pad8(g.Cg), total = g.Cp * g.K * Cgp, weight_blocks = (int)ceil_div(total, 256);
  for (int64_t first = 0; first < g.B; first += slice) {
    const int64_t elements = std::min<int64_t>(slice, g.B - first);
    if (!prepared) {
      const int rc = columns_direct_prepare(g, mm, pix, first, elements, true, false, gb != nullptr, nullptr,
                                            0, first == 0 ? img : nullptr, s, stream);
      if (rc) return rc;
    }
    const WgradShape t = wgrad_shape(g, mm, elements);
    DirectArgs a = direct_args(g, s.img_rows + (size_t)first * g.H * g.W * Cgp, map, wts, s.pix_rows);
    a.B = (int)(g.B - first);   // (where the row of zeros is)
    a.steps = t.steps;
    a.tiles_a = t.tiles_a;
    a.tiles_n = t.tiles_r;
    a.splits = t.splits;
    a.split_steps = t.split_steps;
    a.partial = s.partial;
    const dim3 grid((unsigned)(((int64_t)t.tiles_a * t.tiles_r * t.splits + 7) / 8 * 8));
    const int rc = direct<true>(g, mm, a, t.ra, t.groups, t.samples, grid, stream);
    if (rc) return rc;
    // (the strips of all slices are there with the last)
    const int bias_blocks = gb != nullptr && first + elements == g.B ? (int)ceil_div(g.Cp, 4) : 0;
    launch(columns_gradient_sum_kernel, dim3((unsigned)(weight_blocks + bias_blocks)), dim3(256), stream,
           (const float*)s.partial, gW, t.splits, g.Cg, Cgp, g.K, g.Cp, total, weight_blocks,
           (const float*)s.strip_sums, gb, (int)(g.B * pixel_strips(g)), first > 0 ? 1 : 0);
    SDK_LAUNCH_CHECK("mapped_conv(columns sums)");
  }
  return SDK_OK;
}

}  // namespace sdk
