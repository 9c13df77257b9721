// Weight gradient of mapped convolution from an LDS window, the columns of a quarter tile shared by the
// workgroup (gfx950, float32 tensors; fp32 MFMA, operands split into three bf16 pieces, or rounded to
// bf16):
//
//   gW[n][c][k] += sum_{b, m} pix[b][n][m] * col[b][(c, k)][m]
//   col[b][(c, k)][m] = sum_r coefficient(m, k, r) * img[b][c][tap(m, k, r)]
//
// for the tiles of a plan (conv_plan.hpp) whose taps lie inside the tile's window (or big window)
// and whose samples have at most four plan rows.
//
//   workgroup = 32 image channels (one chunk) x 32 A pixel-side channels x all K samples x one
//               batch element x every groups-th tile of the list
//
// A tile is taken a quarter (32 pixels) at a time.  The column values of a quarter are blended in
// float32 with a lane per pixel (16-byte window reads of neighbouring channels, a row decoded once
// for 16 channels) and left in LDS as [sample][pixel][channel].  So the work of building a quarter is
// shared by the waves and nothing is built twice, while every wave multiplies its own 32 rows of the
// pixel-side tensor, which it reads from memory straight into A operands (A = 2: rows 32 (w % 2) and
// half of the quarter's pixels).
//   bf16: the matrix unit wants the pixel as its reduction index, eight of them side by side in a
//   lane, and the transposing LDS read (ds_read_b64_tr_b16) takes them from there.  Quarter q + 1 is
//   built into one of two buffers between the MFMAs of quarter q: one barrier per quarter.
//   fp32: a step of v_mfma_f32_32x32x2_f32 wants one pixel of each half wave, a 4-byte read.  One
//   buffer, so that two workgroups share a CU; two barriers per quarter.  What bounds it: fp32 MFMAs
//   and vector instructions do not overlap on a SIMD (9 MFMAs 576 cycles, with 18, 36 and 72
//   multiply-adds of either of two waves 654, 723, 862), so the building costs its full time and is
//   worth sharing.
//   split: columns in LDS as for fp32, a lane's eight pixels of a sample split behind the read; bound
//   by that (three pieces stored would leave room for one workgroup).
//
// 8 x 128 x 256 x 512 -> 128, K = 9, four-tap samples (kernel times), tiles inside their window and
// big ones, against a kernel whose lanes owned a channel (a 4-byte window read and an address per tap
// and value, the plan rows of a pixel read from LDS by every lane, the last of nine samples built four
// times): bf16 1886 -> 944 us, 488 -> 249; fp32 2817 -> 2523 (1804 of them MFMAs), 612 -> 458; split
// 2480 -> 2154, 673 -> 436.
// bf16 without its global reads: 600; two workgroups per CU, all that 144 accumulator registers a wave
// allow, leave the rest of the reads' latency exposed.  bf16, eight waves in one workgroup for the
// inside tiles, with the window requested a tile ahead: 1507.  fp32: registers for a second copy of
// the pixel-side values, so that they too are requested before the MFMAs, spill: 2897; wave
// priorities for the building: 2545.
// One plan row a sample, the big tiles of 163842 1-rings of an icosphere, batch 4, 64 -> 64, fp32:
// 279 -> 170.
#pragma once
#include <hip/hip_runtime.h>

#include "conv_fused.hpp"
#include "conv_plan.hpp"
#include "conv_window.hpp"
#include "sdk_host.hpp"
#include "sdk_mfma.hpp"

namespace sdk {

namespace {

constexpr int kWvE = 36;     // floats per window element: 32 channels + 4 of skew
// bytes of one sample's column tile of a quarter: 32 pixels x 32 channels
constexpr int col_bytes(int mm) { return mm == kMmBf16 ? 2048 : 4096; }


// Byte of 16-byte piece q (8 channels) of pixel p in a column tile.  The pieces of each four
// pixels change places in a way of their own, so that equal pieces of the pixels that are written
// together lie in different banks (lanes 0..7 write pixels 0-3 and 16-19, see lane order below).
__device__ __forceinline__ unsigned col_at(int p, int q) {
  return (unsigned)(p * 64 + ((q ^ (((p >> 2) + (p >> 4)) & 3)) << 4));
}

// fp32: 16-byte piece q (4 channels) of pixel p.  Pixels p and p + 8, which a step reads together,
// lie side by side, in different halves of the banks.
__device__ __forceinline__ unsigned col32_at(int p, int q) {
  return (unsigned)(((p & 16) | ((p & 7) << 1) | ((p >> 3) & 1)) * 128 + ((q ^ (p & 7)) << 4));
}

// CAP: kRegionCap: the tiles of `list` lie inside their window; kBigCap: big tiles.
// NW: four waves, two workgroups per CU; eight waves, one workgroup per CU, where the LDS holds no
// second one (big tiles, ten samples): the second four then take the second half of the samples'
// MFMAs, and the registers that frees hold the next tile's window.
// A: row blocks of 32 pixel-side channels, 4, or 2 where there are at most 64.
// ROWS: plan rows per sample that are read and applied; 1 where the plan has no more (nearest taps
// without interpolation weights).
// FAR: planes of which 32 are more than a descriptor's 2^31 bytes; every lane forms its row's address,
// in kernels of their own: behind a branch the address costs registers that the sums of nine samples
// need.  32 -> 96 channels, 4096 x 4112 pixels, all of a backward call without the input's gradient,
// against the kernel that works from global memory: float32 17.2 -> 13.4 ms, bf16 11.6 -> 6.4, split
// 13.2 -> 10.8.
template <int MM, int K, int CAP, int NW, int A, int ROWS, bool FAR>
__global__ __launch_bounds__(64 * NW, 2) void window_wgrad_quarter_kernel(
    const float* __restrict__ pix, const float* __restrict__ img, const int* __restrict__ hdr,
    const int* __restrict__ ns, const int2* __restrict__ taps, const int* __restrict__ list,
    const int* __restrict__ count, float* __restrict__ partial, int Cg, int H, int W, int Cp,
    int S, PixelTiling pt, int groups, int batches, int c_chunks, int n_tiles, int vec4,
    const int* __restrict__ big_lut) {
  constexpr bool BIG = CAP > kRegionCap, WIDE = NW == 8;
  constexpr bool F32 = MM != kMmBf16;   // columns are left in LDS as they are
  constexpr int kColB = col_bytes(MM), BUFS = F32 ? 1 : 2;
  constexpr int STEPS = A == 4 ? 2 : 1;       // 16-pixel halves of a quarter that a wave multiplies
  constexpr int KA = WIDE ? (K + 1) / 2 : K;  // samples a wave multiplies
  constexpr int CW = kCC / NW;                // channels of a window that a wave stages
  constexpr int ITER = (CAP + 63) / 64;
  __shared__ __align__(16) float region[(CAP + 1) * kWvE];
  __shared__ __align__(16) char cols[BUFS * K * kColB];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int j = lane & 31, h = lane >> 5;
  // Workgroup ids go round-robin over the 8 XCDs.  All workgroups of one tile run (every
  // batch element and channel chunk) read the same plan rows, those of one batch element the
  // same pixel-side tiles: they take consecutive slots of one XCD and meet in its L2.
  const int kinds = c_chunks * n_tiles * batches;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;
  const int kind = slot % kinds, group = (slot / kinds) * 8 + xcd;
  if (group >= groups) return;
  const int cnt = *count;
  if (cnt == 0) return;   // (the summing kernel sees the same count and adds nothing)
  const int nt = kind % n_tiles, cc = (kind / n_tiles) % c_chunks;
  const int batch = kind / (n_tiles * c_chunks);
  const int n0 = nt * 128;
  const int M = pt.OH * pt.OW;
  const size_t HW = (size_t)H * W;
  const float* img_b = img + (size_t)batch * Cg * HW;
  const float* pix_b = pix + (size_t)batch * Cp * M;

  // MFMA role: rows 32 wc + j of the pixel-side tile, samples ka0 .. ka0 + KA - 1, pixels from
  // 16 s0 on
  const int wc = wave & (A - 1), ka0 = (wave >> 2) * KA, s0 = A == 2 ? (wave >> 1) & 1 : 0;
  // (rows past the last and pixels outside the grid read zero: past the end of the descriptor)
  const int wrow = __builtin_amdgcn_readfirstlane(min(n0 + 32 * wc, Cp - 1));
  const unsigned pix_bytes = __builtin_amdgcn_readfirstlane(
      (unsigned)max(0, min(32, Cp - (n0 + 32 * wc))) * (unsigned)M * 4u);
  const Rsrc pix_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(pix_b + (size_t)wrow * M), 0, (int)pix_bytes, 0x00020000);
  const unsigned pix_lane = (unsigned)j * (unsigned)M * 4u;
  floatx16 acc[KA];
#pragma unroll
  for (int k = 0; k < KA; ++k)
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[k][v] = 0.0f;
  // reading role.  bf16: row (l % 16) / 4 of four pixels, 8-byte part l % 4 of the 16 channels
  // 16 ((l / 16) % 2) ..; first and second four pixels of the lane's eight.  fp32: channel j of
  // the pixels 16 (s0 + s) + 8 h + i.
  unsigned rd[F32 ? 8 : 2 * STEPS];
  if constexpr (F32) {
#pragma unroll
    for (int i = 0; i < 8; ++i)
      rd[i] = ka0 * kColB + col32_at(16 * s0 + 8 * h + i, j >> 2) + 4 * (j & 3);
  } else {
#pragma unroll
    for (int s = 0; s < STEPS; ++s)
#pragma unroll
      for (int t = 0; t < 2; ++t) {
        const int p = 16 * (s0 + s) + 8 * h + 4 * t + ((lane & 15) >> 2);
        rd[2 * s + t] = col_at(p, 2 * ((lane >> 4) & 1) + ((lane & 3) >> 1)) + (lane & 1) * 8;
      }
  }
  const int pl = lane_pixel(j);   // building role
  // ---- pieces
  const int cw = min(cc * kCC + CW * wave, Cg - 1);   // first channel this wave stages
  const Rsrc img_rs = __builtin_amdgcn_make_buffer_rsrc(
      const_cast<float*>(img_b + (size_t)cw * HW), 0, min(CW, Cg - cw) * (int)(HW * 4u), 0x00020000);
  float wv[ITER][CW];
  int wo[ITER], RS = 0, RS_next = 0;
  // offsets of the window elements this lane stages
  auto fetch_offsets = [&](int tile_) {
    const int* lut = BIG ? big_lut + (size_t)tile_ * kBigStride : hdr + (size_t)tile_ * kHdrStride;
    RS_next = BIG ? min(lut[0], CAP) : lut[2] * lut[3];
#pragma unroll
    for (int it = 0; it < ITER; ++it)
      wo[it] = lut[(BIG ? kBigLut : kHdrLut) + min(lane + 64 * it, CAP - 1)];
  };
  auto fetch_window = [&]() {
    RS = RS_next;
    // Elements outside the image come from an offset past the descriptor's end: such reads
    // return zero.  (The sums of channels past the last are dropped, whatever they read.)
#pragma unroll
    for (int i = 0; i < CW; ++i) {
      const int ch = min(i, Cg - 1 - cw) * (int)(HW * 4u);
#pragma unroll
      for (int it = 0; it < ITER; ++it) {
        const unsigned o = lane + 64 * it < RS && wo[it] >= 0 ? (unsigned)wo[it] * 4u : 0x7ffffffcu;
        wv[it][i] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(img_rs, o, ch, 0));
      }
    }
  };
  auto store_window = [&]() {
#pragma unroll
    for (int it = 0; it < ITER; ++it) {
      const int e = lane + 64 * it;
      if (e < RS) {
        float4* d4 = reinterpret_cast<float4*>(region + e * kWvE + CW * wave);
#pragma unroll
        for (int i = 0; i < CW / 4; ++i)
          d4[i] = make_float4(wv[it][4 * i], wv[it][4 * i + 1], wv[it][4 * i + 2], wv[it][4 * i + 3]);
      }
    }
    if (tid < kWvE) region[RS * kWvE + tid] = 0.0f;   // the zero element inactive rows point at
  };
  // pixel-side values of quarter q_: fp32, 16 pixels a step
  u32x4 af[STEPS][2];
  auto fetch_pix = [&](int tile_, int q_) {
    const int ty0 = (tile_ / pt.tiles_x) * pt.TY(), tx0 = (tile_ % pt.tiles_x) << pt.tx_shift;
    constexpr unsigned kNone = 0xfffffff0u;
    if constexpr (FAR) {
      int row = n0 + 32 * wc + j, first = 32 * q_ + 16 * s0 + 8 * h;
      asm volatile("" : "+v"(row), "+v"(first));   // (addresses formed here, not kept from turn to turn)
      const float* base = pix_b + (size_t)min(row, Cp - 1) * M;
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
#pragma unroll
        for (int i = 0; i < 8; i += 4) {
          if (vec4) {
            const int p = first + 16 * s + i;
            const int y = ty0 + (p >> pt.tx_shift), x = tx0 + (p & (pt.TX() - 1));
            const bool on = row < Cp && y < pt.OH && x < pt.OW;
            const u32x4 v = *reinterpret_cast<const u32x4*>(base + (on ? (size_t)y * pt.OW + x : 0));
            af[s][i >> 2] = on ? v : u32x4(0);
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              const int p = first + 16 * s + i + e;
              const int y = ty0 + (p >> pt.tx_shift), x = tx0 + (p & (pt.TX() - 1));
              const bool on = row < Cp && y < pt.OH && x < pt.OW;
              const float v = base[on ? (size_t)y * pt.OW + x : 0];
              af[s][i >> 2][e] = on ? __float_as_uint(v) : 0u;
            }
          }
        }
      }
      return;
    }
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      const int p0 = 32 * q_ + 16 * (s0 + s) + 8 * h;
      const int oy = ty0 + (p0 >> pt.tx_shift), ox = tx0 + (p0 & (pt.TX() - 1));
      if (vec4) {
        const unsigned at = pix_lane + (unsigned)(oy * pt.OW + ox) * 4u;
#pragma unroll
        for (int i = 0; i < 2; ++i)
          af[s][i] = __builtin_amdgcn_raw_buffer_load_b128(
              pix_rs, oy < pt.OH && ox + 4 * i < pt.OW ? at + 16 * i : kNone, 0, 0);
      } else {
        int first = p0;
        asm volatile("" : "+v"(first));   // (addresses formed here, not kept from turn to turn)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
          const int p = first + i;
          const int y = ty0 + (p >> pt.tx_shift), x = tx0 + (p & (pt.TX() - 1));
          af[s][i >> 2][i & 3] = __builtin_amdgcn_raw_buffer_load_b32(
              pix_rs, y < pt.OH && x < pt.OW ? pix_lane + (unsigned)(y * pt.OW + x) * 4u : kNone, 0,
              0);
        }
      }
    }
  };
  auto pix_frag = [&](int s) {
    float f[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) f[i] = __uint_as_float(af[s][i >> 2][i & 3]);
    return pack_bf16x8(f);
  };
  // Units of building work: PX pixels of one sample, NC channels a lane.  A wave of four takes
  // samples 4 i + wave whole and eight pixels of each of the K % 4 last ones; a wave of eight the
  // half quarters 8 i + wave of all samples.
  constexpr int FULL = WIDE ? 0 : K / 4, PART = WIDE ? 0 : K % 4;
  constexpr int HALF = WIDE ? (2 * K + 7) / 8 : 0;
  constexpr int UNITS = FULL + PART + HALF;
  u32x2 rows[UNITS][ROWS];
  int n_rows[UNITS];
  auto unit_of = [&](int u, int& k, int& p, int& c) {   // sample, pixel of the quarter, first channel
    if (u < FULL) {
      k = 4 * u + wave;
      p = pl;
      c = 16 * h;
    } else if (u < FULL + PART) {
      k = 4 * FULL + (u - FULL);
      p = 8 * wave + (pl & 7);
      c = 4 * ((pl >> 3) + 4 * h);
    } else {
      const int x = 8 * (u - FULL - PART) + wave;
      k = min(x >> 1, K - 1);
      p = 16 * (x & 1) + (pl & 15);
      c = 8 * ((pl >> 4) + 2 * h);
    }
  };
  auto fetch_rows = [&](int tile_, int q_) {
    const Rsrc rs = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<int2*>(taps + (size_t)tile_ * K * S * 128), 0, 0x7fffffff, 0x00020000);
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      int k, p, c;
      unit_of(u, k, p, c);
      n_rows[u] = min(ns[(size_t)tile_ * K + k], ROWS);
#pragma unroll
      for (int r = 0; r < ROWS; ++r)
        rows[u][r] = __builtin_amdgcn_raw_buffer_load_b64(
            rs, p * 8, (k * S + min(r, S - 1)) * 1024 + q_ * 256, 0);
    }
  };
  auto build = [&](int buf) {
#pragma unroll
    for (int u = 0; u < UNITS; ++u) {
      int k, p, c;
      unit_of(u, k, p, c);
      if constexpr (F32) asm volatile("" : "+v"(p), "+v"(c));   // (addresses formed here, not kept)
      if (WIDE && 8 * u + wave >= 2 * K) break;
      __builtin_amdgcn_sched_barrier(0);
      const int nc = u < FULL ? 16 : (u < FULL + PART ? 4 : 8);
      const char* base = reinterpret_cast<const char*>(region) + 4 * c;
      float co[ROWS];
      unsigned at[ROWS];
#pragma unroll
      for (int r = 0; r < ROWS; ++r) {
        co[r] = r < n_rows[u] ? __uint_as_float(rows[u][r].y) : 0.0f;
        at[r] = __umul24(co[r] != 0.0f ? rows[u][r].x : (unsigned)RS, kWvE * 4u);
      }
      // (rows, channel block of eight) in turn, the reads of two turns ahead in flight
      constexpr int DEEP = 3;
      const int blocks = nc == 16 ? 2 : 1, turns = blocks * ROWS, q4 = nc == 4 ? 1 : 2;
      char* dst = cols + (buf * K + k) * kColB;
      float4 d[DEEP][2];
      float v[8];
      auto request = [&](int x) {
        const float4* rp =
            reinterpret_cast<const float4*>(base + at[x % ROWS] + 32 * (x / ROWS));
#pragma unroll
        for (int i = 0; i < 2; ++i)
          if (i < q4) d[x % DEEP][i] = rp[i];
      };
#pragma unroll
      for (int x = 0; x < DEEP - 1; ++x)
        if (x < turns) request(x);
#pragma unroll
      for (int x = 0; x < 2 * ROWS; ++x) {
        if (x < turns) {
          if (x + DEEP - 1 < turns) {
            request(x + DEEP - 1);
            asm volatile("" ::: "memory");
          }
          const int r = x % ROWS;
#pragma unroll
          for (int i = 0; i < 2; ++i) {
            if (i < q4) {
              const float4 t = d[x % DEEP][i];
              const float f[4] = {t.x, t.y, t.z, t.w};
#pragma unroll
              for (int y = 0; y < 4; ++y)
                v[4 * i + y] = r == 0 ? co[r] * f[y] : __builtin_fmaf(co[r], f[y], v[4 * i + y]);
            }
          }
          if (r == ROWS - 1) {
            if (F32) {
              const int piece = (c >> 2) + 2 * (x / ROWS);
#pragma unroll
              for (int i = 0; i < 2; ++i)
                if (i < q4)
                  *reinterpret_cast<float4*>(dst + col32_at(p, piece + i)) =
                      make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
            } else if (nc == 4) {
              u32x2 o;
              o.x = pack_bf16x2(v[0], v[1]);
              o.y = pack_bf16x2(v[2], v[3]);
              *reinterpret_cast<u32x2*>(dst + col_at(p, c >> 3) + ((c >> 2) & 1) * 8) = o;
            } else {
              u32x4 o;
              o.x = pack_bf16x2(v[0], v[1]);
              o.y = pack_bf16x2(v[2], v[3]);
              o.z = pack_bf16x2(v[4], v[5]);
              o.w = pack_bf16x2(v[6], v[7]);
              *reinterpret_cast<u32x4*>(dst + col_at(p, (c >> 3) + x / ROWS)) = o;
            }
          }
        }
      }
    }
  };
  // (the reads of a sample's operands stand behind the MFMAs of the sample before: the fences keep
  // the compiler from requesting all of them at once, which costs the registers of the sums)
  // kOdd: the second four of eight waves have one sample less
  constexpr bool kOdd = WIDE && K % 2 == 1;
  auto multiply16 = [&](int buf, const Bf16Frag (&a)[STEPS]) {
    if (kOdd && ka0 >= K) return;
    const char* src = cols + (buf * K + ka0) * kColB;
    Bf16Frag b[2][STEPS];
#pragma unroll
    for (int s = 0; s < STEPS; ++s) b[0][s] = tr_frag(src + rd[2 * s], src + rd[2 * s + 1]);
#pragma unroll
    for (int k = 0; k < KA; ++k) {
      if (WIDE && ka0 + k >= K) break;
      if (k + 1 < KA && !(kOdd && k + 2 == KA && ka0 != 0)) {
        const char* t = src + (k + 1) * kColB;
#pragma unroll
        for (int s = 0; s < STEPS; ++s)
          b[(k + 1) & 1][s] = tr_frag(t + rd[2 * s], t + rd[2 * s + 1]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int s = 0; s < STEPS; ++s) acc[k] = mfma_bf16(a[s], b[k & 1][s], acc[k]);
    }
    __builtin_amdgcn_sched_barrier(0);
  };
  // units of eight steps, the reads of a unit behind the MFMAs of the one before
  auto multiply32 = [&]() {
    Bf16Split a3[MM == kMmSplit ? STEPS : 1];
    if constexpr (MM == kMmSplit) {
#pragma unroll
      for (int s = 0; s < STEPS; ++s) {
        float f[8];
#pragma unroll
        for (int i = 0; i < 8; ++i) f[i] = __uint_as_float(af[s][i >> 2][i & 3]);
        a3[s] = split_bf16x8(f);
      }
    }
    if (kOdd && ka0 >= K) return;
    constexpr int UN = KA * STEPS;
    float b[2][8];
    auto request = [&](int x) {
#pragma unroll
      for (int i = 0; i < 8; ++i)
        b[x & 1][i] = *reinterpret_cast<const float*>(cols + rd[i % (F32 ? 8 : 1)] +
                                                      (x / STEPS) * kColB + (x % STEPS) * 2048);
    };
    request(0);
#pragma unroll
    for (int x = 0; x < UN; ++x) {
      if (WIDE && ka0 + x / STEPS >= K) break;
      if (x + 1 < UN && !(kOdd && (x + 1) / STEPS == KA - 1 && ka0 != 0)) request(x + 1);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (MM == kMmSplit) {
        acc[x / STEPS] = mfma_split(a3[x % STEPS], split_bf16x8(b[x & 1]), acc[x / STEPS]);
      } else {
#pragma unroll
        for (int i = 0; i < 8; ++i)
          acc[x / STEPS] = __builtin_amdgcn_mfma_f32_32x32x2f32(
              __uint_as_float(af[x % STEPS][i >> 2][i & 3]), b[x & 1][i], acc[x / STEPS], 0, 0, 0);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
  };

  // The workgroups of one XCD take neighbouring tiles of the list at the same time: their
  // windows share cache lines, which then meet in that XCD's L2.
  int ti = (group & 7) * (groups >> 3) + (group >> 3);
  // (one workgroup per CU: nothing else covers the window's reads, and the registers are there to
  // request it ahead; with two workgroups they are not)
  if (ti < cnt) {
    if (WIDE || F32) fetch_offsets(list[ti]);
    if (WIDE) fetch_window();
    if (F32) {
      fetch_rows(list[ti], 0);
      fetch_pix(list[ti], 0);
    }
  }
#pragma unroll 1
  for (; ti < cnt; ti += groups) {
    const int tile = list[ti];
    const bool has_next = ti + groups < cnt;
    const int tile_next = has_next ? list[ti + groups] : tile;
    // (every wave has built the last quarter of the previous tile: a barrier lies between)
    if (!WIDE) {
      if (!F32) fetch_offsets(tile);
      fetch_window();
    }
    if (!F32) {
      fetch_rows(tile, 0);
      fetch_pix(tile, 0);
    }
    store_window();
    __syncthreads();
    if constexpr (F32) {
#pragma unroll 1
      for (int q = 0; q < 4; ++q) {
        build(0);
        __syncthreads();
        // what the next quarter needs, of this tile or the next: its plan rows, answered while this
        // one's MFMAs run, and its pixel-side values, answered while its columns are built
        const int tile_q = q < 3 ? tile : tile_next, q_q = (q + 1) & 3;
        if (q == 2) fetch_offsets(tile_next);
        if (WIDE && q == 3) fetch_window();
        fetch_rows(tile_q, q_q);
        asm volatile("" ::: "memory");
        multiply32();
        fetch_pix(tile_q, q_q);
        asm volatile("" ::: "memory");
        if (q < 3) __syncthreads();   // (behind the last quarter stands the next window's)
      }
    } else {
      Bf16Frag a[STEPS];
#pragma unroll 1
      for (int q = 0; q < 4; ++q) {
        if (q > 0) {
#pragma unroll
          for (int s = 0; s < STEPS; ++s) a[s] = pix_frag(s);
          // this quarter's plan rows and pixel-side values, answered while the MFMAs of the one
          // before it run
          fetch_rows(tile, q);
          fetch_pix(tile, q);
          asm volatile("" ::: "memory");
          multiply16((q - 1) & 1, a);
        }
        build(q & 1);
        __syncthreads();
      }
#pragma unroll
      for (int s = 0; s < STEPS; ++s) a[s] = pix_frag(s);
      if (WIDE && has_next) {
        fetch_offsets(tile_next);
        fetch_window();
      }
      asm volatile("" ::: "memory");
      multiply16(1, a);
    }
  }

  // ---- every accumulator register is stored as it lies (register-major, thread fastest)
  float* dst = partial + (size_t)blockIdx.x * (K * 16 * 256) + ((wave & 3) * 64 + lane);
#pragma unroll
  for (int k = 0; k < KA; ++k) {
    if (WIDE && ka0 + k >= K) break;
#pragma unroll
    for (int v = 0; v < 16; ++v) dst[((ka0 + k) * 16 + v) * 256] = acc[k][v];
  }
}

}  // namespace

// The launch for one matrix arithmetic (an instantiation for each in a file of its own).
template <int MM>
int window_wgrad_quarter_launch(const ConvGeom& g, const Plan& plan, const int* list,
                                const int* count, bool big, const float* pix, const float* img,
                                float* partial, int groups, int c_chunks, int n_tiles,
                                int64_t slots, hipStream_t stream) {
  const dim3 grid((unsigned)slots);
  const int vec4 =
      (g.OW % 4 == 0 && plan.pt.TX() >= 8 && reinterpret_cast<uintptr_t>(pix) % 16 == 0) ? 1 : 0;
  const bool two = window_wgrad_blocks(g) == 2, one = plan.S == 1;
  const bool far = g.M > (1 << 24);
#define WW3(Kv, CAPv, NWv, Av, ROWSv, FARv)                                                     \
  launch(window_wgrad_quarter_kernel<MM, Kv, CAPv, NWv, Av, ROWSv, FARv>, grid, dim3(64 * NWv), stream, \
         pix, img, plan.hdr, plan.ns, plan.taps, list, count, partial, g.Cg, g.H, g.W, g.Cp,    \
         plan.S, plan.pt, groups, (int)g.B, c_chunks, n_tiles, vec4, plan.big_lut)
#define WW2(Kv, CAPv, NWv, Av)                                                                   \
  do {                                                                                           \
    if (far) WW3(Kv, CAPv, NWv, Av, 4, true);                                                    \
    else if (one) WW3(Kv, CAPv, NWv, Av, 1, false);                                              \
    else WW3(Kv, CAPv, NWv, Av, 4, false);                                                       \
  } while (0)
#define WW1(Kv, CAPv, NWv)                                                                       \
  do {                                                                                           \
    if (two) WW2(Kv, CAPv, NWv, 2); else WW2(Kv, CAPv, NWv, 4);                                  \
  } while (0)
#define WW(Kv)                                                                   \
  case Kv:                                                                       \
    if (big) WW1(Kv, kBigCap, 8); else WW1(Kv, kRegionCap, (Kv < 10 ? 4 : 8));   \
    break
  switch (g.K) {
    WW(1); WW(2); WW(3); WW(4); WW(5); WW(6); WW(7); WW(8); WW(9); WW(10);
    default: return fail(SDK_ERR_UNSUPPORTED, "window_wgrad: more than ten samples");
  }
#undef WW
#undef WW1
#undef WW2
#undef WW3
  SDK_LAUNCH_CHECK(big ? "window_wgrad(big)" : "window_wgrad");
  return SDK_OK;
}

}  // namespace sdk
