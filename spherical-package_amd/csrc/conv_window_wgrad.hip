// Weight gradient of mapped convolution from an LDS window: which layers take it, the launches and the
// sum over workgroups of what conv_window_wgrad_quarter.hpp leaves.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "conv_fused.hpp"
#include "conv_plan.hpp"
#include "conv_window.hpp"
#include "sdk_host.hpp"

namespace sdk {

namespace {

constexpr int kWwThreads = 256;

// Sums the accumulator copies of window_wgrad_quarter_kernel and adds them to gW.  Block (x, y, z):
// accumulator register x of thread threadIdx.x, for the workgroup kind y = (channel chunk,
// row tile), over every z-th of the batches * groups workgroups of that kind.  A: the row blocks
// of the summing kernel.
__global__ __launch_bounds__(kWwThreads) void window_wgrad_reduce_kernel(
    const float* __restrict__ partial, float* __restrict__ gW, int Cg, int Cp, int K, int A,
    int groups, int batches, int c_chunks, int n_tiles, const int* __restrict__ count) {
  if (*count == 0) return;   // nothing was summed
  const int tid = threadIdx.x, reg = blockIdx.x;
  const int nt = blockIdx.y % n_tiles, cc = blockIdx.y / n_tiles;
  const int kinds = c_chunks * n_tiles * batches;
  const int total = batches * groups;
  const size_t per_wg = (size_t)K * 16 * kWwThreads;
  // four reads in flight per thread (a plain loop waits for each in turn)
  auto at = [&](int i) {
    const int ic = min(i, total - 1);
    const int b = ic / groups, grp = ic % groups;
    const int kind = (b * c_chunks + cc) * n_tiles + nt;
    const size_t wg = ((size_t)(grp >> 3) * kinds + kind) * 8 + (grp & 7);
    const float v = partial[wg * per_wg + (size_t)reg * kWwThreads + tid];
    return i < total ? v : 0.0f;
  };
  float s0 = 0.0f, s1 = 0.0f, s2 = 0.0f, s3 = 0.0f;
  const int step = gridDim.z;
  for (int i = blockIdx.z; i < total; i += 4 * step) {
    const float v0 = at(i), v1 = at(i + step), v2 = at(i + 2 * step), v3 = at(i + 3 * step);
    s0 += v0;
    s1 += v1;
    s2 += v2;
    s3 += v3;
  }
  const float s = (s0 + s1) + (s2 + s3);
  const int wave = tid >> 6, lane = tid & 63, j = lane & 31, h = lane >> 5;
  const int v = reg & 15, k = reg >> 4, a = wave & (A - 1);
  const int n = nt * 128 + 32 * a + 8 * (v >> 2) + 4 * h + (v & 3);
  const int c = cc * kCC + j;
  if (c < Cg && n < Cp) atomic_add_noret(gW + (size_t)n * Cg * K + (size_t)c * K + k, s);
}

struct WwGrid {
  int c_chunks, n_tiles, groups, nreg;
  int64_t kinds, slots;
};
// big: the launch over the big tiles (one workgroup per CU).
WwGrid ww_grid(const ConvGeom& g, int tiles, bool big) {
  WwGrid w;
  w.c_chunks = (int)ceil_div(g.Cg, kCC);
  w.n_tiles = (int)ceil_div(g.Cp, 128);
  w.kinds = (int64_t)w.c_chunks * w.n_tiles * g.B;
  // tile runs: a multiple of 8 (one set per XCD), about two workgroups per CU overall (one
  // for the big windows)
  const int64_t want = std::max<int64_t>(8, ceil_div(ceil_div(big ? 256 : 512, w.kinds), 8) * 8);
  w.groups = (int)std::min<int64_t>(ceil_div(tiles, 8) * 8, want);
  // ten samples: one workgroup per CU (conv_window_wgrad_quarter.hpp), and what the last ones leave idle
  // counts: the runs of which up to three rounds of 256 workgroups take the fewest tiles one after
  // another (2 x 177 -> 209 channels, 172 x 346 pixels, one row a sample, float32: 24 runs of 21 tiles
  // in three rounds of which the last is a quarter full 2197 us, 32 runs of 16 in three full ones
  // 1683; four waves that built their own columns 1789)
  if (!big && g.K == 10) {
    auto in_turn = [&](int64_t n) { return ceil_div(n * w.kinds, 256) * ceil_div(tiles, n); };
    for (int64_t n = 8; n * w.kinds <= 768 && n <= ceil_div(tiles, 8) * 8; n += 8)
      if (in_turn(n) < in_turn(w.groups)) w.groups = (int)n;
  }
  w.slots = (int64_t)w.groups * w.kinds;
  w.nreg = g.K * 16;
  return w;
}
}  // namespace

bool window_wgrad_big_supported(const ConvGeom& g) {
  // (32-bit byte offsets over 32 planes of the image)
  return planned_wgrad_supported(g) && g.K >= 1 && g.K <= 10 && g.Cp >= 1 &&
         (int64_t)g.H * g.W <= ((int64_t)1 << 24);
}

bool window_wgrad_supported(const ConvGeom& g, int mm) {
  // (single-row plans and at most 64 rows: window_wgrad_narrow, whose operands are copies.  The
  // kernel that works from global memory, which took the other layers of at most 64 rows before, is
  // the slower one down to 8 rows and 8 channels.  9 samples, 256 x 512, batch 8, weight gradient in
  // us, there and here: 64 -> 64 float32 1627 / 953, split 1558 / 853, bf16 1248 / 508;
  // 128 -> 32 float32 2773 / 1800; 8 -> 16 float32 658 / 460; 220 x 440, batch 1, 48 -> 40 252 / 135)
  return window_wgrad_big_supported(g) && (g.Cp > 64 || !window_wgrad_narrow_supported(g, mm));
}

size_t window_wgrad_partial_bytes(const ConvGeom& g) {
  if (g.B == 0) return 0;
  // (one buffer serves whichever window kernels the call runs, one after the other)
  const size_t narrow =
      window_wgrad_narrow_supported(g, kMmF32) ? window_wgrad_narrow_partial_bytes(g) : 0;
  if (!window_wgrad_big_supported(g)) return narrow;
  const PixelTiling pt = plan_tiling(g.M / g.OW, g.OW);
  const int tiles = pt.tiles_x * pt.tiles_y;
  const WwGrid w = ww_grid(g, tiles, false), wb = ww_grid(g, tiles, true);
  return std::max(narrow,
                  (size_t)std::max(w.slots, wb.slots) * w.nreg * kWwThreads * sizeof(float));
}

int window_wgrad(const ConvGeom& g, int mm, const Plan& plan, const TileLists& tl,
                 const float* pix, const float* img, float* gW, float* partial,
                 hipStream_t stream, bool big) {
  if (big && plan.big_lut == nullptr) return SDK_OK;
  const WwGrid w = ww_grid(g, plan.tiles, big);
  const int* list = big ? tl.big : tl.inside;
  const int* count = big ? tl.count + 2 : tl.count;
  if (w.slots >= ((int64_t)1 << 31)) return fail(SDK_ERR_UNSUPPORTED, "window_wgrad: grid too large");
  const int rc = (mm == kMmBf16 ? window_wgrad16 : mm == kMmSplit ? window_wgrad_split
                                                                 : window_wgrad32)(
      g, plan, list, count, big, pix, img, partial, w.groups, w.c_chunks, w.n_tiles, w.slots, stream);
  if (rc) return rc;
  const int kinds0 = w.c_chunks * w.n_tiles, total = (int)g.B * w.groups;
  const int parts = (int)std::min<int64_t>(std::min(total, 16),
                                           ceil_div(2048, (int64_t)w.nreg * kinds0));
  launch(window_wgrad_reduce_kernel, dim3((unsigned)w.nreg, (unsigned)kinds0, (unsigned)std::max(parts, 1)),
         dim3(kWwThreads), stream, (const float*)partial, gW, g.Cg, g.Cp, g.K,
         window_wgrad_blocks(g), w.groups, (int)g.B, w.c_chunks, w.n_tiles, count);
  SDK_LAUNCH_CHECK("window_wgrad_reduce");
  return SDK_OK;
}

}  // namespace sdk
