// Voting resample: integer labels scattered through an integer sample map; every output pixel
// keeps the label most of its sources carry.  Reference: votes with 64-bit atomic adds into a
// [C, OH, OW, candidates] int64 histogram per batch element, then argmax over the last axis
// (ext_modules/include/core/interpolation.h:249-265, core/resample.h:163-172,
// common/resample.h:109-130, src/cpp/voting_resample_layer.cpp:8-37).  Here the histogram is a
// caller-provided workspace of 32-bit counters (a pixel cannot collect 2^31 votes), reused
// pass after pass for as many batch elements as it holds; the first label with the most votes wins,
// label 0 where nobody voted.  Where the map is coherent the histogram never leaves LDS (below).
// With more than one channel the reference's histograms overlap (its channel offset lacks the
// factor `candidates`); label images have one channel, and the overlap is reproduced as it is.
#include <hip/hip_runtime.h>

#include <algorithm>

#include "sdk_host.hpp"
#include "sdk_lane_runs.hpp"

namespace sdk {

constexpr int kVoteBlock = 256;

// ---------------------------------------------------------------------------------------------
// Coherent maps: neighbouring pixels vote for neighbouring cells.  vote_boxes_kernel leaves, per
// tile of 16 x 16 input pixels, the box of the cells its pixels vote for; a workgroup of
// vote_tile_kernel owns a tile of output cells, finds the input tiles whose box meets it, counts
// their votes in LDS and writes the winners.  Every label is read about once, every histogram
// counter stays in LDS: 4 x 512 x 1024 labels, 13 classes, halved: clear 12 + votes 35 + argmax 10
// us (27 MB of counters cleared, added to by atomics and scanned) -> boxes 4 + cells 10.  A cell tile
// that more than kVoteMeet input tiles vote into is crowded: its workgroup clears its counters in memory
// instead and marks it, and the histogram kernels, launched behind, cast and count the votes of crowded
// cell tiles alone; they cost 2 us each where there is none.  A call, with the histogram alone, with one
// flag that had everything done again in memory, and so: 57, 18.5, 16 us; the upper half of the map in
// random order 81, 88, 65; a pixel in 256 voting for one far cell 65, 98, 69; all of it in random order
// 103, 113, 111 (60 classes 163, 180, 175; one picture 30, 39, 38: what finding out costs).
constexpr int kVoteTile = 16;        // input tile side
constexpr int kVoteMeet = 64;        // input tiles (16384 pixels) a workgroup takes on
constexpr int kVoteWide = 8;         // ... of which one with a box of more than 16 cell squares is as many
constexpr int kVoteTiles = 8192;     // input tiles: every workgroup looks through all boxes (64 KB)
constexpr size_t kVoteBoxBytes = (size_t)kVoteTiles * sizeof(ushort4);
constexpr int kVoteCounters = 4096;  // LDS counters of a workgroup
// Histograms of fewer bytes than this in all stay in memory: the caches hold them, and five launches
// cost more than three.  (4 x 101 x 314 labels halved, 25 classes, 3.1 MB: 11.2 us there, 12.6 here;
// 5 x 128 x 529, 26 classes, 8.8 MB: 20.2 and 14.3; below 0.5 MB 7 and 14.)
constexpr size_t kVoteBytes = (size_t)4 << 20;
constexpr int kVoteGridX = 256;      // blocks per plane of a launch that may find nothing to do

// One wave per input tile, four rows of it a step.
__global__ __launch_bounds__(kVoteBlock) void vote_boxes_kernel(
    const int64_t* __restrict__ map, ushort4* __restrict__ boxes, int* __restrict__ flag, int IH,
    int IW, int tiles, int tiles_x, int OH, int OW) {
  const int lane = threadIdx.x & 63;
  const int tile = blockIdx.x * (kVoteBlock / 64) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  if (blockIdx.x == 0 && threadIdx.x == 0) *flag = 0;
  if (tile >= tiles) return;
  const int ix = (tile % tiles_x) * kVoteTile + lane % kVoteTile;
  const int iy0 = (tile / tiles_x) * kVoteTile + lane / kVoteTile;
  longlong2 t[4];
#pragma unroll
  for (int r = 0; r < 4; ++r)
    t[r] = reinterpret_cast<const longlong2*>(map)[(size_t)min(iy0 + 4 * r, IH - 1) * IW +
                                                   min(ix, IW - 1)];
  int x0 = 0xffff, y0 = 0xffff, x1 = 0, y1 = 0;   // (x1, y1: one past the last)
#pragma unroll
  for (int r = 0; r < 4; ++r)   // (past the edge: the last pixel again)
    if (t[r].x >= 0 && t[r].x < OW && t[r].y >= 0 && t[r].y < OH) {
      x0 = min(x0, (int)t[r].x);
      y0 = min(y0, (int)t[r].y);
      x1 = max(x1, (int)t[r].x + 1);
      y1 = max(y1, (int)t[r].y + 1);
    }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    x0 = min(x0, __shfl_xor(x0, o));
    y0 = min(y0, __shfl_xor(y0, o));
    x1 = max(x1, __shfl_xor(x1, o));
    y1 = max(y1, __shfl_xor(y1, o));
  }
  if (lane == 0)
    boxes[tile] = make_ushort4((unsigned short)x0, (unsigned short)y0, (unsigned short)x1,
                               (unsigned short)y1);
}

// Workgroup: 2^cell_shift x 2^cell_shift output cells (at most one a thread) of batch element
// blockIdx.y of this pass.  crowded: a mark for each tile of cells, written by the first element's workgroups;
// hist: the elements' histograms, element_stride counters apart.
__global__ __launch_bounds__(kVoteBlock) void vote_tile_kernel(
    const int64_t* __restrict__ labels, const int64_t* __restrict__ map,
    const ushort4* __restrict__ boxes, int* __restrict__ flag, unsigned char* __restrict__ crowded,
    unsigned* __restrict__ hist, size_t element_stride, int64_t* __restrict__ out, int IH, int IW,
    int tiles, int tiles_x, int OH, int OW, int cells_x, int cell_shift, int candidates) {
  __shared__ unsigned votes[kVoteCounters];
  __shared__ int meet[kVoteMeet];
  __shared__ int n_meet, n_wide;
  const int tid = threadIdx.x, side = 1 << cell_shift, cells = side << cell_shift;
  const int ox0 = (blockIdx.x % cells_x) << cell_shift, oy0 = (blockIdx.x / cells_x) << cell_shift;
  const int ox1 = min(ox0 + side, OW), oy1 = min(oy0 + side, OH);
  if (tid == 0) n_meet = n_wide = 0;
  __syncthreads();
  auto look = [&](const ushort4& b, int t) {
    const bool meets =
        t < tiles && b.x < ox0 + side && b.z > ox0 && b.y < oy0 + side && b.w > oy0;
    const unsigned long long all = __ballot(meets);
    if (all == 0) return;
    const unsigned long long wide = __ballot(meets && (b.z - b.x) * (b.w - b.y) > 16 * cells);
    int at = 0;
    if ((tid & 63) == 0) {
      at = atomicAdd(&n_meet, __popcll(all));
      if (wide != 0) atomicAdd(&n_wide, __popcll(wide));
    }
    at = __builtin_amdgcn_readfirstlane(at) + __popcll(all & ((1ull << (tid & 63)) - 1));
    if (meets && at < kVoteMeet) meet[at] = t;
  };
  bool crowd = false;
  for (int seen = 0; seen < tiles && !crowd; seen += 8 * kVoteBlock) {
    ushort4 b[8];   // (eight reads in flight)
#pragma unroll
    for (int u = 0; u < 8; ++u) b[u] = boxes[min(seen + tid + u * kVoteBlock, tiles - 1)];
#pragma unroll
    for (int u = 0; u < 8; ++u) look(b[u], seen + tid + u * kVoteBlock);
    __syncthreads();
    crowd = n_meet + (kVoteWide - 1) * n_wide > kVoteMeet;
    if (seen + 8 * kVoteBlock < tiles) __syncthreads();   // (read by all before the next are counted)
  }
  if (tid == 0 && blockIdx.y == 0) crowded[blockIdx.x] = crowd ? 1 : 0;
  if (crowd) {
    if (tid == 0) *flag = 1;   // (every writer writes the same)
    const int run = (ox1 - ox0) * candidates;
    for (int y = oy0 + (tid >> 6); y < oy1; y += kVoteBlock / 64) {
      unsigned* row =
          hist + blockIdx.y * element_stride + ((size_t)y * OW + ox0) * (size_t)candidates;
      for (int i = tid & 63; i < run; i += 64) row[i] = 0;
    }
    return;
  }
  for (int i = tid; i < cells * candidates; i += kVoteBlock) votes[i] = 0;
  __syncthreads();
  const int64_t* plane = labels + (size_t)blockIdx.y * IH * IW;
  const int py = tid / kVoteTile, px = tid % kVoteTile;
  constexpr int U = 4;   // input tiles whose pixels are requested together
  for (int i0 = 0; i0 < n_meet; i0 += U) {
    longlong2 t[U];
    long long label[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int m = meet[min(i0 + u, n_meet - 1)];
      const int iy = (m / tiles_x) * kVoteTile + py, ix = (m % tiles_x) * kVoteTile + px;
      const size_t at = iy < IH && ix < IW ? (size_t)iy * IW + ix : 0;
      t[u] = reinterpret_cast<const longlong2*>(map)[at];
      label[u] = plane[at];
      if (i0 + u >= n_meet || iy >= IH || ix >= IW) label[u] = -1;   // no pixel: no vote
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      // (cells past the image's edge belong to no workgroup: such votes are not cast)
      if (t[u].x >= ox0 && t[u].x < ox1 && t[u].y >= oy0 && t[u].y < oy1 && label[u] >= 0 &&
          label[u] < candidates) {
        const int cell = (((int)t[u].y - oy0) << cell_shift) + ((int)t[u].x - ox0);
        atomicAdd(&votes[cell * candidates + (int)label[u]], 1u);
      }
    }
  }
  __syncthreads();
  const int ox = ox0 + (tid & (side - 1)), oy = oy0 + (tid >> cell_shift);
  if (tid < cells && ox < OW && oy < OH) {
    const unsigned* v = votes + tid * candidates;
    unsigned best = 0;
    int arg = 0;
    for (int k = 0; k < candidates; ++k) {
      const unsigned n = v[k];
      if (n > best) {   // strict: the first of equal counts stays
        best = n;
        arg = k;
      }
    }
    out[((size_t)blockIdx.y * OH + oy) * OW + ox] = arg;
  }
}

__global__ __launch_bounds__(kVoteBlock) void vote_clear_kernel(uint4* __restrict__ p, size_t n16) {
  const size_t stride = (size_t)gridDim.x * kVoteBlock;
  for (size_t i = (size_t)blockIdx.x * kVoteBlock + threadIdx.x; i < n16; i += stride)
    p[i] = make_uint4(0, 0, 0, 0);
}

// The cell tiles that the histogram kernels are for behind the LDS kernels (CROWD): those marked, if there
// are any (*flag != 0).
struct VoteCrowd {
  const int* flag;
  const unsigned char* marks;
  int cells_x, shift;
  __device__ bool at(int x, int y) const {
    return marks[(y >> shift) * cells_x + (x >> shift)] != 0;
  }
};

// One thread per input pixel (and grid width), grid.y over (batch element of this pass, channel): the plane
// arithmetic is per workgroup, and the pixel's target (16 bytes of the map) and its label are
// requested together.  A label outside [0, candidates) casts no vote (the reference would
// write outside its histogram).  Neighbouring lanes often vote for the same cell (pixels of a
// label image that share a target): a run of them casts its votes with one atomic, from its
// last lane.
template <bool CROWD>
__global__ __launch_bounds__(kVoteBlock) void vote_kernel(
    const int64_t* __restrict__ labels, const int64_t* __restrict__ map,
    unsigned* __restrict__ votes, int in_pixels, int channels, int OH, int OW, int candidates,
    size_t element_stride, VoteCrowd crowd) {
  if (CROWD && *crowd.flag == 0) return;
  const unsigned plane = blockIdx.y;
  const unsigned e = plane / (unsigned)channels, c = plane - e * (unsigned)channels;
  for (long long first = (long long)blockIdx.x * kVoteBlock; first < in_pixels;
       first += (long long)gridDim.x * kVoteBlock) {
    const long long pix = first + threadIdx.x;
    const int at = (int)min(pix, (long long)in_pixels - 1);
    const long long x = map[(size_t)at * 2], y = map[(size_t)at * 2 + 1];
    const long long label = labels[(size_t)plane * in_pixels + at];
    const bool ok = pix < in_pixels && x >= 0 && x <= OW - 1 && y >= 0 && y <= OH - 1 &&
                    label >= 0 && label < candidates && (!CROWD || crowd.at((int)x, (int)y));
    // channel offset in histogram elements as the reference has it (common/resample.h:127-129):
    // c * OH * OW, not c whole histograms, so the histograms of several channels overlap
    const long long cell = ok ? (long long)(e * element_stride + (size_t)c * OH * OW +
                                            ((size_t)y * OW + (size_t)x) * candidates +
                                            (size_t)label)
                              : -1;
    const long long below = __shfl_up(cell, 1);
    const LaneRuns runs(below == cell);
    if (ok && runs.tail) atomicAdd(&votes[cell], (unsigned)(runs.dist + 1));
  }
}

// One thread per output pixel, grid.y over (batch element of this pass, channel): index of
// the first largest count.  The counts are read eight at a time, all eight requested before
// the first is compared.
template <bool CROWD>
__global__ __launch_bounds__(kVoteBlock) void vote_argmax_kernel(
    const unsigned* __restrict__ votes, int64_t* __restrict__ out, int out_pixels, int OW,
    int channels, int candidates, size_t element_stride, VoteCrowd crowd) {
  if (CROWD && *crowd.flag == 0) return;
  const unsigned plane = blockIdx.y;
  const unsigned e = plane / (unsigned)channels, c = plane - e * (unsigned)channels;
  for (long long pix = (long long)blockIdx.x * kVoteBlock + threadIdx.x; pix < out_pixels;
       pix += (long long)gridDim.x * kVoteBlock) {
    if (CROWD && !crowd.at((int)pix % OW, (int)pix / OW)) continue;
    const unsigned* v =
        votes + e * element_stride + ((size_t)c * out_pixels + pix) * (size_t)candidates;
    unsigned best = 0;
    int arg = 0;
    for (int k0 = 0; k0 < candidates; k0 += 8) {
      unsigned n[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) n[i] = v[min(k0 + i, candidates - 1)];
#pragma unroll
      for (int i = 0; i < 8; ++i)
        if (k0 + i < candidates && n[i] > best) {   // strict: the first of equal counts stays
          best = n[i];
          arg = k0 + i;
        }
    }
    out[(size_t)plane * out_pixels + pix] = arg;
  }
}

static size_t vote_bytes(int64_t channels, int64_t oh, int64_t ow, int64_t candidates) {
  const size_t n = (size_t)channels * oh * ow * candidates * sizeof(unsigned);
  return (n + 255) & ~(size_t)255;
}
constexpr size_t kVoteFlagBytes = 256;

// Side (a power of two, as its exponent) of a workgroup's tile of cells: as many as its counters allow,
// 0 where they allow less than 4 x 4.
static int vote_cell_shift(int64_t candidates) {
  for (int shift = 4; shift >= 2; --shift)
    if ((candidates << (2 * shift)) <= kVoteCounters) return shift;
  return 0;
}

// What the LDS kernels need beside the histograms: the flag, the boxes, a mark for each tile of cells.  0 where
// they do not run: several channels (whose histograms overlap), coordinates past 16 bits, many classes.
static size_t vote_tile_bytes(int64_t channels, int64_t oh, int64_t ow, int64_t candidates) {
  const int shift = vote_cell_shift(candidates);
  if (channels != 1 || oh >= 0xffff || ow >= 0xffff || shift == 0) return 0;
  const size_t marks = (size_t)ceil_div(oh, 1 << shift) * ceil_div(ow, 1 << shift);
  return kVoteFlagBytes + kVoteBoxBytes + ((marks + 255) & ~(size_t)255);
}

}  // namespace sdk

using namespace sdk;

extern "C" {

size_t sdk_voting_resample_workspace_bytes(int64_t channels, int64_t out_height,
                                           int64_t out_width, int64_t num_candidates) {
  if (channels < 1 || out_height < 1 || out_width < 1 || num_candidates < 1) return 0;
  // (small histograms, of which such a call has a batch of 4 MB in all, bring the room together)
  const size_t need = vote_bytes(channels, out_height, out_width, num_candidates);
  return need + std::min(vote_tile_bytes(channels, out_height, out_width, num_candidates),
                         (need / 16 + 255) & ~(size_t)255);
}

int sdk_voting_resample_to_map(const int64_t* input, const int64_t* sample_map, int64_t* out,
                               void* workspace, size_t workspace_bytes, int64_t batch,
                               int64_t channels, int64_t in_height, int64_t in_width,
                               int64_t out_height, int64_t out_width, int64_t num_candidates,
                               sdk_stream_t stream) {
  SDK_REQUIRE(batch >= 0 && channels >= 0, "voting_resample_to_map: negative size");
  SDK_REQUIRE(in_height >= 1 && in_width >= 1 && in_height * in_width < ((int64_t)1 << 31) &&
                  out_height >= 1 && out_width >= 1 &&
                  out_height * out_width < ((int64_t)1 << 31),
              "voting_resample_to_map: planes must have 1 .. 2^31-1 elements");
  SDK_REQUIRE(num_candidates >= 1 && num_candidates < ((int64_t)1 << 31),
              "voting_resample_to_map: num_candidates = %lld", (long long)num_candidates);
  if (batch * channels == 0) return SDK_OK;
  SDK_REQUIRE(input && sample_map && out, "voting_resample_to_map: NULL pointer");
  const size_t need = vote_bytes(channels, out_height, out_width, num_candidates);
  if (workspace == nullptr || workspace_bytes < need)
    return fail(SDK_ERR_WORKSPACE, "voting_resample_to_map: workspace of %zu bytes needed, got %zu",
                need, workspace_bytes);
  SDK_REQUIRE((uintptr_t)workspace % 16 == 0, "voting_resample_to_map: workspace not 16-byte aligned");
  hipStream_t s = (hipStream_t)stream;
  unsigned* votes = static_cast<unsigned*>(workspace);
  const int in_pixels = (int)(in_height * in_width);
  const int out_pixels = (int)(out_height * out_width);
  const size_t n_in = (size_t)channels * in_pixels;
  const size_t n_out = (size_t)channels * out_height * out_width;
  SDK_REQUIRE(channels <= 65535, "voting_resample_to_map: more than 65535 channels");
  // The LDS kernels: few enough input tiles, histograms worth it, and a workspace with room for what
  // they need behind at least one (else: the histograms alone).
  const int tiles_x = (int)ceil_div(in_width, kVoteTile);
  const int64_t tiles = (int64_t)tiles_x * ceil_div(in_height, kVoteTile);
  const size_t beside = vote_tile_bytes(channels, out_height, out_width, num_candidates);
  const bool by_tile = beside != 0 && tiles <= kVoteTiles && need * (size_t)batch >= kVoteBytes &&
                       (uintptr_t)sample_map % 16 == 0 && workspace_bytes >= need + beside;
  // as many batch elements per pass as the workspace holds histograms (and grid.y planes)
  const int64_t per_pass = std::min<int64_t>(
      std::min<int64_t>(batch, (int64_t)((workspace_bytes - (by_tile ? beside : 0)) / need)),
      65535 / channels);
  VoteCrowd crowd = {nullptr, nullptr, 0, 0};
  int* flag = nullptr;
  ushort4* boxes = nullptr;
  unsigned char* marks = nullptr;
  unsigned cell_tiles = 0;
  if (by_tile) {
    char* p = static_cast<char*>(workspace) + need * (size_t)per_pass;
    flag = reinterpret_cast<int*>(p);
    boxes = reinterpret_cast<ushort4*>(p + kVoteFlagBytes);
    marks = reinterpret_cast<unsigned char*>(p + kVoteFlagBytes + kVoteBoxBytes);
    crowd.flag = flag;
    crowd.marks = marks;
    crowd.shift = vote_cell_shift(num_candidates);
    crowd.cells_x = (int)ceil_div(out_width, 1 << crowd.shift);
    cell_tiles = (unsigned)(crowd.cells_x * ceil_div(out_height, 1 << crowd.shift));
    launch(vote_boxes_kernel, dim3((unsigned)ceil_div(tiles, kVoteBlock / 64)), dim3(kVoteBlock), s,
           sample_map, boxes, flag, (int)in_height, (int)in_width, (int)tiles, tiles_x,
           (int)out_height, (int)out_width);
  }
  // (behind the LDS kernels: narrow grids, whose blocks are quick to find nothing to do)
  const int64_t most = by_tile ? kVoteGridX : ((int64_t)1 << 31) - 1;
  for (int64_t b = 0; b < batch; b += per_pass) {
    const int64_t nb = std::min<int64_t>(per_pass, batch - b);
    if (by_tile) {
      launch(vote_tile_kernel, dim3(cell_tiles, (unsigned)nb), dim3(kVoteBlock), s,
             input + (size_t)b * n_in, sample_map, (const ushort4*)boxes, flag, marks, votes,
             need / sizeof(unsigned), out + (size_t)b * n_out, (int)in_height, (int)in_width,
             (int)tiles, tiles_x, (int)out_height, (int)out_width, crowd.cells_x, crowd.shift,
             (int)num_candidates);
    } else {
      const size_t n16 = need / 16 * (size_t)nb;
      const int clear_blocks = (int)std::min<int64_t>(ceil_div((int64_t)n16, kVoteBlock), 4096);
      launch(vote_clear_kernel, dim3(clear_blocks), dim3(kVoteBlock), s, (uint4*)workspace, n16);
    }
    const unsigned planes = (unsigned)(nb * channels);
#define VOTES(CROWDv)                                                                              \
  do {                                                                                             \
    launch(vote_kernel<CROWDv>,                                                                    \
           dim3((unsigned)std::min(ceil_div(in_pixels, kVoteBlock), most), planes),                \
           dim3(kVoteBlock), s, input + (size_t)b * n_in, sample_map, votes, in_pixels,            \
           (int)channels, (int)out_height, (int)out_width, (int)num_candidates,                    \
           need / sizeof(unsigned), crowd);                                                        \
    launch(vote_argmax_kernel<CROWDv>,                                                             \
           dim3((unsigned)std::min(ceil_div(out_pixels, kVoteBlock), most), planes),               \
           dim3(kVoteBlock), s, (const unsigned*)votes, out + (size_t)b * n_out, out_pixels,       \
           (int)out_width, (int)channels, (int)num_candidates, need / sizeof(unsigned), crowd);    \
  } while (0)
    if (by_tile) VOTES(true); else VOTES(false);
#undef VOTES
  }
  SDK_LAUNCH_CHECK("voting_resample_to_map");
  return SDK_OK;
}

}  // extern "C"
