// Mapped convolution of small calls as explicit columns and plain matrix products
// (conv_columns.hip), float32 tensors, all three matrix arithmetics.
#pragma once
#include <hip/hip_runtime.h>

#include "conv_internal.hpp"

namespace sdk {

inline int pad8(int c) { return (c + 7) & ~7; }

// One 64-element x 32-channel tile of src[C][N] into dst[N][Cp8] (256 threads; channels C .. Cp8 - 1 are
// zeros): through LDS, reads along n, 16-byte writes along c.
__device__ __forceinline__ void channels_last_tile(const float* __restrict__ src, float* __restrict__ dst, int C,
                                                   int Cp8, int N, int n0, int c0, float (*tile)[65]) {
  typedef float vec4 __attribute__((ext_vector_type(4)));
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
#pragma unroll
  for (int i = 0; i < 8; ++i) {
    const int c = c0 + w + 4 * i, n = n0 + lane;
    const float v = src[(size_t)min(c, C - 1) * N + min(n, N - 1)];
    tile[w + 4 * i][lane] = (c < C && n < N) ? v : 0.0f;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 2; ++i) {   // 64 n x 8 channel quads
    const int item = threadIdx.x + 256 * i;
    const int n = item >> 3, q = item & 7;
    if (n0 + n < N && c0 + 4 * q < Cp8) {
      vec4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = tile[4 * q + e][n];
      *reinterpret_cast<vec4*>(dst + (size_t)(n0 + n) * Cp8 + c0 + 4 * q) = v;
    }
  }
}

// The contractions without a column matrix in front of them (conv_columns_direct.hip): of the calls of the
// route on maps that columns_direct() takes, the forwards and the backwards that ..._gather and ..._backward do.
struct ColumnsScratch {
  float* img_rows;      // B * H * W + 1 rows of pad8(Cg) floats
  void* weights;        // columns_weight_bytes()
  void *pix_rows, *pix_cols;   // columns_pixel_row_bytes(), columns_pixel_column_bytes()
  float* strip_sums;    // columns_strip_bytes()
  float* col;           // the products of a scatter
  float* partial;       // columns_partial_bytes(), or columns_forward_sum_bytes()
};
bool columns_direct(const ConvGeom& g);
bool columns_direct_gather(const ConvGeom& g, int mm);
bool columns_direct_backward(const ConvGeom& g, int mm);
size_t columns_weight_bytes(const ConvGeom& g, int mm);
size_t columns_forward_sum_bytes(const ConvGeom& g, int mm);
size_t columns_pixel_row_bytes(const ConvGeom& g, int mm, int64_t elements);
size_t columns_pixel_column_bytes(const ConvGeom& g, int mm, int64_t elements);
size_t columns_partial_bytes(const ConvGeom& g, int mm, int64_t elements);
size_t columns_strip_bytes(const ConvGeom& g);
int columns_direct_forward(const ConvGeom& g, int mm, const float* img, const float* map, const float* wts,
                           const float* Wm, const float* bias, float* pix, const ColumnsScratch& s,
                           hipStream_t stream);
// Lays out, in one launch, the pixels of batch elements first .. first + elements - 1 as operands of the weight
// gradient (rows) and of the scatter's product (cols), the sums of their strips, and, where they are given, the
// product's weights, in chunks of so many channels (multiples of 32, or all of them), and the whole image.
int columns_direct_prepare(const ConvGeom& g, int mm, const float* pix, int64_t first, int64_t elements, bool rows,
                           bool cols, bool strip_sums, const float* Wm, int channels, const float* img,
                           const ColumnsScratch& s, hipStream_t stream);
// s.col[b][m][(k, c)] = sum over n of pix * Wm, of elements first .. first + elements - 1 of those whose cols are laid
// out and of the chunk of channels c0 .. c0 + channels - 1.
int columns_direct_product(const ConvGeom& g, int mm, int64_t first, int64_t elements, int c0, int channels,
                           const ColumnsScratch& s, hipStream_t stream);
// `slice` batch elements at a time.  prepared: image, rows of the whole batch, one slice, and the sums of its strips
// are laid out.  gb: also gb[n] = sum of pix[b][n][m] (optional).
int columns_direct_wgrad(const ConvGeom& g, int mm, const float* pix, const float* map, const float* wts,
                         const float* img, float* gW, int64_t slice, const ColumnsScratch& s, bool prepared, float* gb,
                         hipStream_t stream);

// Maps whose kept plan holds the inverted lists the route's scatter reads (H, W, M, K, P and
// interp of g).
bool columns_map(const ConvGeom& g);
// Calls that take the route.
bool columns_route(const ConvGeom& g);
size_t columns_workspace_bytes(const ConvGeom& g);

// pix[b] = Wm x im2col(img[b]) + bias (bias may be nullptr).
int columns_gather_gemm(const ConvGeom& g, int mm, const float* img, const float* map,
                        const float* wts, const float* Wm, const float* bias, float* pix,
                        void* workspace, hipStream_t stream);
// img[b] = bias + col2im(Wm^T x pix[b]); every element of img is written.  lists: the inverted
// map of a kept plan, or nullptr: built in the workspace.  wgrad_img (optional): the image of a
// columns_gather_wgrad of the same call that follows with `prepared`; bias_sum: it is asked for the bias gradient.
int columns_gemm_scatter(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* Wm, const float* bias, float* img,
                         void* workspace, hipStream_t stream, const void* lists,
                         const float* wgrad_img, bool bias_sum);
// gW = sum_b pix[b] x im2col(img[b])^T; every element of gW is written.  prepared: the workspace
// still holds what a columns_gemm_scatter of the same g and mm may have laid out for it.  gb
// (columns_sums_bias): also gb[n] = sum of pix[b][n][m].
bool columns_sums_bias(const ConvGeom& g, int mm);
int columns_gather_wgrad(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* img, float* gW, void* workspace,
                         hipStream_t stream, bool prepared, float* gb);

}  // namespace sdk
