// Mapped convolution of small calls as explicit columns and plain matrix products
// (conv_columns.hip), float32 tensors, all three matrix arithmetics.
#pragma once
#include <hip/hip_runtime.h>

#include "conv_internal.hpp"

namespace sdk {

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
// map of a kept plan, or nullptr: built in the workspace.
int columns_gemm_scatter(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* Wm, const float* bias, float* img,
                         void* workspace, hipStream_t stream, const void* lists);
// gW = sum_b pix[b] x im2col(img[b])^T; every element of gW is written.  pix_ready: the
// workspace still holds the channels-last copy of pix a columns_gemm_scatter of the same g left.
int columns_gather_wgrad(const ConvGeom& g, int mm, const float* pix, const float* map,
                         const float* wts, const float* img, float* gW, void* workspace,
                         hipStream_t stream, bool pix_ready);

}  // namespace sdk
