// Weight gradient from an LDS window, the columns shared by the workgroup: operands split into
// three bf16 pieces (conv_window_wgrad_quarter.hpp).
#include "conv_window_wgrad_quarter.hpp"

namespace sdk {

int window_wgrad_split(const ConvGeom& g, const Plan& plan, const int* list, const int* count, bool big,
                   const float* pix, const float* img, float* partial, int groups, int c_chunks,
                   int n_tiles, int64_t slots, hipStream_t stream) {
  return window_wgrad_quarter_launch<kMmSplit>(g, plan, list, count, big, pix, img, partial, groups,
                                          c_chunks, n_tiles, slots, stream);
}

}  // namespace sdk
