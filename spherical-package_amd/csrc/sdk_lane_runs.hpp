// Runs of neighbouring lanes that hold the same key, found with one ballot.
#pragma once
#include <hip/hip_runtime.h>

namespace sdk {

// Runs of equal keys over the lanes of a wave: distance of each lane to the first lane of its
// run and whether it is the last one.  `same` = this lane continues the run of the lane below.
struct LaneRuns {
  int dist;
  bool tail;
  __device__ __forceinline__ LaneRuns(bool same) {
    const int lane = threadIdx.x & 63;
    const unsigned long long heads = __ballot(lane == 0 || !same);
    const unsigned long long upto = heads & (~0ull >> (63 - lane));
    dist = lane - (63 - __clzll((long long)upto));
    tail = lane == 63 || (((heads >> 1) >> lane) & 1ull);
  }
};

// v of the lane D below in the same row of 16 lanes (0 past its start): a vector instruction, where
// a shuffle is a round trip through the LDS pipe.
template <int D>
__device__ __forceinline__ int row_below(int v) {
  return __builtin_amdgcn_update_dpp(0, v, 0x110 + D, 0xf, 0xf, true);   // row_shr:D
}
template <int D>
__device__ __forceinline__ float row_below(float v) {
  return __int_as_float(row_below<D>(__float_as_int(v)));
}
template <int D>
__device__ __forceinline__ double row_below(double v) {
  return __hiloint2double(row_below<D>(__double2hiint(v)), row_below<D>(__double2loint(v)));
}

// The same runs within rows of 16 lanes: a longer one ends at its row's last lane and goes on as
// another, so that its sums need no shuffles.
struct RowRuns {
  int dist;
  bool tail;
  bool any1, any2, any4, any8;   // some lane is that far into its run (the same in all lanes)
  __device__ __forceinline__ RowRuns(bool same) {
    const int lane = threadIdx.x & 63;
    const unsigned long long heads = __ballot((lane & 15) == 0 || !same);
    const unsigned long long upto = heads & (~0ull >> (63 - lane));
    dist = lane - (63 - __clzll((long long)upto));
    tail = (lane & 15) == 15 || (((heads >> 1) >> lane) & 1ull);
    any1 = __any(dist >= 1);
    any2 = __any(dist >= 2);
    any4 = __any(dist >= 4);
    any8 = __any(dist >= 8);
  }
  // inclusive sum of v over the lanes of the run up to this one
  template <typename T>
  __device__ __forceinline__ T sum(T v) const {
    if (any1) {
      const T b = row_below<1>(v);
      v += dist >= 1 ? b : T(0);
    }
    if (any2) {
      const T b = row_below<2>(v);
      v += dist >= 2 ? b : T(0);
    }
    if (any4) {
      const T b = row_below<4>(v);
      v += dist >= 4 ? b : T(0);
    }
    if (any8) {
      const T b = row_below<8>(v);
      v += dist >= 8 ? b : T(0);
    }
    return v;
  }
};

}  // namespace sdk
