// Device fills the C-ABI issues as kernels, so that launch sequences recorded
// into a HIP graph and replayed reset their counters themselves (a memset
// node in a replayed graph is avoided).
#pragma once
#include <hip/hip_runtime.h>

#include "model_ops.h"

namespace cdm {

// p[0..n) = 0 on stream s.
hipError_t zero_ints(int* p, int n, hipStream_t s);

// The combinations of a search grid from its parameters' value lists, the last
// parameter fastest: values [n][ngp], indices (the sum of ids), and, when order is
// not null, the tables of a GridPlan (levels: combinations of each level).
struct GridAxis {
  int param, level;  // 0 shared, 1 other basis, 2 weight parameter
  int first, size;   // its values are vals[first, first + size)
};
struct GridFill {
  int n, ngp, nparams;
  GridAxis axis[kMaxParams];
  int levels[3];
  const double* vals;
  const int* ids;
  double* grid_d;
  float* grid_f;
  int* comb_id;
  float *outer, *inner;
  int* order;
};
hipError_t grid_fill(const GridFill& f, hipStream_t s);

}  // namespace cdm
