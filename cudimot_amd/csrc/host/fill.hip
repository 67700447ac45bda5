// Device fills of the C-ABI (fill.h).
#include "fill.h"

namespace {

__global__ void __launch_bounds__(256) zero_ints_kernel(int* p, int n) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = 0;
}

// One thread per combination.  Bound by its stores, 16 or more bytes per
// parameter; 262,144 combinations of three parameters: 12 us.
__global__ void __launch_bounds__(256) grid_fill_kernel(cdm::GridFill f) {
  const int c = blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= f.n) return;
  int rest = c, id = 0;
  int pos[3] = {0, 0, 0}, mult[3] = {1, 1, 1};  // place within each level
  for (int k = f.ngp - 1; k >= 0; --k) {
    const cdm::GridAxis a = f.axis[k];
    const int d = rest % a.size;
    rest /= a.size;
    const double v = f.vals[a.first + d];
    id += f.ids[a.first + d];
    f.grid_d[(size_t)c * f.ngp + k] = v;
    f.grid_f[(size_t)c * f.ngp + k] = (float)v;
#pragma unroll
    for (int l = 0; l < 3; ++l)
      if (a.level == l) {
        pos[l] += d * mult[l];
        mult[l] *= a.size;
      }
  }
  f.comb_id[c] = id;
  if (!f.order) return;
  const size_t o = (size_t)pos[0] * f.levels[1] + pos[1];
  f.order[o * f.levels[2] + pos[2]] = c;
  for (int side = 0; side < 2; ++side) {  // the tables' rows: the first thread of an outer, of an inner combination
    if (side == 0 ? pos[2] != 0 : o != 0) continue;
    float* row = side == 0 ? f.outer + o * f.nparams : f.inner + (size_t)pos[2] * f.nparams;
    for (int p = 0; p < f.nparams; ++p) row[p] = 0.0f;
    for (int k = 0; k < f.ngp; ++k) row[f.axis[k].param] = f.grid_f[(size_t)c * f.ngp + k];
  }
}

}  // namespace

namespace cdm {

hipError_t zero_ints(int* p, int n, hipStream_t s) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(zero_ints_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, p, n);
  return hipGetLastError();
}

hipError_t grid_fill(const GridFill& f, hipStream_t s) {
  if (f.n <= 0) return hipSuccess;
  hipLaunchKernelGGL(grid_fill_kernel, dim3((unsigned)(((size_t)f.n + 255) / 256)), dim3(256), 0, s, f);
  return hipGetLastError();
}

}  // namespace cdm
