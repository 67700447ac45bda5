// Derived maps of the reference's <Model>_finish.sh steps, computed from
// the MCMC samples [nvox][nparams][nsamples] where they lie in device
// memory: per-parameter sample means (fslmaths -Tmean), mean fibre
// orientations from the mean dyadic tensor (FSL make_dyadic_vectors; the
// reference's utils/getFanningOrientation.cc:39-76 for Bingham fanning
// directions) and the NODDI dispersion indices
// (NODDI_Watson_finish.sh:35, NODDI_Bingham_finish.sh:46-56).
//
// All three read each sample once and write a few values per voxel: HBM
// bound, 16 lanes per row of samples, so that a wave reads runs of adjacent
// values (one thread per row had every lane of a wave on another row: 1.02 ms
// for the 280 MB of 200k voxels x 7 x 50, against 0.105 ms; dyads 0.36-0.58 ->
// 0.06-0.08 ms, maps 0.37 -> 0.035 ms).  Rows of few samples lie near enough for
// a thread each, and 16 lanes would mostly idle: a million voxels, means of 1 / 4 /
// 12 / 15 / 16 samples 25 / 46 / 157 / 219 / 272 us by threads and 196 / 199 / 244 /
// 248 / 257 by 16 lanes; dyads of 1 / 4 / 8 / 12 samples 53 / 99 / 166 / 256 and 110 /
// 166 / 167 / 179; Bingham maps of 4 / 8 samples 43 / 136 and 100 / 100, Watson's (one
// row a voxel) of 2 / 4 23 / 64 and 50 / 51.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>

#include "../../../include/cudimot_amd.h"
#include "../engine/wave.h"
#include "../host/model_ops.h"

namespace {

constexpr int kBlock = 256;
constexpr float kTwoDivPi = 0.636619772367581f;  // the finish scripts' Two_div_pi

constexpr int kLanes = 16;  // lanes per row of samples, from kFew* samples on (one below)
constexpr int kFewMean = 16, kFewDyads = 8, kFewBingham = 8, kFewWatson = 4;

template <int LANES>
__global__ __launch_bounds__(kBlock) void sample_mean_kernel(long long rows, int ns, const float* __restrict__ x,
                                                             float* __restrict__ out) {
  constexpr int kPer = kBlock / LANES;
  const int lane = threadIdx.x % LANES;
  for (long long r = (long long)blockIdx.x * kPer + threadIdx.x / LANES; r < rows; r += (long long)gridDim.x * kPer) {
    const float* p = x + r * ns;
    double s = 0.0;
#pragma unroll 4
    for (int k = lane; k < ns; k += LANES) s += p[k];
    s = cdm::Group<LANES>::sum(s);
    if (lane == 0) out[r] = (float)(s / ns);
  }
}

// Cyclic Jacobi rotations of a symmetric 3x3 matrix a (upper triangle
// a00 a01 a02 a11 a12 a22); v receives the eigenvectors as columns.
__device__ void jacobi3(double a[3][3], double v[3][3]) {
  for (int i = 0; i < 3; ++i)
    for (int j = 0; j < 3; ++j) v[i][j] = i == j;
  for (int sweep = 0; sweep < 32; ++sweep) {
    const double off = fabs(a[0][1]) + fabs(a[0][2]) + fabs(a[1][2]);
    const double diag = fabs(a[0][0]) + fabs(a[1][1]) + fabs(a[2][2]);
    if (off <= 1e-15 * diag || off == 0.0) break;
    for (int p = 0; p < 2; ++p) {
      for (int q = p + 1; q < 3; ++q) {
        if (a[p][q] == 0.0) continue;
        // rotation angle that zeroes a[p][q]: tan(2t) = 2 a_pq / (a_qq - a_pp)
        const double theta = (a[q][q] - a[p][p]) / (2.0 * a[p][q]);
        const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double c = 1.0 / sqrt(t * t + 1.0), s = t * c;
        for (int k = 0; k < 3; ++k) {  // columns p, q of A
          const double akp = a[k][p], akq = a[k][q];
          a[k][p] = c * akp - s * akq;
          a[k][q] = s * akp + c * akq;
        }
        for (int k = 0; k < 3; ++k) {  // rows p, q
          const double apk = a[p][k], aqk = a[q][k];
          a[p][k] = c * apk - s * aqk;
          a[q][k] = s * apk + c * aqk;
        }
        for (int k = 0; k < 3; ++k) {
          const double vkp = v[k][p], vkq = v[k][q];
          v[k][p] = c * vkp - s * vkq;
          v[k][q] = s * vkp + c * vkq;
        }
      }
    }
  }
}

// A block handles 64 voxels (a thread per row: 256): the dyadic sums, 16 lanes per
// voxel, into LDS, then one thread per voxel for the eigenvectors (a thousand
// serial FP64 instructions that 16 lanes would repeat).
template <int LANES>
constexpr int kDyadVoxels = LANES == 1 ? kBlock : 64;

// Blocks of a launch over `n` units, `per` a block: at most kMaxBlocks (a launch
// has fewer than 2^32 threads), which then take several each.
constexpr long long kMaxBlocks = 1 << 20;
unsigned blocks_for(long long n, int per) { return (unsigned)std::min((n + per - 1) / per, kMaxBlocks); }

template <int LANES>
__global__ __launch_bounds__(kBlock) void dyads_kernel(int n, int np, int ns, const float* __restrict__ x, int th,
                                                       int ph, int psi, float* __restrict__ dyads,
                                                       float* __restrict__ disp) {
  constexpr int kVoxels = kDyadVoxels<LANES>, kPer = kBlock / LANES;
  __shared__ double sums[kVoxels][7];  // 7: an odd stride over the banks
  const int lane = threadIdx.x % LANES;
  for (long long v0 = (long long)blockIdx.x * kVoxels; v0 < n; v0 += (long long)gridDim.x * kVoxels) {
    for (int q = threadIdx.x / LANES; q < kVoxels; q += kPer) {
      const long long v = v0 + q;
      if (v >= n) break;
      const float* base = x + (size_t)v * np * ns;
      double m[6] = {};
      for (int k = lane; k < ns; k += LANES) {
        const float t = base[th * ns + k], f = base[ph * ns + k];
        float st, ct, sf, cf;
        sincosf(t, &st, &ct);
        sincosf(f, &sf, &cf);
        float d[3];
        if (psi < 0) {  // fibre direction
          d[0] = st * cf;
          d[1] = st * sf;
          d[2] = ct;
        } else {  // fanning direction (getFanningOrientation.cc:49-51)
          float sp, cp;
          sincosf(base[psi * ns + k], &sp, &cp);
          d[0] = -cp * sf - ct * cf * sp;
          d[1] = cf * cp - ct * sf * sp;
          d[2] = st * sp;
        }
        int e = 0;
#pragma unroll
        for (int i = 0; i < 3; ++i)
#pragma unroll
          for (int j = i; j < 3; ++j) m[e++] += (double)d[i] * d[j];
      }
#pragma unroll
      for (int e = 0; e < 6; ++e) {
        const double t = cdm::Group<LANES>::sum(m[e]);
        if (lane == 0) sums[q][e] = t;
      }
    }
    __syncthreads();
    const long long v = v0 + threadIdx.x;
    if (threadIdx.x < kVoxels && v < n) {
      double m[3][3];
      for (int i = 0, e = 0; i < 3; ++i)
        for (int j = i; j < 3; ++j, ++e) m[j][i] = m[i][j] = sums[threadIdx.x][e] / ns;
      double vec[3][3];
      jacobi3(m, vec);
      int b = 0;
      for (int i = 1; i < 3; ++i)
        if (m[i][i] > m[b][b]) b = i;
      double e[3] = {vec[0][b], vec[1][b], vec[2][b]};
      const double nrm = sqrt(e[0] * e[0] + e[1] * e[1] + e[2] * e[2]);
      // An eigenvector's sign is arbitrary: report the one with z >= 0 (then
      // y, then x, for vectors in the xy-plane).
      const double key = e[2] != 0.0 ? e[2] : (e[1] != 0.0 ? e[1] : e[0]);
      const double sg = (key < 0 ? -1.0 : 1.0) / (nrm > 0 ? nrm : 1.0);
      for (int i = 0; i < 3; ++i) dyads[(size_t)v * 3 + i] = (float)(e[i] * sg);
      if (disp) {
        double lmax = 0.0;
        for (int i = 0; i < 3; ++i) lmax = fmax(lmax, fabs(m[i][i]));
        disp[v] = (float)(1.0 - lmax);
      }
    }
    __syncthreads();  // the next voxels' sums
  }
}

template <int LANES>
__global__ __launch_bounds__(kBlock) void noddi_maps_kernel(int n, int np, int ns, const float* __restrict__ x,
                                                            int kappa, int beta, float* __restrict__ maps) {
  constexpr int kPer = kBlock / LANES;
  const int lane = threadIdx.x % LANES;
  for (long long v = (long long)blockIdx.x * kPer + threadIdx.x / LANES; v < n; v += (long long)gridDim.x * kPer) {
    const float* base = x + (size_t)v * np * ns;
    double sk = 0.0, sb = 0.0, sk2 = 0.0;
#pragma unroll 4
    for (int k = lane; k < ns; k += LANES) {
      const float kk = base[kappa * ns + k];
      sk += kk;
      if (beta >= 0) {
        const float bb = base[beta * ns + k];
        sb += bb;
        sk2 += (float)(kk - bb);  // the k2 = kappa - beta sample volume
      }
    }
    sk = cdm::Group<LANES>::sum(sk);
    if (beta >= 0) {
      sb = cdm::Group<LANES>::sum(sb);
      sk2 = cdm::Group<LANES>::sum(sk2);
    }
    if (lane != 0) continue;
    const float mk = (float)(sk / ns);
    if (beta < 0) {  // Watson: OD = 2/pi atan(1/kappa)
      maps[v] = atanf(1.0f / mk) * kTwoDivPi;
      continue;
    }
    const float mb = (float)(sb / ns), mk2 = (float)(sk2 / ns);
    float* o = maps + (size_t)v * 5;
    o[0] = mk2;
    o[1] = atanf(1.0f / mk2) * kTwoDivPi;                                // ODIp
    o[2] = atanf(1.0f / mk) * kTwoDivPi;                                 // ODIs
    o[3] = atanf(fabsf(sqrtf((1.0f / mk) * (1.0f / mk2)))) * kTwoDivPi;  // ODItot
    o[4] = atanf(mb / mk2) * kTwoDivPi;                                  // DA
  }
}

int launch_check(const char* what) {
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return cdm::set_error(std::string(what) + ": " + hipGetErrorString(e));
  return 0;
}

}  // namespace

extern "C" {

int cdm_sample_mean(int nvox, int nparams, int nsamples, const float* samples, float* mean, void* stream) {
  if (nvox < 0 || nparams <= 0 || nsamples <= 0) return cdm::set_error("cdm_sample_mean: bad sizes");
  if (nvox == 0) return 0;
  if (!samples || !mean) return cdm::set_error("cdm_sample_mean: null pointer");
  const long long rows = (long long)nvox * nparams;
  const bool few = nsamples < kFewMean;
  hipLaunchKernelGGL(few ? sample_mean_kernel<1> : sample_mean_kernel<kLanes>,
                     dim3(blocks_for(rows, few ? kBlock : kBlock / kLanes)), dim3(kBlock), 0, (hipStream_t)stream, rows,
                     nsamples, samples, mean);
  return launch_check("cdm_sample_mean");
}

int cdm_dyads(int nvox, int nparams, int nsamples, const float* samples, int theta, int phi, int psi, float* dyads,
              float* dispersion, void* stream) {
  if (nvox < 0 || nparams <= 0 || nsamples <= 0) return cdm::set_error("cdm_dyads: bad sizes");
  if (theta < 0 || theta >= nparams || phi < 0 || phi >= nparams || psi >= nparams)
    return cdm::set_error("cdm_dyads: parameter index out of range");
  if (nvox == 0) return 0;
  if (!samples || !dyads) return cdm::set_error("cdm_dyads: null pointer");
  const bool few = nsamples < kFewDyads;
  hipLaunchKernelGGL(few ? dyads_kernel<1> : dyads_kernel<kLanes>,
                     dim3(blocks_for(nvox, few ? kDyadVoxels<1> : kDyadVoxels<kLanes>)), dim3(kBlock), 0,
                     (hipStream_t)stream, nvox, nparams, nsamples, samples, theta, phi, psi, dyads, dispersion);
  return launch_check("cdm_dyads");
}

int cdm_noddi_maps(int nvox, int nparams, int nsamples, const float* samples, int kappa, int beta, float* maps,
                   void* stream) {
  if (nvox < 0 || nparams <= 0 || nsamples <= 0) return cdm::set_error("cdm_noddi_maps: bad sizes");
  if (kappa < 0 || kappa >= nparams || beta >= nparams) return cdm::set_error("cdm_noddi_maps: parameter index out of range");
  if (nvox == 0) return 0;
  if (!samples || !maps) return cdm::set_error("cdm_noddi_maps: null pointer");
  const bool few = nsamples < (beta >= 0 ? kFewBingham : kFewWatson);
  hipLaunchKernelGGL(few ? noddi_maps_kernel<1> : noddi_maps_kernel<kLanes>,
                     dim3(blocks_for(nvox, few ? kBlock : kBlock / kLanes)), dim3(kBlock), 0, (hipStream_t)stream, nvox,
                     nparams, nsamples, samples, kappa, beta, maps);
  return launch_check("cdm_noddi_maps");
}

}  // extern "C"
