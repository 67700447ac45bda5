// Bingham-NODDI: one fanning fibre population.
//   S = S0 [ (1-fiso) ((1-fintra) E + fintra I) + fiso exp(-b Diso) ]
// P: fiso, fintra, kappa, beta, th, ph, psi (kappa = kappa1,
// beta = kappa1 - kappa2).  CFP: g (3), b (1).  FixP: S0.
// Follows NODDI_Bingham/modelfunctions.h:37-246: analytic derivatives in
// fiso and fintra (the latter ignoring the tortuosity dependence of E, as
// the reference), central differences for the rest.
//
// Engine cache hooks: the normaliser 1F1(kappa, beta, 0) and the hindered
// diffusivities (five 1F1 evaluations) depend on fintra, kappa and beta
// only, so they are computed once per parameter vector (Voxel_Cache) instead
// of once per measurement; the intra-axonal signal of each measurement does
// not depend on fiso or fintra, so an MCMC step in those two reuses it
// (Meas_Voxel_Cache, Predicted_Signal_MV; Predicted_Signal_MV_Fill does both
// from one evaluation of the local gradient); the five 1F1 evaluations
// depend on kappa and beta only, so an MCMC step in fintra recombines them.
#include "bingham_math.h"

#define CDM_VOXEL_CACHE 4
#define CDM_VOXEL_CACHE_DEPENDS 0x0Eu       // fintra, kappa, beta
#define CDM_VOXEL_CACHE_JOBS 5              // its five 1F1 evaluations
#define CDM_VOXEL_CACHE_JOBS_DEPENDS 0x0Cu  // kappa, beta
#define CDM_NUMERICAL_MASK 0x7Cu            // kappa, beta, th, ph, psi
#define CDM_MEAS_VOXEL_CACHE 1              // intra-axonal signal per measurement
#define CDM_MEAS_VOXEL_CACHE_DEPENDS 0x7Cu  // kappa, beta, th, ph, psi
#define CDM_MEAS_VOXEL_CACHE_FILL 1         // cache row and signal together
#define CDM_SIGNAL_PARTIALS 1               // signal and analytic entries together
#define CDM_MEAS_CACHE 1                    // exp(-b Diso) per measurement
#define CDM_SIGNAL_FRAME 6                  // sine and cosine of th, ph, psi
#define CDM_SIGNAL_FRAME_DEPENDS 0x70u
#define CDM_LM_ROW_PASSES 2                 // 64-lane LM: the Jacobian rows in two passes
// GridSearch: S = S0 (1-fiso) fan + S0 fiso iso; the intra-axonal signal and
// the local gradient are shared by every fintra and fiso.
#define CDM_GRID_LINEAR 0x01u          // fiso
#define CDM_GRID_SHARED 0x7Cu          // kappa, beta, th, ph, psi
#define CDM_GRID_SHARED_VALUES 3       // intra, cos^2 along the fibre, its complement's part along the azimuth
#define CDM_GRID_SHARED_BASIS 1        // iso
#define CDM_GRID_OUTER_BASIS 1         // fan
#define CDM_GRID_COMMON 2              // b, iso
#define CDM_GRID_TABLE 3               // normaliser and hindered moments of (kappa, beta)
#define CDM_GRID_TABLE_DEPENDS 0x0Cu
#define CDM_GRID_FRAME 9               // the fan's local frame
#define CDM_GRID_FRAME_DEPENDS 0x70u
#define CDM_GRID_OUTER 4               // fintra and the hindered diffusivities

MACRO void Voxel_Cache(int npar, T* P, T* FixP, CDM_F64* vc) {
  bingham_fan f;
  bingham_fan_setup((CDM_F64)P[1], (CDM_F64)P[2], (CDM_F64)P[3], f);
  vc[0] = f.lnc4;
  vc[1] = f.dpar;
  vc[2] = f.dperp1;
  vc[3] = f.dperp2;
}

// The isotropic compartment depends on the b-value only.
MACRO void Meas_Cache(T* CFP, CDM_F64* mc) { mc[0] = exp(-(CDM_F64)CFP[3] * CDM_NODDI_DISO); }

MACRO CDM_F64 Voxel_Cache_Job(int job, int npar, T* P, T* FixP) {
  return bingham_fan_job(job, (CDM_F64)P[2], (CDM_F64)P[3]);
}

MACRO void Voxel_Cache_Combine(int npar, T* P, T* FixP, const CDM_F64* jobs, CDM_F64* vc) {
  bingham_fan f;
  bingham_fan_combine((CDM_F64)P[1], jobs, f);
  vc[0] = f.lnc4;
  vc[1] = f.dpar;
  vc[2] = f.dperp1;
  vc[3] = f.dperp2;
}

MACRO void bingham1_parts(T* P, T* CFP, const CDM_F64* vc, T& fan, T& e, T& i) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  bingham_fan_signal_parts(P[2], P[3], P[4], P[5], P[6], f, CFP, e, i);
  fan = ((T)1 - P[1]) * e + P[1] * i;
}

MACRO T Predicted_Signal_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc) {
  T fan, e, i;
  bingham1_parts(P, CFP, vc, fan, e, i);
  const T iso = (T)mc[0];
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO void Meas_Voxel_Cache(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, T* mvc) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  mvc[0] = bingham_fan_intra(P[2], P[3], P[4], P[5], P[6], f, CFP);
}

MACRO T Predicted_Signal_MV(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, const T* mvc) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  const T e = bingham_fan_extra(P[4], P[5], P[6], f, CFP);
  const T fan = ((T)1 - P[1]) * e + P[1] * mvc[0];
  const T iso = (T)mc[0];
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

// The same from the sines and cosines of the angles (the frame).
MACRO void Signal_Frame(int npar, T* P, T* fr, int changed) {
  T s, c;
  tsincos(changed == 4 ? P[4] : changed == 5 ? P[5] : P[6], &s, &c);
  for (int k = 0; k < 3; ++k) {
    if (changed != 4 + k) continue;
    fr[2 * k] = s;
    fr[2 * k + 1] = c;
  }
}

MACRO T Predicted_Signal_MV_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, const T* mvc,
                                   const T* fr) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  T gx, gy, gn;
  bingham_trig_local(fr, CFP, gx, gy, gn);
  const T e = bingham_fan_extra_local(gx, gy, gn, CFP[3], f);
  const T fan = ((T)1 - P[1]) * e + P[1] * mvc[0];
  const T iso = (T)mc[0];
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO T Predicted_Signal_MV_Fill_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, T* mvc,
                                        const T* fr) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  T gx, gy, gn;
  bingham_trig_local(fr, CFP, gx, gy, gn);
  const T e = bingham_fan_extra_local(gx, gy, gn, CFP[3], f);
  mvc[0] = bingham_fan_intra_local(P[2], P[3], gx, gy, gn, CFP[3], f);
  const T fan = ((T)1 - P[1]) * e + P[1] * mvc[0];
  const T iso = (T)mc[0];
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO T Predicted_Signal_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, const T* fr) {
  T mvc[1];
  return Predicted_Signal_MV_Fill_Framed(npar, P, CFP, FixP, vc, mc, mvc, fr);
}

// Meas_Voxel_Cache and Predicted_Signal_MV from one local gradient.
MACRO T Predicted_Signal_MV_Fill(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, T* mvc) {
  T fan, e, i;
  bingham1_parts(P, CFP, vc, fan, e, i);
  mvc[0] = i;
  const T iso = (T)mc[0];
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO T Predicted_Signal(int npar, T* P, T* CFP, T* FixP) {
  CDM_F64 vc[4], mc[1];
  Voxel_Cache(npar, P, FixP, vc);
  Meas_Cache(CFP, mc);
  return Predicted_Signal_Cached(npar, P, CFP, FixP, vc, mc);
}

// GridSearch hooks: the same compartments from their shared parts.
MACRO void Grid_Table(int npar, T* P, CDM_F64* tb) {
  const CDM_F64 k = (CDM_F64)P[2], b = (CDM_F64)P[3];
  CDM_F64 h[5];
  for (int j = 0; j < 5; ++j) h[j] = bingham_fan_job(j, k, b);
  tb[0] = log(4.0 * h[0]);
  tb[1] = ((h[1] - h[2]) / (2.0 * bingham_fd_delta)) / h[0];
  tb[2] = ((h[3] - h[4]) / (2.0 * bingham_fd_delta)) / h[0];
}

MACRO void Grid_Frame(int npar, T* P, T* fr) { bingham_fan_frame_of<T>(P[4], P[5], P[6], fr); }

MACRO void Grid_Shared(int npar, T* P, T* CFP, T* FixP, const CDM_F64* tb, const T* fr, const CDM_F64* mc, T* sh) {
  const T gx = CFP[0] * fr[0] + CFP[1] * fr[1] + CFP[2] * fr[2];
  const T gy = CFP[0] * fr[3] + CFP[1] * fr[4] + CFP[2] * fr[5];
  const T gn = CFP[0] * fr[6] + CFP[1] * fr[7] + CFP[2] * fr[8];
  bingham_fan f;
  f.lnc4 = tb[0];
  sh[0] = bingham_fan_intra_local(P[2], P[3], gx, gy, gn, CFP[3], f);
  const T c2 = gn * gn, s2 = (T)1 - c2, gxy = gx * gx + gy * gy;
  const T caz2 = gxy > (T)0 ? tdiv_fast(gx * gx, gxy) : (T)1;
  sh[1] = c2;
  sh[2] = s2 * caz2;
}

MACRO void Grid_Common(int npar, T* CFP, const CDM_F64* mc, T* cm) {
  cm[0] = CFP[3];
  cm[1] = (T)mc[0];
}

MACRO void Grid_Shared_Basis(int npar, const T* sh, const T* cm, T* basis) { basis[0] = cm[1]; }

MACRO void Grid_Outer(int npar, T* P, const CDM_F64* tb, T* so) {
  const CDM_F64 dperp = CDM_NODDI_DPAR * (1.0 - (CDM_F64)P[1]), dd = CDM_NODDI_DPAR - dperp;
  const CDM_F64 dpar = dperp + dd * tb[1], dperp1 = dperp + dd * tb[2];
  so[0] = P[1];
  so[1] = (T)dpar;
  so[2] = (T)dperp1;
  so[3] = (T)(CDM_NODDI_DPAR + 2 * dperp - dpar - dperp1);
}

MACRO void Grid_Outer_Basis(int npar, T* P, const T* cm, const T* so, const T* sh, T* basis) {
  const T s2 = (T)1 - sh[1];
  const T e = texp_fast(-cm[0] * (so[1] * sh[1] + (so[2] * (s2 - sh[2]) + so[3] * sh[2])));
  basis[0] = ((T)1 - so[0]) * e + so[0] * sh[0];
}

MACRO void Grid_Weights(int npar, T* P, T* FixP, T* w) {
  w[0] = FixP[0] * P[0];
  w[1] = FixP[0] * ((T)1 - P[0]);
}

// kappa must exceed beta by 0.05 (NODDI_Bingham/modelfunctions.h:169-178).
MACRO bool ConstraintsMCMC(int npar, T* P) { return !((P[2] - (T)0.05) < P[3]); }

// Analytic entries (fiso, fintra); the engine forms the others.
MACRO void Partial_Derivatives_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                      T* derivatives) {
  T fan, e, i;
  bingham1_parts(P, CFP, vc, fan, e, i);
  const T iso = (T)mc[0];
  derivatives[0] = FixP[0] * (iso - fan);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (i - e);
}

// The signal of Predicted_Signal_Cached with the analytic entries of
// Partial_Derivatives_Cached, from one evaluation of the fan's parts.
MACRO T Predicted_Signal_Partials_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                         T* derivatives) {
  T fan, e, i;
  bingham1_parts(P, CFP, vc, fan, e, i);
  const T iso = (T)mc[0];
  derivatives[0] = FixP[0] * (iso - fan);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (i - e);
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO T Predicted_Signal_Partials_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                         T* derivatives, const T* fr) {
  bingham_fan f;
  f.lnc4 = vc[0];
  f.dpar = vc[1];
  f.dperp1 = vc[2];
  f.dperp2 = vc[3];
  T gx, gy, gn;
  bingham_trig_local(fr, CFP, gx, gy, gn);
  const T e = bingham_fan_extra_local(gx, gy, gn, CFP[3], f);
  const T i = bingham_fan_intra_local(P[2], P[3], gx, gy, gn, CFP[3], f);
  const T fan = ((T)1 - P[1]) * e + P[1] * i;
  const T iso = (T)mc[0];
  derivatives[0] = FixP[0] * (iso - fan);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (i - e);
  return FixP[0] * (((T)1 - P[0]) * fan + P[0] * iso);
}

MACRO void Partial_Derivatives(int npar, T* P, T* CFP, T* FixP, T* derivatives) {
  CDM_F64 vc[4], mc[1];
  Voxel_Cache(npar, P, FixP, vc);
  Meas_Cache(CFP, mc);
  Partial_Derivatives_Cached(npar, P, CFP, FixP, vc, mc, derivatives);
  derivatives[2] = NUMERICAL(2);
  derivatives[3] = NUMERICAL(3);
  derivatives[4] = NUMERICAL(4);
  derivatives[5] = NUMERICAL(5);
  derivatives[6] = NUMERICAL(6);
}

// After LM: beta may not exceed kappa (NODDI_Bingham/modelfunctions.h:228-236).
MACRO void FixConstraintsLM(int npar, T* P) {
  if (P[2] < P[3]) P[3] = P[2] - (T)0.05;
}

MACRO T custom_priors(int id_p, T* P, int nmeas, T* CFP, T* FixP) { return (T)0; }
