// NODDI with a Watson orientation distribution.
//   S = S0 [ (1-fiso) ((1-fintra) E + fintra I) + fiso exp(-b Diso) ]
// E: hindered compartment, exp(-b ((dpar_eq - dperp_eq) (g.n)^2 + dperp_eq))
//    with dperp = Dpar (1 - fintra) (tortuosity);
// I: intra-axonal sticks, 1/2 sum_l L_l(b Dpar) c_l(kappa) Y_2l(g.n),
//    floored at 1e-3 before the 1/2 when negative.
// P: fiso, fintra, kappa, th, ph.  CFP: g (3), b (1).  FixP: S0.
// Follows NODDI_Watson/modelfunctions.h:68-216.  The derivative in fintra
// is the reference's (it ignores the tortuosity dependence of E).
//
// Engine cache hooks: the hindered diffusivities and the SH coefficients
// depend on (fintra, kappa) only (Voxel_Cache); the Legendre-Gaussian
// integrals and the isotropic term depend on the b-value only (Meas_Cache).
#include "watson_math.h"

#define CDM_VOXEL_CACHE 9              // dpar_eq, dperp_eq, c_0..c_6
#define CDM_VOXEL_CACHE_DEPENDS 0x06u  // fintra, kappa
#define CDM_MEAS_CACHE 8               // L_0..L_6 (b Dpar), exp(-b Diso)
#define CDM_NUMERICAL_MASK 0x1Cu       // kappa, th, ph
#define CDM_SIGNAL_PARTIALS 1          // signal and analytic entries together
#define CDM_SIGNAL_FRAME 4             // sine and cosine of th, ph
#define CDM_SIGNAL_FRAME_DEPENDS 0x18u
// GridSearch: S = S0 (1-fiso) aniso + S0 fiso iso; the intra-axonal signal is
// shared by every fintra and fiso.
#define CDM_GRID_LINEAR 0x01u          // fiso
#define CDM_GRID_SHARED 0x1Cu          // kappa, th, ph
#define CDM_GRID_SHARED_VALUES 2       // intra, (g.n)^2
#define CDM_GRID_SHARED_BASIS 1        // iso
#define CDM_GRID_OUTER_BASIS 1         // aniso
#define CDM_GRID_COMMON 2              // b, iso
#define CDM_GRID_TABLE 8               // c_0..c_6, the hindered moment of kappa
#define CDM_GRID_TABLE_DEPENDS 0x04u
#define CDM_GRID_FRAME 3               // the fibre
#define CDM_GRID_FRAME_DEPENDS 0x18u
#define CDM_GRID_OUTER 3               // fintra and the hindered diffusivities

MACRO void Voxel_Cache(int npar, T* P, T* FixP, CDM_F64* vc) {
  noddi_watson_hindered((CDM_F64)P[2], CDM_NODDI_DPAR * (1.0 - (CDM_F64)P[1]), vc[0], vc[1]);
  noddi_watson_sh((CDM_F64)P[2], vc + 2);
}

MACRO void Meas_Cache(T* CFP, CDM_F64* mc) {
  noddi_lgi((CDM_F64)CFP[3] * CDM_NODDI_DPAR, mc);
  mc[7] = exp(-(CDM_F64)CFP[3] * CDM_NODDI_DISO);
}

// tr: sine and cosine of th and of ph.
MACRO void watson_parts_of(const T* tr, T* P, T* CFP, const CDM_F64* vc, const CDM_F64* mc, T& extra, T& intra) {
  const T st = tr[0], ct = tr[1], sp = tr[2], cp = tr[3];
  T gn = CFP[0] * st * cp + CFP[1] * st * sp + CFP[2] * ct;
#ifdef CDM_WATSON_REFERENCE_FORMS
  extra = exp_gpu(-CFP[3] * ((T)(vc[0] - vc[1]) * gn * gn + (T)vc[1]));
#else
  // the hardware 2^x form in single precision: its error is below the float
  // rounding the argument already carries (exact exp in double)
  extra = texp_fast(-CFP[3] * ((T)(vc[0] - vc[1]) * gn * gn + (T)vc[1]));
#endif
  if (gn > (T)1) gn = (T)1;
  if (gn < (T)-1) gn = (T)-1;
  T sh[7];
  noddi_even_sh(gn, sh);
  CDM_F64 s = 0.0;
  for (int l = 0; l < 7; ++l) s += mc[l] * vc[2 + l] * (CDM_F64)sh[l];
  if (s < 0) s = 1e-3;
  intra = (T)(0.5 * s);
}

MACRO void watson_parts(T* P, T* CFP, const CDM_F64* vc, const CDM_F64* mc, T& extra, T& intra) {
  T tr[4];
  tsincos(P[3], &tr[0], &tr[1]);
  tsincos(P[4], &tr[2], &tr[3]);
  watson_parts_of(tr, P, CFP, vc, mc, extra, intra);
}

MACRO void Signal_Frame(int npar, T* P, T* fr, int changed) {
  T s, c;
  tsincos(changed == 3 ? P[3] : P[4], &s, &c);
  for (int k = 0; k < 2; ++k) {
    if (changed != 3 + k) continue;
    fr[2 * k] = s;
    fr[2 * k + 1] = c;
  }
}

MACRO T Predicted_Signal_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc, const T* fr) {
  T extra, intra;
  watson_parts_of(fr, P, CFP, vc, mc, extra, intra);
  const T aniso = ((T)1 - P[1]) * extra + P[1] * intra;
  return FixP[0] * (((T)1 - P[0]) * aniso + P[0] * (T)mc[7]);
}

MACRO T Predicted_Signal_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc) {
  T extra, intra;
  watson_parts(P, CFP, vc, mc, extra, intra);
  const T aniso = ((T)1 - P[1]) * extra + P[1] * intra;
  return FixP[0] * (((T)1 - P[0]) * aniso + P[0] * (T)mc[7]);
}

MACRO T Predicted_Signal(int npar, T* P, T* CFP, T* FixP) {
  CDM_F64 vc[9], mc[8];
  Voxel_Cache(npar, P, FixP, vc);
  Meas_Cache(CFP, mc);
  return Predicted_Signal_Cached(npar, P, CFP, FixP, vc, mc);
}

// GridSearch hooks: the same compartments from their shared parts.
MACRO void Grid_Table(int npar, T* P, CDM_F64* tb) {
  noddi_watson_sh((CDM_F64)P[2], tb);
  // dpar_eq of unit intra-axonal excess over zero perpendicular diffusivity:
  // both hindered diffusivities are linear in dpar - dperp (Grid_Outer)
  CDM_F64 dpar_eq, dperp_eq;
  noddi_watson_hindered((CDM_F64)P[2], 0.0, dpar_eq, dperp_eq);
  tb[7] = dpar_eq * (1.0 / CDM_NODDI_DPAR);
}

MACRO void Grid_Frame(int npar, T* P, T* fr) {
  T st, ct, sp, cp;
  tsincos(P[3], &st, &ct);
  tsincos(P[4], &sp, &cp);
  fr[0] = st * cp;
  fr[1] = st * sp;
  fr[2] = ct;
}

MACRO void Grid_Shared(int npar, T* P, T* CFP, T* FixP, const CDM_F64* tb, const T* fr, const CDM_F64* mc, T* sh) {
  T gn = CFP[0] * fr[0] + CFP[1] * fr[1] + CFP[2] * fr[2];
  sh[1] = gn * gn;
  if (gn > (T)1) gn = (T)1;
  if (gn < (T)-1) gn = (T)-1;
  CDM_F64 p[7], s = 0.0;
  noddi_even_legendre((CDM_F64)gn * (CDM_F64)gn, p);
  const CDM_F64 norm[7] = {0.28209479177387814, 0.6307831305050401, 0.8462843753216345, 1.0171072362820548,
                           1.1631066229203197,  1.2927207364566028, 1.4104739588693906};
  for (int l = 0; l < 7; ++l) s += mc[l] * tb[l] * (norm[l] * p[l]);
  if (s < 0) s = 1e-3;
  sh[0] = (T)(0.5 * s);
}

MACRO void Grid_Common(int npar, T* CFP, const CDM_F64* mc, T* cm) {
  cm[0] = CFP[3];
  cm[1] = (T)mc[7];
}

MACRO void Grid_Shared_Basis(int npar, const T* sh, const T* cm, T* basis) { basis[0] = cm[1]; }

MACRO void Grid_Outer(int npar, T* P, const CDM_F64* tb, T* so) {
  const CDM_F64 dperp = CDM_NODDI_DPAR * (1.0 - (CDM_F64)P[1]), d = CDM_NODDI_DPAR - dperp;
  const CDM_F64 dpar_eq = dperp + d * tb[7], dperp_eq = 0.5 * (CDM_NODDI_DPAR + dperp - d * tb[7]);
  so[0] = P[1];
  so[1] = (T)(dpar_eq - dperp_eq);
  so[2] = (T)dperp_eq;
}

MACRO void Grid_Outer_Basis(int npar, T* P, const T* cm, const T* so, const T* sh, T* basis) {
#ifdef CDM_WATSON_REFERENCE_FORMS
  const T e = exp_gpu(-cm[0] * (so[1] * sh[1] + so[2]));
#else
  const T e = texp_fast(-cm[0] * (so[1] * sh[1] + so[2]));
#endif
  basis[0] = ((T)1 - so[0]) * e + so[0] * sh[0];
}

MACRO void Grid_Weights(int npar, T* P, T* FixP, T* w) {
  w[0] = FixP[0] * P[0];
  w[1] = FixP[0] * ((T)1 - P[0]);
}

MACRO bool ConstraintsMCMC(int npar, T* P) { return true; }

// Analytic entries (fiso, fintra); the engine forms the others.
MACRO void Partial_Derivatives_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                      T* derivatives) {
  T extra, intra;
  watson_parts(P, CFP, vc, mc, extra, intra);
  const T aniso = ((T)1 - P[1]) * extra + P[1] * intra;
  derivatives[0] = FixP[0] * ((T)mc[7] - aniso);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (intra - extra);
}

// The signal of Predicted_Signal_Cached with the analytic entries of
// Partial_Derivatives_Cached, from one evaluation of the parts.
MACRO T Predicted_Signal_Partials_Cached(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                         T* derivatives) {
  T extra, intra;
  watson_parts(P, CFP, vc, mc, extra, intra);
  const T aniso = ((T)1 - P[1]) * extra + P[1] * intra;
  derivatives[0] = FixP[0] * ((T)mc[7] - aniso);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (intra - extra);
  return FixP[0] * (((T)1 - P[0]) * aniso + P[0] * (T)mc[7]);
}

MACRO T Predicted_Signal_Partials_Framed(int npar, T* P, T* CFP, T* FixP, const CDM_F64* vc, const CDM_F64* mc,
                                         T* derivatives, const T* fr) {
  T extra, intra;
  watson_parts_of(fr, P, CFP, vc, mc, extra, intra);
  const T aniso = ((T)1 - P[1]) * extra + P[1] * intra;
  derivatives[0] = FixP[0] * ((T)mc[7] - aniso);
  derivatives[1] = FixP[0] * ((T)1 - P[0]) * (intra - extra);
  return FixP[0] * (((T)1 - P[0]) * aniso + P[0] * (T)mc[7]);
}

MACRO void Partial_Derivatives(int npar, T* P, T* CFP, T* FixP, T* derivatives) {
  CDM_F64 vc[9], mc[8];
  Voxel_Cache(npar, P, FixP, vc);
  Meas_Cache(CFP, mc);
  Partial_Derivatives_Cached(npar, P, CFP, FixP, vc, mc, derivatives);
  derivatives[2] = NUMERICAL(2);
  derivatives[3] = NUMERICAL(3);
  derivatives[4] = NUMERICAL(4);
}

MACRO void FixConstraintsLM(int npar, T* P) {}

MACRO T custom_priors(int id_p, T* P, int nmeas, T* CFP, T* FixP) { return (T)0; }
