// Ball and two sticks.
//   S = S0 * [ (1-f1-f2) exp(-b d) + f1 exp(-b d (g.n1)^2) + f2 exp(-b d (g.n2)^2) ]
// P: S0, d, f1, th1, ph1, f2, th2, ph2.  CFP: g (3), b (1).
// Follows Ball_2_Sticks/modelfunctions.h:7-123.
//
// Reference parity: the reference's dS/dph2 reuses the th2 chain factor
// (Ball_2_Sticks/modelfunctions.h:99-103), so its Levenberg-Marquardt moves
// ph2 along the th2 derivative.  That behaviour is kept by default so fits
// reproduce the reference; define CDM_B2S_EXACT_PHI2 to use the true
// derivative.
// The compartment exponentials use texp_fast (in single precision the
// hardware 2^y of y = x log2(e): relative error about |x| 2^-24 + 1 ulp,
// below what the float rounding of the argument b d (g.n)^2 itself
// brings); double-precision evaluations use the exact exp.

// tr: sine and cosine of th and of ph.
MACRO void b2s_directions(const T* CFP, const T* tr, T& gn, T& dth, T& dph) {
  const T st = tr[0], ct = tr[1], sp = tr[2], cp = tr[3];
  const T gxy = CFP[0] * cp + CFP[1] * sp;
  gn = st * gxy + CFP[2] * ct;
  dth = ct * gxy - st * CFP[2];
  dph = st * (CFP[1] * cp - CFP[0] * sp);
}

MACRO void b2s_stick(const T* CFP, T th, T ph, T& gn, T& dth, T& dph) {
  T tr[4];
  tsincos(th, &tr[0], &tr[1]);
  tsincos(ph, &tr[2], &tr[3]);
  b2s_directions(CFP, tr, gn, dth, dph);
}

MACRO T Predicted_Signal(int npar, T* P, T* CFP, T* FixP) {
  T g1, g2, u, v;
  b2s_stick(CFP, P[3], P[4], g1, u, v);
  b2s_stick(CFP, P[6], P[7], g2, u, v);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T s1 = texp_fast(-bd * g1 * g1);
  const T s2 = texp_fast(-bd * g2 * g2);
  return P[0] * (((T)1 - P[2] - P[5]) * ball + P[2] * s1 + P[5] * s2);
}

// MCMC hooks: the signal from the sines and cosines of the sticks' angles.
#define CDM_SIGNAL_FRAME 8
#define CDM_SIGNAL_FRAME_DEPENDS 0xD8u

MACRO void Signal_Frame(int npar, T* P, T* fr, int changed) {
  const int angle[4] = {3, 4, 6, 7};
  T s, c;
  tsincos(changed == 3 ? P[3] : changed == 4 ? P[4] : changed == 6 ? P[6] : P[7], &s, &c);
  for (int k = 0; k < 4; ++k) {
    if (changed != angle[k]) continue;
    fr[2 * k] = s;
    fr[2 * k + 1] = c;
  }
}

MACRO T b2s_along(const T* CFP, const T* tr) {
  const T gxy = CFP[0] * tr[3] + CFP[1] * tr[2];
  return tr[0] * gxy + CFP[2] * tr[1];
}

MACRO T Predicted_Signal_Framed(int npar, T* P, T* CFP, T* FixP, const double* vc, const double* mc, const T* fr) {
  const T g1 = b2s_along(CFP, fr), g2 = b2s_along(CFP, fr + 4);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T s1 = texp_fast(-bd * g1 * g1);
  const T s2 = texp_fast(-bd * g2 * g2);
  return P[0] * (((T)1 - P[2] - P[5]) * ball + P[2] * s1 + P[5] * s2);
}

// GridSearch hooks: the signal is linear in the fractions and S0; the ball and the first stick
// are shared by the combinations of the last stick's angles.
#define CDM_GRID_LINEAR 0x25u        // S0, f1, f2
#define CDM_GRID_SHARED 0x1Au        // d, th1, ph1
#define CDM_GRID_SHARED_VALUES 2
#define CDM_GRID_SHARED_BASIS 2
#define CDM_GRID_OUTER_BASIS 1
#define CDM_GRID_COMMON 4              // g, b
#define CDM_GRID_FRAME 3
#define CDM_GRID_FRAME_DEPENDS 0x18u
#define CDM_GRID_OUTER 3

MACRO void b2s_axis(T th, T ph, T* n) {
  T st, ct, sp, cp;
  tsincos(th, &st, &ct);
  tsincos(ph, &sp, &cp);
  n[0] = st * cp;
  n[1] = st * sp;
  n[2] = ct;
}

MACRO T b2s_compartment(const T* CFP, T d, const T* n) {
  const T g = CFP[0] * n[0] + CFP[1] * n[1] + CFP[2] * n[2];
  return texp_fast(-(CFP[3] * d) * g * g);
}

MACRO void Grid_Frame(int npar, T* P, T* fr) {
  b2s_axis(P[3], P[4], fr + 0);
}

MACRO void Grid_Shared(int npar, T* P, T* CFP, T* FixP, const double* tb, const T* fr, const double* mc, T* sh) {
  sh[0] = texp_fast(-(CFP[3] * P[1]));
  sh[1] = b2s_compartment(CFP, P[1], fr + 0);
}

MACRO void Grid_Common(int npar, T* CFP, const double* mc, T* cm) {
  for (int k = 0; k < 4; ++k) cm[k] = CFP[k];
}

MACRO void Grid_Shared_Basis(int npar, const T* sh, const T* cm, T* basis) {
  basis[0] = sh[0];
  basis[1] = sh[1];
}

MACRO void Grid_Outer(int npar, T* P, const double* tb, T* so) { b2s_axis(P[6], P[7], so); }

MACRO void Grid_Outer_Basis(int npar, T* P, const T* cm, const T* so, const T* sh, T* basis) {
  basis[0] = b2s_compartment(cm, P[1], so);
}

MACRO void Grid_Weights(int npar, T* P, T* FixP, T* w) {
  w[0] = P[0] * ((T)1 - P[2] - P[5]);
  w[1] = P[0] * P[2];
  w[2] = P[0] * P[5];
}

MACRO bool ConstraintsMCMC(int npar, T* P) { return !(P[2] < P[5]); }

MACRO void Partial_Derivatives_Framed(int npar, T* P, T* CFP, T* FixP, T* derivatives, const T* fr) {
  T g1, d1th, d1ph, g2, d2th, d2ph;
  b2s_directions(CFP, fr, g1, d1th, d1ph);
  b2s_directions(CFP, fr + 4, g2, d2th, d2ph);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T s1 = texp_fast(-bd * g1 * g1);
  const T s2 = texp_fast(-bd * g2 * g2);
  const T fb = (T)1 - P[2] - P[5];
  derivatives[0] = fb * ball + P[2] * s1 + P[5] * s2;
  derivatives[1] = -P[0] * CFP[3] * (fb * ball + P[2] * g1 * g1 * s1 + P[5] * g2 * g2 * s2);
  derivatives[2] = P[0] * (s1 - ball);
  const T c1 = -(T)2 * P[0] * bd * P[2] * g1 * s1;
  derivatives[3] = c1 * d1th;
  derivatives[4] = c1 * d1ph;
  derivatives[5] = P[0] * (s2 - ball);
  const T c2 = -(T)2 * P[0] * bd * P[5] * g2 * s2;
  derivatives[6] = c2 * d2th;
#ifdef CDM_B2S_EXACT_PHI2
  derivatives[7] = c2 * d2ph;
#else
  derivatives[7] = c2 * d2th;
#endif
}

MACRO void Partial_Derivatives(int npar, T* P, T* CFP, T* FixP, T* derivatives) {
  T fr[8];
  tsincos(P[3], &fr[0], &fr[1]);
  tsincos(P[4], &fr[2], &fr[3]);
  tsincos(P[6], &fr[4], &fr[5]);
  tsincos(P[7], &fr[6], &fr[7]);
  Partial_Derivatives_Framed(npar, P, CFP, FixP, derivatives, fr);
}

// After LM: keep the larger stick first (swap f, th, ph of the two sticks).
MACRO void FixConstraintsLM(int npar, T* P) {
  if (P[2] < P[5]) {
    for (int k = 0; k < 3; ++k) {
      const T t = P[2 + k];
      P[2 + k] = P[5 + k];
      P[5 + k] = t;
    }
  }
}

MACRO T custom_priors(int id_p, T* P, int nmeas, T* CFP, T* FixP) { return (T)0; }
