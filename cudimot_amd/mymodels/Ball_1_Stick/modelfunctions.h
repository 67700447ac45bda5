// Ball and one stick.
//   S = S0 * [ (1-f) exp(-b d) + f exp(-b d (g.n)^2) ]
//   n = (sin th cos ph, sin th sin ph, cos th)
// P: S0, d, f, th, ph.  CFP: g (3), b (1).
// Forward model and analytic Jacobian follow Ball_1_Stick/modelfunctions.h:11-77.
// The compartment exponentials use texp_fast (in single precision the
// hardware 2^y of y = x log2(e): relative error about |x| 2^-24 + 1 ulp,
// below what the float rounding of the argument b d (g.n)^2 itself
// brings); double-precision evaluations use the exact exp.

// tr: sine and cosine of th and of ph.
MACRO void b1s_directions(const T* CFP, const T* tr, T& gn, T& dgn_dth, T& dgn_dph) {
  const T st = tr[0], ct = tr[1], sp = tr[2], cp = tr[3];
  const T gxy = CFP[0] * cp + CFP[1] * sp;  // g projected on the stick azimuth
  gn = st * gxy + CFP[2] * ct;
  dgn_dth = ct * gxy - st * CFP[2];
  dgn_dph = st * (CFP[1] * cp - CFP[0] * sp);
}

MACRO void b1s_geometry(const T* P, const T* CFP, T& gn, T& dgn_dth, T& dgn_dph) {
  T tr[4];
  tsincos(P[3], &tr[0], &tr[1]);
  tsincos(P[4], &tr[2], &tr[3]);
  b1s_directions(CFP, tr, gn, dgn_dth, dgn_dph);
}

MACRO T Predicted_Signal(int npar, T* P, T* CFP, T* FixP) {
  T gn, a, b;
  b1s_geometry(P, CFP, gn, a, b);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T stick = texp_fast(-bd * gn * gn);
  return P[0] * (((T)1 - P[2]) * ball + P[2] * stick);
}

// MCMC hooks: the signal from the sines and cosines of the stick's angles.
#define CDM_SIGNAL_FRAME 4
#define CDM_SIGNAL_FRAME_DEPENDS 0x18u

MACRO void Signal_Frame(int npar, T* P, T* fr, int changed) {
  const int angle[2] = {3, 4};
  T s, c;
  tsincos(changed == 3 ? P[3] : P[4], &s, &c);
  for (int k = 0; k < 2; ++k) {
    if (changed != angle[k]) continue;
    fr[2 * k] = s;
    fr[2 * k + 1] = c;
  }
}

MACRO T b1s_along(const T* CFP, const T* tr) {
  const T gxy = CFP[0] * tr[3] + CFP[1] * tr[2];
  return tr[0] * gxy + CFP[2] * tr[1];
}

MACRO T Predicted_Signal_Framed(int npar, T* P, T* CFP, T* FixP, const double* vc, const double* mc, const T* fr) {
  const T gn = b1s_along(CFP, fr);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T stick = texp_fast(-bd * gn * gn);
  return P[0] * (((T)1 - P[2]) * ball + P[2] * stick);
}

// GridSearch hooks: the signal is linear in the fraction and S0; the ball is
// shared by the combinations of the stick's angles.
#define CDM_GRID_LINEAR 0x05u        // S0, f
#define CDM_GRID_SHARED 0x02u        // d
#define CDM_GRID_SHARED_VALUES 1
#define CDM_GRID_SHARED_BASIS 1
#define CDM_GRID_OUTER_BASIS 1
#define CDM_GRID_COMMON 4              // g, b
#define CDM_GRID_FRAME 0
#define CDM_GRID_FRAME_DEPENDS 0x00u
#define CDM_GRID_OUTER 3

MACRO void b1s_axis(T th, T ph, T* n) {
  T st, ct, sp, cp;
  tsincos(th, &st, &ct);
  tsincos(ph, &sp, &cp);
  n[0] = st * cp;
  n[1] = st * sp;
  n[2] = ct;
}

MACRO T b1s_compartment(const T* CFP, T d, const T* n) {
  const T g = CFP[0] * n[0] + CFP[1] * n[1] + CFP[2] * n[2];
  return texp_fast(-(CFP[3] * d) * g * g);
}

MACRO void Grid_Frame(int npar, T* P, T* fr) {}

MACRO void Grid_Shared(int npar, T* P, T* CFP, T* FixP, const double* tb, const T* fr, const double* mc, T* sh) {
  sh[0] = texp_fast(-(CFP[3] * P[1]));
}

MACRO void Grid_Common(int npar, T* CFP, const double* mc, T* cm) {
  for (int k = 0; k < 4; ++k) cm[k] = CFP[k];
}

MACRO void Grid_Shared_Basis(int npar, const T* sh, const T* cm, T* basis) {
  basis[0] = sh[0];
}

MACRO void Grid_Outer(int npar, T* P, const double* tb, T* so) { b1s_axis(P[3], P[4], so); }

MACRO void Grid_Outer_Basis(int npar, T* P, const T* cm, const T* so, const T* sh, T* basis) {
  basis[0] = b1s_compartment(cm, P[1], so);
}

MACRO void Grid_Weights(int npar, T* P, T* FixP, T* w) {
  w[0] = P[0] * ((T)1 - P[2]);
  w[1] = P[0] * P[2];
}

MACRO bool ConstraintsMCMC(int npar, T* P) { return true; }

MACRO void Partial_Derivatives_Framed(int npar, T* P, T* CFP, T* FixP, T* derivatives, const T* fr) {
  T gn, dth, dph;
  b1s_directions(CFP, fr, gn, dth, dph);
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T stick = texp_fast(-bd * gn * gn);
  const T f = P[2];
  derivatives[0] = ((T)1 - f) * ball + f * stick;
  derivatives[1] = -P[0] * CFP[3] * (((T)1 - f) * ball + f * gn * gn * stick);
  derivatives[2] = P[0] * (stick - ball);
  const T common = -(T)2 * P[0] * bd * f * gn * stick;  // dS/d(gn) / ... chain factor
  derivatives[3] = common * dth;
  derivatives[4] = common * dph;
}

MACRO void Partial_Derivatives(int npar, T* P, T* CFP, T* FixP, T* derivatives) {
  T fr[4];
  tsincos(P[3], &fr[0], &fr[1]);
  tsincos(P[4], &fr[2], &fr[3]);
  Partial_Derivatives_Framed(npar, P, CFP, FixP, derivatives, fr);
}

MACRO void FixConstraintsLM(int npar, T* P) {}

MACRO T custom_priors(int id_p, T* P, int nmeas, T* CFP, T* FixP) { return (T)0; }
