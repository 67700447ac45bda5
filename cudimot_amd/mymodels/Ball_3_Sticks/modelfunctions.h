// Ball and three sticks (no plain counterpart in the reference; written in
// the plug-in format by analogy with Ball_2_Sticks/modelfunctions.h:7-123).
//   S = S0 * [ (1-f1-f2-f3) exp(-b d) + sum_i fi exp(-b d (g.ni)^2) ]
// P: S0, d, f1, th1, ph1, f2, th2, ph2, f3, th3, ph3.  CFP: g (3), b (1).
// The Jacobian is the exact one (no ph2 quirk).
// The compartment exponentials use texp_fast (in single precision the
// hardware 2^y of y = x log2(e): relative error about |x| 2^-24 + 1 ulp,
// below what the float rounding of the argument b d (g.n)^2 itself
// brings); double-precision evaluations use the exact exp.

// tr: sine and cosine of th and of ph.
MACRO void b3s_directions(const T* CFP, const T* tr, T& gn, T& dth, T& dph) {
  const T st = tr[0], ct = tr[1], sp = tr[2], cp = tr[3];
  const T gxy = CFP[0] * cp + CFP[1] * sp;
  gn = st * gxy + CFP[2] * ct;
  dth = ct * gxy - st * CFP[2];
  dph = st * (CFP[1] * cp - CFP[0] * sp);
}

MACRO void b3s_stick(const T* CFP, T th, T ph, T& gn, T& dth, T& dph) {
  T tr[4];
  tsincos(th, &tr[0], &tr[1]);
  tsincos(ph, &tr[2], &tr[3]);
  b3s_directions(CFP, tr, gn, dth, dph);
}

MACRO T Predicted_Signal(int npar, T* P, T* CFP, T* FixP) {
  const T bd = CFP[3] * P[1];
  T s = ((T)1 - P[2] - P[5] - P[8]) * texp_fast(-bd);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    T g, u, v;
    b3s_stick(CFP, P[3 + 3 * k], P[4 + 3 * k], g, u, v);
    s += P[2 + 3 * k] * texp_fast(-bd * g * g);
  }
  return P[0] * s;
}

// MCMC hooks: the signal from the sines and cosines of the sticks' angles.
#define CDM_SIGNAL_FRAME 12
#define CDM_SIGNAL_FRAME_DEPENDS 0x6D8u

MACRO void Signal_Frame(int npar, T* P, T* fr, int changed) {
  const int angle[6] = {3, 4, 6, 7, 9, 10};
  T s, c;
  tsincos(changed == 3 ? P[3] : changed == 4 ? P[4] : changed == 6 ? P[6] : changed == 7 ? P[7] : changed == 9 ? P[9] : P[10], &s, &c);
  for (int k = 0; k < 6; ++k) {
    if (changed != angle[k]) continue;
    fr[2 * k] = s;
    fr[2 * k + 1] = c;
  }
}

MACRO T b3s_along(const T* CFP, const T* tr) {
  const T gxy = CFP[0] * tr[3] + CFP[1] * tr[2];
  return tr[0] * gxy + CFP[2] * tr[1];
}

MACRO T Predicted_Signal_Framed(int npar, T* P, T* CFP, T* FixP, const double* vc, const double* mc, const T* fr) {
  const T bd = CFP[3] * P[1];
  T s = ((T)1 - P[2] - P[5] - P[8]) * texp_fast(-bd);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const T g = b3s_along(CFP, fr + 4 * k);
    s += P[2 + 3 * k] * texp_fast(-bd * g * g);
  }
  return P[0] * s;
}

// GridSearch hooks: the signal is linear in the fractions and S0; the ball and the first two sticks
// are shared by the combinations of the last stick's angles.
#define CDM_GRID_LINEAR 0x125u        // S0, f1, f2, f3
#define CDM_GRID_SHARED 0xDAu        // d, th1, ph1, th2, ph2
#define CDM_GRID_SHARED_VALUES 3
#define CDM_GRID_SHARED_BASIS 3
#define CDM_GRID_OUTER_BASIS 1
#define CDM_GRID_COMMON 4              // g, b
#define CDM_GRID_FRAME 6
#define CDM_GRID_FRAME_DEPENDS 0xD8u
#define CDM_GRID_OUTER 3

MACRO void b3s_axis(T th, T ph, T* n) {
  T st, ct, sp, cp;
  tsincos(th, &st, &ct);
  tsincos(ph, &sp, &cp);
  n[0] = st * cp;
  n[1] = st * sp;
  n[2] = ct;
}

MACRO T b3s_compartment(const T* CFP, T d, const T* n) {
  const T g = CFP[0] * n[0] + CFP[1] * n[1] + CFP[2] * n[2];
  return texp_fast(-(CFP[3] * d) * g * g);
}

MACRO void Grid_Frame(int npar, T* P, T* fr) {
  b3s_axis(P[3], P[4], fr + 0);
  b3s_axis(P[6], P[7], fr + 3);
}

MACRO void Grid_Shared(int npar, T* P, T* CFP, T* FixP, const double* tb, const T* fr, const double* mc, T* sh) {
  sh[0] = texp_fast(-(CFP[3] * P[1]));
  sh[1] = b3s_compartment(CFP, P[1], fr + 0);
  sh[2] = b3s_compartment(CFP, P[1], fr + 3);
}

MACRO void Grid_Common(int npar, T* CFP, const double* mc, T* cm) {
  for (int k = 0; k < 4; ++k) cm[k] = CFP[k];
}

MACRO void Grid_Shared_Basis(int npar, const T* sh, const T* cm, T* basis) {
  basis[0] = sh[0];
  basis[1] = sh[1];
  basis[2] = sh[2];
}

MACRO void Grid_Outer(int npar, T* P, const double* tb, T* so) { b3s_axis(P[9], P[10], so); }

MACRO void Grid_Outer_Basis(int npar, T* P, const T* cm, const T* so, const T* sh, T* basis) {
  basis[0] = b3s_compartment(cm, P[1], so);
}

MACRO void Grid_Weights(int npar, T* P, T* FixP, T* w) {
  w[0] = P[0] * ((T)1 - P[2] - P[5] - P[8]);
  w[1] = P[0] * P[2];
  w[2] = P[0] * P[5];
  w[3] = P[0] * P[8];
}

MACRO bool ConstraintsMCMC(int npar, T* P) { return !(P[2] < P[5]) && !(P[5] < P[8]); }

MACRO void Partial_Derivatives_Framed(int npar, T* P, T* CFP, T* FixP, T* derivatives, const T* fr) {
  const T bd = CFP[3] * P[1];
  const T ball = texp_fast(-bd);
  const T fb = (T)1 - P[2] - P[5] - P[8];
  T mix = fb * ball, dmix = fb * ball;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    T g, dth, dph;
    b3s_directions(CFP, fr + 4 * k, g, dth, dph);
    const T sk = texp_fast(-bd * g * g);
    const T fk = P[2 + 3 * k];
    mix += fk * sk;
    dmix += fk * g * g * sk;
    derivatives[2 + 3 * k] = P[0] * (sk - ball);
    const T c = -(T)2 * P[0] * bd * fk * g * sk;
    derivatives[3 + 3 * k] = c * dth;
    derivatives[4 + 3 * k] = c * dph;
  }
  derivatives[0] = mix;
  derivatives[1] = -P[0] * CFP[3] * dmix;
}

MACRO void Partial_Derivatives(int npar, T* P, T* CFP, T* FixP, T* derivatives) {
  T fr[12];
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    tsincos(P[3 + 3 * k], &fr[4 * k], &fr[4 * k + 1]);
    tsincos(P[4 + 3 * k], &fr[4 * k + 2], &fr[4 * k + 3]);
  }
  Partial_Derivatives_Framed(npar, P, CFP, FixP, derivatives, fr);
}

// After LM: order the sticks by decreasing fraction.
MACRO void FixConstraintsLM(int npar, T* P) {
  for (int pass = 0; pass < 2; ++pass) {
    for (int a = 0; a < 2 - pass; ++a) {
      const int i = 2 + 3 * a, j = 2 + 3 * (a + 1);
      if (P[i] < P[j]) {
        for (int k = 0; k < 3; ++k) {
          const T t = P[i + k];
          P[i + k] = P[j + k];
          P[j + k] = t;
        }
      }
    }
  }
}

MACRO T custom_priors(int id_p, T* P, int nmeas, T* CFP, T* FixP) { return (T)0; }
