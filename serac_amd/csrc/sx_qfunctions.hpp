// sx_qfunctions.hpp -- device quadrature-point functions (the compiled
// integrand registry) and the single-direction dual number they run on.
//
// Each functor evaluates physical-space (source, flux) from physical-space
// (value, grad) for a scalar type T in {double, sxk::d1}; directional
// derivatives (the shape gradient) come from running the same code on d1 with
// one seeded direction per pass (fn/dual.hpp:28-147 propagates every gradient
// slot by this same arithmetic); the stored tangent has a closed form.
#pragma once

#include <hip/hip_runtime.h>

namespace sxk {

// ---------------------------------------------------------------------------
// single-direction dual number: value v, directional derivative d
// ---------------------------------------------------------------------------
struct d1 {
  double v, d;
  __device__ __forceinline__ d1() : v(0.0), d(0.0) {}
  __device__ __forceinline__ d1(double x) : v(x), d(0.0) {}
  __device__ __forceinline__ d1(double x, double y) : v(x), d(y) {}
};
__device__ __forceinline__ d1 operator+(d1 a, d1 b) { return d1(a.v + b.v, a.d + b.d); }
__device__ __forceinline__ d1 operator-(d1 a, d1 b) { return d1(a.v - b.v, a.d - b.d); }
__device__ __forceinline__ d1 operator-(d1 a) { return d1(-a.v, -a.d); }
__device__ __forceinline__ d1 operator*(d1 a, d1 b) { return d1(a.v * b.v, a.v * b.d + a.d * b.v); }
__device__ __forceinline__ d1 operator*(double a, d1 b) { return d1(a * b.v, a * b.d); }
__device__ __forceinline__ d1 operator*(d1 b, double a) { return d1(a * b.v, a * b.d); }
__device__ __forceinline__ d1 operator+(d1 a, double b) { return d1(a.v + b, a.d); }
__device__ __forceinline__ d1 operator+(double b, d1 a) { return d1(a.v + b, a.d); }
__device__ __forceinline__ d1 operator-(d1 a, double b) { return d1(a.v - b, a.d); }
__device__ __forceinline__ d1 operator/(d1 a, d1 b)
{
  return d1(a.v / b.v, (a.d * b.v - a.v * b.d) / (b.v * b.v));
}
__device__ __forceinline__ d1 operator/(d1 a, double b) { return d1(a.v / b, a.d / b); }
__device__ __forceinline__ d1 operator/(double a, d1 b) { return d1(a / b.v, -(a / (b.v * b.v)) * b.d); }
__device__ __forceinline__ d1 dlog1p(d1 a) { return d1(::log1p(a.v), a.d / (1.0 + a.v)); }
__device__ __forceinline__ d1 dsqrt(d1 a) { return d1(::sqrt(a.v), a.d / (2.0 * ::sqrt(a.v))); }
__device__ __forceinline__ double dsqrt(double a) { return ::sqrt(a); }
// the derivative of a root x(q) of f(x, q) = 0 with df/dq = 1: x' = -q' / df_dx
__device__ __forceinline__ double root_dual(double x, double, double) { return x; }
__device__ __forceinline__ d1 root_dual(double x, d1 q, double df_dx) { return d1(x, -q.d / df_dx); }
__device__ __forceinline__ double dlog1p(double a) { return ::log1p(a); }
__device__ __forceinline__ double vpart(double a) { return a; }
__device__ __forceinline__ double vpart(d1 a) { return a.v; }
__device__ __forceinline__ double dpart(double) { return 0.0; }
__device__ __forceinline__ double dpart(d1 a) { return a.d; }

// ---------------------------------------------------------------------------
// 3x3 helpers on row-major arrays, restating fn/tensor.hpp:1242-1290 (det,
// detApIm1) and :1610-1630 (inv)
// ---------------------------------------------------------------------------
template <typename T>
__device__ __forceinline__ T det3(const T* A)
{
  return A[0] * A[4] * A[8] + A[1] * A[5] * A[6] + A[2] * A[3] * A[7] - A[0] * A[5] * A[7] - A[1] * A[3] * A[8] -
         A[2] * A[4] * A[6];
}

// det(A + I) - 1 = tr A + I2(A) + det A, evaluated without cancellation
template <typename T>
__device__ __forceinline__ T det_ap_i_m1(const T* A)
{
  return A[0] + A[4] + A[8] - A[1] * A[3] * (1.0 + A[8]) + A[0] * A[4] * (1.0 + A[8]) -
         A[2] * A[6] * (1.0 + A[4]) - A[5] * A[7] * (1.0 + A[0]) + A[0] * A[8] + A[4] * A[8] +
         A[1] * A[5] * A[6] + A[2] * A[3] * A[7];
}

template <typename T>
__device__ __forceinline__ void inv3(const T* A, T* R)
{
  T id = 1.0 / det3(A);
  R[0] = (A[4] * A[8] - A[5] * A[7]) * id;
  R[1] = (A[2] * A[7] - A[1] * A[8]) * id;
  R[2] = (A[1] * A[5] - A[2] * A[4]) * id;
  R[3] = (A[5] * A[6] - A[3] * A[8]) * id;
  R[4] = (A[0] * A[8] - A[2] * A[6]) * id;
  R[5] = (A[2] * A[3] - A[0] * A[5]) * id;
  R[6] = (A[3] * A[7] - A[4] * A[6]) * id;
  R[7] = (A[1] * A[6] - A[0] * A[7]) * id;
  R[8] = (A[0] * A[4] - A[1] * A[3]) * id;
}

// cofactors of F = I + H: C = det(F) inv(F)^T
template <typename T>
__device__ __forceinline__ void cof_i_plus(const T* H, T* C)
{
  const T a = H[0] + 1.0, e = H[4] + 1.0, i = H[8] + 1.0;
  C[0] = e * i - H[5] * H[7];
  C[1] = H[5] * H[6] - H[3] * i;
  C[2] = H[3] * H[7] - e * H[6];
  C[3] = H[2] * H[7] - H[1] * i;
  C[4] = a * i - H[2] * H[6];
  C[5] = H[1] * H[6] - a * H[7];
  C[6] = H[1] * H[5] - H[2] * e;
  C[7] = H[2] * H[3] - a * H[5];
  C[8] = a * e - H[1] * H[3];
}

// R[c][a] = sum_k A[c][k] Ji[a][k]: a physical-space index taken to the parent element
__device__ __forceinline__ void to_parent(const double* A, const double* Ji, double* R)
{
#pragma unroll
  for (int c = 0; c < 3; c++)
#pragma unroll
    for (int a = 0; a < 3; a++)
      R[c * 3 + a] = A[c * 3 + 0] * Ji[a * 3 + 0] + A[c * 3 + 1] * Ji[a * 3 + 1] + A[c * 3 + 2] * Ji[a * 3 + 2];
}

// M = f Ji Ji^T
__device__ __forceinline__ void gram(const double* Ji, double f, double* M)
{
#pragma unroll
  for (int a = 0; a < 3; a++)
#pragma unroll
    for (int b = a; b < 3; b++)
      M[a * 3 + b] = M[b * 3 + a] =
          f * (Ji[a * 3 + 0] * Ji[b * 3 + 0] + Ji[a * 3 + 1] * Ji[b * 3 + 1] + Ji[a * 3 + 2] * Ji[b * 3 + 2]);
}

// ---------------------------------------------------------------------------
// qfunctions.  tangent() gives the derivative of the parent-space outputs
// ([source] and flux, times det J) with respect to the parent-space inputs
// ([value] and gradient) entry by entry: emit(r, s, D(r, s)) for every stored
// entry, column s by column s with r increasing (the upper triangle of a
// symmetric tangent).  It restates eval()'s derivative in closed form: the
// forward-mode passes it stands for carried the whole integrand through one
// dual per column, 9 (12) times the work of the values, and made the
// linearization compute-bound (Neo-Hookean p = 3 on 48x40x44 elements: 1196
// us of kernel time with the passes, 505 with the closed form, 330 for the
// tangent's bytes alone; J2 p = 2 on 56x48x50: 1463, 672 and 400).
// CONSTANT_TANGENT: it does not depend on the field.  HAS_SOURCE: the source
// output is nonzero; USES_VALUE: the outputs depend on the field value (not only
// its gradient).
// ---------------------------------------------------------------------------

// steady heat conduction: ThermalMaterialIntegrand<LinearIsotropicConductor>
// plus setSource (phy/heat_transfer.hpp:381-406, 493-503;
// phy/materials/thermal_material.hpp:50-55).  p = {k, s}
struct QFHeat {
  static constexpr int  NC         = 1;
  static constexpr bool HAS_SOURCE = true;
  static constexpr bool USES_VALUE = false;
  static constexpr int  STATE      = 0;
  static constexpr bool CONSTANT_TANGENT = true;
  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T*, const T* g, T* src, T* flux)
  {
    src[0]  = T(-p[1]);
    flux[0] = p[0] * g[0];
    flux[1] = p[0] * g[1];
    flux[2] = p[0] * g[2];
  }
  template <class Emit>
  __device__ __forceinline__ static void tangent(const double* p, const double*, const double* Ji, double dJ,
                                                 const double*, Emit&& emit)
  {
    double M[9];
    gram(Ji, p[0] * dJ, M);
#pragma unroll
    for (int s = 0; s < 3; s++)
#pragma unroll
      for (int r = 0; r <= s; r++) emit(r, s, M[r * 3 + s]);
  }
};

// mass + diffusion {a u, b grad u} (fn/tests/functional_comparisons.cpp:32-33)
template <int C>
struct QFMassDiffusion {
  static constexpr int  NC         = C;
  static constexpr bool HAS_SOURCE = true;
  static constexpr bool USES_VALUE = true;
  static constexpr int  STATE      = 0;
  static constexpr bool CONSTANT_TANGENT = true;
  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T* v, const T* g, T* src, T* flux)
  {
#pragma unroll
    for (int c = 0; c < C; c++) {
      src[c] = p[0] * v[c];
#pragma unroll
      for (int d = 0; d < 3; d++) flux[c * 3 + d] = p[1] * g[c * 3 + d];
    }
  }
  template <class Emit>
  __device__ __forceinline__ static void tangent(const double* p, const double*, const double* Ji, double dJ,
                                                 const double*, Emit&& emit)
  {
    double M[9];
    gram(Ji, p[1] * dJ, M);
#pragma unroll
    for (int s = 0; s < 4 * C; s++)
#pragma unroll
      for (int r = 0; r <= s; r++) {
        double v = 0.0;
        if (s < C && r == s) v = p[0] * dJ;
        if (r >= C && (r - C) / 3 == (s - C) / 3) v = M[((r - C) % 3) * 3 + (s - C) % 3];
        emit(r, s, v);
      }
  }
};

// MaterialStressFunctor<NeoHookean> with geometric nonlinearity
// (phy/solid_mechanics.hpp:834-852; phy/materials/solid_material.hpp:112-122):
//   sigma = (lambda log1p(J-1) I + G (H H^T + H^T + H)) / J,  lambda = K - 2G/3
//   flux  = sigma . inv(I + H)^T . det(I + H);   source = density * 0 (quasi-static)
// p = {density, K, G}
struct QFNeoHookean {
  static constexpr int  NC         = 3;
  static constexpr bool HAS_SOURCE = false;
  static constexpr bool USES_VALUE = false;
  static constexpr int  STATE      = 0;
  static constexpr bool CONSTANT_TANGENT = false;
  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T*, const T* H, T*, T* flux)
  {
    const double K = p[1], G = p[2];
    const double lambda = K - (2.0 / 3.0) * G;
    T            Jm1, iJ, C[9];
    kinematics(H, &Jm1, &iJ, C);
    const T L = lambda * dlog1p(Jm1);
    T       tau[9];  // J sigma, without the cancellation of F F^T - I
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = i; j < 3; j++) {
        const T hht = H[i * 3 + 0] * H[j * 3 + 0] + H[i * 3 + 1] * H[j * 3 + 1] + H[i * 3 + 2] * H[j * 3 + 2];
        T       v   = G * (hht + H[j * 3 + i] + H[i * 3 + j]);
        if (i == j) v = v + L;
        tau[i * 3 + j] = tau[j * 3 + i] = v;
      }
    // (tau / J) inv(F)^T det(F) = tau cof(F) / J: one division in all
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++)
        flux[i * 3 + j] =
            (tau[i * 3 + 0] * C[0 * 3 + j] + tau[i * 3 + 1] * C[1 * 3 + j] + tau[i * 3 + 2] * C[2 * 3 + j]) * iJ;
  }
  // det(F) - 1, 1 / det(F) and the cofactors of F = I + H
  template <typename T>
  __device__ __forceinline__ static void kinematics(const T* H, T* Jm1, T* iJ, T* C)
  {
    *Jm1 = det_ap_i_m1(H);
    *iJ  = 1.0 / (*Jm1 + 1.0);
    cof_i_plus(H, C);
  }
  // dP = G dF + lambda (F^-T : dF) F^-T + (G - lambda ln J) F^-T dF^T F^-T, with each slot of dF and of dP taken to
  // the parent element: W = F^-T Ji^T, M = Ji Ji^T
  template <class Emit>
  __device__ __forceinline__ static void tangent(const double* p, const double* H, const double* Ji, double dJ,
                                                 const double*, Emit&& emit)
  {
    const double K = p[1], G = p[2];
    const double lambda = K - (2.0 / 3.0) * G;
    double       Jm1, iJ, C[9], W[9], M[9];
    kinematics(H, &Jm1, &iJ, C);
    to_parent(C, Ji, W);
#pragma unroll
    for (int k = 0; k < 9; k++) W[k] *= iJ;
    gram(Ji, G * dJ, M);
    const double cl = dJ * lambda, cg = dJ * (G - lambda * dlog1p(Jm1));
#pragma unroll
    for (int s = 0; s < 9; s++) {
      const int    c2 = s / 3, b = s % 3;
      const double wl = cl * W[s];
#pragma unroll
      for (int r = 0; r <= s; r++) {
        const int c = r / 3, a = r % 3;
        double    v = wl * W[r] + (cg * W[c * 3 + b]) * W[c2 * 3 + a];
        if (c == c2) v += M[a * 3 + b];
        emit(r, s, v);
      }
    }
  }
};

// gradient of the quantity of interest  int u_c dV  (Functional<double(trial)>,
// fn/functional_qoi.inl): source e_c, no flux.  p = {c}
template <int C>
struct QFQoiValue {
  static constexpr int  NC         = C;
  static constexpr bool HAS_SOURCE = true;
  static constexpr bool USES_VALUE = false;
  static constexpr int  STATE      = 0;
  static constexpr bool CONSTANT_TANGENT = true;
  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T*, const T*, T* src, T* flux)
  {
    const int c0 = int(p[0]);
#pragma unroll
    for (int c = 0; c < C; c++) {
      src[c] = T(c == c0 ? 1.0 : 0.0);
#pragma unroll
      for (int d = 0; d < 3; d++) flux[c * 3 + d] = T(0.0);
    }
  }
};

// small-strain linear elasticity: sigma = lambda tr(eps) I + 2 mu eps.  p = {lambda, mu}
struct QFLinearElastic {
  static constexpr int  NC         = 3;
  static constexpr bool HAS_SOURCE = false;
  static constexpr bool USES_VALUE = false;
  static constexpr int  STATE      = 0;
  static constexpr bool CONSTANT_TANGENT = true;
  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T*, const T* g, T*, T* flux)
  {
    const double lam = p[0], mu = p[1];
    T            tr  = g[0] + g[4] + g[8];
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) {
        T v = mu * (g[i * 3 + j] + g[j * 3 + i]);
        if (i == j) v = v + lam * tr;
        flux[i * 3 + j] = v;
      }
  }
  template <class Emit>
  __device__ __forceinline__ static void tangent(const double* p, const double*, const double* Ji, double dJ,
                                                 const double*, Emit&& emit)
  {
    const double cl = p[0] * dJ, cm = p[1] * dJ;
    double       M[9];
    gram(Ji, cm, M);
#pragma unroll
    for (int s = 0; s < 9; s++) {
      const int c2 = s / 3, b = s % 3;
#pragma unroll
      for (int r = 0; r <= s; r++) {
        const int c = r / 3, a = r % 3;
        double    v = cl * (Ji[a * 3 + c] * Ji[b * 3 + c2]) + cm * (Ji[a * 3 + c2] * Ji[b * 3 + c]);
        if (c == c2) v += M[a * 3 + b];
        emit(r, s, v);
      }
    }
  }
};

// flux = sigma . inv(F)^T . det(F), F = I + H (MaterialStressFunctor with
// geometric nonlinearity, phy/solid_mechanics.hpp:843-849)
template <typename T>
__device__ __forceinline__ void stress_to_flux_large(const T* sig, const T* H, T* flux)
{
  T C[9];  // inv(F)^T det(F)
  cof_i_plus(H, C);
#pragma unroll
  for (int i = 0; i < 3; i++)
#pragma unroll
    for (int j = 0; j < 3; j++)
      flux[i * 3 + j] = sig[i * 3 + 0] * C[0 * 3 + j] + sig[i * 3 + 1] * C[1 * 3 + j] + sig[i * 3 + 2] * C[2 * 3 + j];
}

// MaterialStressFunctor<J2SmallStrain<LinearHardening>>, quasi-static
// (phy/materials/solid_material.hpp:132-148, 199-258; phy/solid_mechanics.hpp:834-852).
// p = {E, nu, sigma_y, Hi, Hk, density, geom_nonlin}.  st = {plastic strain
// [3][3] row-major, accumulated plastic strain}: the caller's copy of the
// point's state, updated in place when the return map runs.
//
// The return map solves the consistency residual
//   f(x) = q - (3G + Hk) x - (sigma_y + Hi (eqps_old + x))
// with the bracketed Newton/bisection of solve_scalar_equation
// (fn/tuple_tensor_dual_functions.hpp:573-672) on values; the dual part of
// the root is -q' / df_dx.  A root that is not bracketed (the reference
// aborts there) returns NaN stresses.
struct QFJ2 {
  static constexpr int    NC         = 3;
  static constexpr bool   HAS_SOURCE = false;
  static constexpr bool   USES_VALUE = false;
  static constexpr int    STATE      = 10;
  static constexpr bool CONSTANT_TANGENT = false;
  static constexpr double TOL        = 1e-10;

  __device__ __forceinline__ static double solve(double q, double a, double sy, double Hi, double e0, double hi,
                                                 double* df_out)
  {
    const double dfdx = -a - Hi;
    const double lo   = 0.0;
    const double rtol = TOL * sy;
    auto         f    = [&](double x) { return q - a * x - (sy + Hi * (e0 + x)); };
    const double fl = f(lo), fh = f(hi);
    *df_out         = dfdx;
    if (fl * fh > 0) return __builtin_nan("");
    if (fl == 0) return lo;
    if (fh == 0) return hi;
    double xl = lo, xh = hi;
    if (fl > 0) {
      xl = hi;
      xh = lo;
    }
    double x = 0.0;  // initial guess, inside [lo, hi]
    double dx_old = fabs(hi - lo), dx = dx_old, fval = f(x);
    bool   conv = false;
    for (int it = 0; it < 25 && !conv; it++) {
      if ((x - xh) * dfdx - fval > 0 || (x - xl) * dfdx - fval < 0 || fabs(2. * fval) > fabs(dx_old * dfdx)) {
        dx_old = dx;
        dx     = 0.5 * (xh - xl);
        x      = xl + dx;
        conv   = (x == xl);
      } else {
        dx_old         = dx;
        dx             = fval / dfdx;
        const double t = x;
        x -= dx;
        conv = (x == t);
      }
      fval = f(x);
      conv = conv || (fabs(fval) < rtol);
      if (fval < 0)
        xl = x;
      else
        xh = x;
    }
    return x;
  }

  // elastic trial state: s = 2G dev(eps_e) (with dev taken of the trace part only), eta = s - (2/3) Hk plastic
  // strain, pr = K tr(eps_e); returns q = sqrt(3/2) |eta|
  template <typename T>
  __device__ __forceinline__ static T trial(double K, double G, double Hk, const T* H, const double* st, T* s, T* eta,
                                            T* pr)
  {
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int j = 0; j < 3; j++) s[i * 3 + j] = 0.5 * (H[i * 3 + j] + H[j * 3 + i]) - st[i * 3 + j];
    const T tr = s[0] + s[4] + s[8];
    *pr        = K * tr;
#pragma unroll
    for (int i = 0; i < 3; i++) s[i * 4] = s[i * 4] - tr / 3.0;
    T sq = T(0.0);
#pragma unroll
    for (int k = 0; k < 9; k++) {
      s[k]   = (2.0 * G) * s[k];
      eta[k] = s[k] - ((2.0 / 3.0) * Hk) * st[k];
      sq     = sq + eta[k] * eta[k];
    }
    return 1.2247448713915890491 * dsqrt(sq);  // sqrt(1.5)
  }

  template <typename T>
  __device__ __forceinline__ static void eval(const double* p, const T*, const T* H, T*, T* flux, double* st)
  {
    const double E = p[0], nu = p[1], sy = p[2], Hi = p[3], Hk = p[4];
    const double K = E / (3.0 * (1.0 - 2.0 * nu));
    const double G = 0.5 * E / (1.0 + nu);
    T            s[9], eta[9], pr;
    const T      q  = trial(K, G, Hk, H, st, s, eta, &pr);
    const double qv = vpart(q), e0 = st[9], a = 3.0 * G + Hk;
    if (qv - a * 0.0 - (sy + Hi * (e0 + 0.0)) > TOL * sy) {
      double       df_dx;
      const double x     = solve(qv, a, sy, Hi, e0, (qv - (sy + Hi * e0)) / a, &df_dx);
      const T      delta = root_dual(x, q, df_dx);
      const T      c     = (2.0 * G) * delta;
      const T      iq    = 1.5 / q;
#pragma unroll
      for (int k = 0; k < 9; k++) {
        const T Np = eta[k] * iq;
        s[k]       = s[k] - c * Np;
        st[k] += x * vpart(Np);
      }
      st[9] += x;
    }
    s[0] = s[0] + pr;
    s[4] = s[4] + pr;
    s[8] = s[8] + pr;
    if (p[6] != 0.0) {
      stress_to_flux_large(s, H, flux);
    } else {
#pragma unroll
      for (int k = 0; k < 9; k++) flux[k] = s[k];
    }
  }

  // The consistent tangent.  With x the plastic increment, dx = dq / (3G + Hk + Hi) and dq = 1.5 eta : deta / q,
  //   dsigma = c1 sym(dH) + (K - c1/3) tr(dH) I - c2 eta (etas : dH),
  //   c1 = 2G (1 - 3G x / q),  c2 = 2G 3G (1 / (3G + Hk + Hi) - x / q) 1.5 / q^2,
  // etas the symmetric deviator of eta (x = c2 = 0 where the point stays elastic).  With large displacements
  // flux = sigma cof(F), and row c of sigma dcof(F) in direction (c', b) is, at parent slot a, component c' of
  // X_ab x sigma_c with X_ab = F (Ji_a x Ji_b) (no division by det F).  Slots are taken to the parent element as
  // in the Neo-Hookean tangent: W = cof Ji^T.
  template <class Emit>
  __device__ __forceinline__ static void tangent(const double* p, const double* H, const double* Ji, double dJ,
                                                 const double* st, Emit&& emit)
  {
    const double E = p[0], nu = p[1], sy = p[2], Hi = p[3], Hk = p[4];
    const double K = E / (3.0 * (1.0 - 2.0 * nu));
    const double G = 0.5 * E / (1.0 + nu);
    double       s[9], eta[9], pr;
    const double q = trial(K, G, Hk, H, st, s, eta, &pr), e0 = st[9], a3 = 3.0 * G + Hk;
    double       c1 = 2.0 * G, c2 = 0.0;
    if (q - a3 * 0.0 - (sy + Hi * (e0 + 0.0)) > TOL * sy) {
      double       df_dx;
      const double x  = solve(q, a3, sy, Hi, e0, (q - (sy + Hi * e0)) / a3, &df_dx);
      const double iq = 1.0 / q, xq = x * iq;
      c1 -= 6.0 * G * G * xq;
      c2 = 6.0 * G * G * (-1.0 / df_dx - xq) * (1.5 * iq * iq);
#pragma unroll
      for (int k = 0; k < 9; k++) s[k] -= (3.0 * G * xq) * eta[k];
    }
    s[0] += pr;
    s[4] += pr;
    s[8] += pr;
    double W[9], X[9];  // X: the pairs (a, b) = (1, 2), (2, 0), (0, 1)
#pragma unroll
    for (int k = 0; k < 9; k++) X[k] = 0.0;
    if (p[6] != 0.0) {
      double C[9];
      cof_i_plus(H, C);
      to_parent(C, Ji, W);
#pragma unroll
      for (int k = 0; k < 3; k++) {
        const double *u = Ji + ((k + 1) % 3) * 3, *v = Ji + ((k + 2) % 3) * 3;
        const double  y[3] = {dJ * (u[1] * v[2] - u[2] * v[1]), dJ * (u[2] * v[0] - u[0] * v[2]),
                              dJ * (u[0] * v[1] - u[1] * v[0])};
#pragma unroll
        for (int r = 0; r < 3; r++)
          X[k * 3 + r] = y[r] + (H[r * 3 + 0] * y[0] + H[r * 3 + 1] * y[1] + H[r * 3 + 2] * y[2]);
      }
    } else {
#pragma unroll
      for (int m = 0; m < 3; m++)
#pragma unroll
        for (int a = 0; a < 3; a++) W[m * 3 + a] = Ji[a * 3 + m];
    }
    double Q[9], Et[9], h[9];
    const double third = (eta[0] + eta[4] + eta[8]) / 3.0;
#pragma unroll
    for (int i = 0; i < 3; i++)
#pragma unroll
      for (int b = 0; b < 3; b++) {
        double vq = 0.0, ve = 0.0, vh = 0.0;
#pragma unroll
        for (int m = 0; m < 3; m++) {
          const double es = 0.5 * (eta[i * 3 + m] + eta[m * 3 + i]) - (i == m ? third : 0.0);
          vq += Ji[i * 3 + m] * W[m * 3 + b];
          ve += eta[i * 3 + m] * W[m * 3 + b];
          vh += es * Ji[b * 3 + m];
        }
        Q[i * 3 + b]  = (0.5 * c1 * dJ) * vq;
        Et[i * 3 + b] = (c2 * dJ) * ve;
        h[i * 3 + b]  = vh;
      }
    const double ch = 0.5 * c1 * dJ, ck = (K - c1 / 3.0) * dJ;
#pragma unroll
    for (int t = 0; t < 9; t++) {
      const int    c2i = t / 3, b = t % 3;
      const double kb  = ck * Ji[b * 3 + c2i];
#pragma unroll
      for (int r = 0; r < 9; r++) {
        const int c = r / 3, a = r % 3;
        double    v = (ch * Ji[b * 3 + c]) * W[c2i * 3 + a] + kb * W[r] - h[t] * Et[r];
        if (a != b) {
          const double* x = X + (3 - a - b) * 3;
          const int     i1 = (c2i + 1) % 3, i2 = (c2i + 2) % 3;
          const double  z = x[i1] * s[c * 3 + i2] - x[i2] * s[c * 3 + i1];
          v += (b - a + 3) % 3 == 1 ? z : -z;
        }
        if (c == c2i) v += Q[b * 3 + a];
        emit(r, t, v);
      }
    }
  }
};

}  // namespace sxk
