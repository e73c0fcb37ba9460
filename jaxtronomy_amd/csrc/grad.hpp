// Profiles written once for plain scalars and forward-mode duals (gm::Dual):
// the gradient kernels evaluate one profile with its own parameters as dual
// seeds, so every derivative is taken with respect to the reference's kwargs
// (theta_E, gamma, e1, e2, ...), through the same parameter conversions and
// floors as the forward path (floors and branches are decided on values, as
// jnp.maximum / jnp.where are under JAX differentiation).
#pragma once

#include "dual.hpp"
#include "profiles.hpp"

namespace lensim {
namespace gm {

template <typename T, int N>
__device__ __forceinline__ Dual<T, N> lift(T x, const Dual<T, N> &) {
  return Dual<T, N>(x);
}
template <typename T>
__device__ __forceinline__ T lift(T x, T) {
  return x;
}

// c + dc * (dt/dseeds): a series coefficient F_n(t) as a function of the seeds
template <typename T, int N>
__device__ __forceinline__ Dual<T, N> coef_of_t(T c, T dc, const Dual<T, N> &t) {
  Dual<T, N> r;
  r.v = c;
#pragma unroll
  for (int i = 0; i < N; ++i) r.d[i] = dc * t.d[i];
  return r;
}
template <typename T>
__device__ __forceinline__ T coef_of_t(T c, T, T) {
  return c;
}

template <typename S>
__device__ __forceinline__ bool is_nan(const S &x) {
  const auto v = val(x);
  return v != v;
}

// Sum_{n<N} c_n(t) w^n (quadratic-division form; see real_poly_at_complex)
template <typename T, typename S>
__device__ __forceinline__ void series_g(const T *__restrict__ c, const T *__restrict__ dc, int n, const S &t,
                                         const S &wr, const S &wi, S &pr, S &pi) {
  if (n == 1) {
    pr = coef_of_t(c[0], dc[0], t);
    pi = lift(T(0), t);
    return;
  }
  const S sw = T(2) * wr, tw = wr * wr + wi * wi;
  S b2 = lift(T(0), t), b1 = coef_of_t(c[n - 1], dc[n - 1], t);
  for (int k = n - 2; k >= 1; --k) {
    const S b0 = sw * b1 - tw * b2 + coef_of_t(c[k], dc[k], t);
    b2 = b1;
    b1 = b0;
  }
  pr = b1 * wr - tw * b2 + coef_of_t(c[0], dc[0], t);
  pi = b1 * wi;
}

// Clenshaw form of sum_{k<n} a(k) w^k for real coefficients a(k) at complex w
// (sw = 2 Re w, tw = |w|^2), as series_g's value.
template <typename T, typename A>
__device__ __forceinline__ void clenshaw_c(A a, int n, T wr, T wi, T sw, T tw, T &pr, T &pi) {
  if (n <= 0) {
    pr = pi = T(0);
    return;
  }
  if (n == 1) {
    pr = a(0);
    pi = T(0);
    return;
  }
  T b2 = T(0), b1 = a(n - 1);
  for (int k = n - 2; k >= 1; --k) {
    const T b0 = sw * b1 - tw * b2 + a(k);
    b2 = b1;
    b1 = b0;
  }
  pr = b1 * wr - tw * b2 + a(0);
  pi = b1 * wi;
}

// The series in duals without dual arithmetic inside the loop: the sum is
// holomorphic in w, so its tangents are S'(w) dw + U(w) dt with
// S'(w) = sum (k+1) c_{k+1} w^k and U(w) = sum dc_k w^k, three scalar
// recurrences instead of one recurrence on N + 1 components.
template <typename T, int N>
__device__ __forceinline__ void series_g(const T *__restrict__ c, const T *__restrict__ dc, int n,
                                         const Dual<T, N> &t, const Dual<T, N> &wr, const Dual<T, N> &wi,
                                         Dual<T, N> &pr, Dual<T, N> &pi) {
  const T wrv = wr.v, wiv = wi.v;
  const T sw = T(2) * wrv, tw = wrv * wrv + wiv * wiv;
  T sr, si, dr, di, ur, ui;
  clenshaw_c<T>([&](int k) { return c[k]; }, n, wrv, wiv, sw, tw, sr, si);
  clenshaw_c<T>([&](int k) { return T(k + 1) * c[k + 1]; }, n - 1, wrv, wiv, sw, tw, dr, di);
  clenshaw_c<T>([&](int k) { return dc[k]; }, n, wrv, wiv, sw, tw, ur, ui);
  pr.v = sr;
  pi.v = si;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    pr.d[i] = dr * wr.d[i] - di * wi.d[i] + ur * t.d[i];
    pi.d[i] = dr * wi.d[i] + di * wr.d[i] + ui * t.d[i];
  }
}

// EPL, LensModel/Profiles/epl.py:109-124, :178-200, :364-394.  p: theta_E,
// gamma, e1, e2, center_x, center_y.  nser: series length (from the value of f).
// q, cs, sn: the axis ratio and cos / sin of the orientation (from the record).
template <typename T, typename S>
__device__ __forceinline__ void epl_g_geo(const S *p, const S &q, const S &cs, const S &sn,
                                          const T *__restrict__ c, const T *__restrict__ dc, int nser, const S &x,
                                          const S &y, S &ax, S &ay) {
  const S t = p[1] - T(1);
  const S b = p[0] * sqrt(q);
  const S f = (T(1) - q) / (T(1) + q);
  const S dx = x - p[4], dy = y - p[5];
  const S xr = dx * cs + dy * sn;
  const S yr = dy * cs - dx * sn;
  const S Zr = q * xr, Zi = yr;
  const S R2 = Zr * Zr + Zi * Zi;
  if (val(R2) == T(0)) return;  // the reference's NaN at Z = 0 becomes 0 (epl.py:391-392)
  const S R = fmax(sqrt(R2), T(0.000000001));
  S Or, Oi;
  if (val(f) == T(0)) {
    Or = Zr;
    Oi = Zi;
  } else {
    const S zr = -f * (Zr * Zr - Zi * Zi) / R2;
    const S zi = -f * (T(2) * Zr * Zi) / R2;
    const S dr = zr - T(2);
    const S dd = T(1) / (dr * dr + zi * zi);
    const S wr = (zr * dr + zi * zi) * dd;
    const S wi = (zi * dr - zr * zi) * dd;
    S Sr, Si;
    series_g<T>(c, dc, nser, t, wr, wi, Sr, Si);
    const S er = T(1) - zr * T(0.5), ei = zi * T(-0.5);
    const S ed = T(1) / (er * er + ei * ei);
    const S hr = (Sr * er + Si * ei) * ed;
    const S hi = (Si * er - Sr * ei) * ed;
    Or = Zr * hr - Zi * hi;
    Oi = Zr * hi + Zi * hr;
  }
  const S scale = T(2) / (T(1) + q) * exp(t * log(b / R));
  S fr = scale * Or, fi = scale * Oi;
  if (is_nan(fr)) fr = lift(T(0), t);
  if (is_nan(fi)) fi = lift(T(0), t);
  ax = ax + (fr * cs - fi * sn);
  ay = ay + (fr * sn + fi * cs);
}

// NIE / SIE, LensModel/Profiles/nie.py:86-107, :182-200, :280-295, from the
// axis ratio q and the orientation's cos / sin (cs, sn).
template <typename T, typename S>
__device__ __forceinline__ void nie_g_geo(const S &theta_E, const S &q, const S &cs, const S &sn, const S &s_scale,
                                          const S &cx, const S &cy, const S &x, const S &y, S &ax, S &ay) {
  const S theta_E_conv = theta_E / sqrt((T(1) + q * q) / (T(2) * q));
  const S b = theta_E_conv * sqrt((T(1) + q * q) * T(0.5));
  const S s = s_scale / sqrt(q);
  const S dx = x - cx, dy = y - cy;
  const S xr = dx * cs + dy * sn;
  const S yr = dy * cs - dx * sn;
  const S qc = val(q) >= T(1) ? lift(T(0.99999999), q) : q;
  const S psi = sqrt(qc * qc * (s * s + xr * xr) + yr * yr);
  const S sq = sqrt(T(1) - qc * qc);
  const S fx = b / sq * atan(sq * xr / (psi + s));
  const S fy = b / sq * atanh(sq * yr / (psi + qc * qc * s));
  ax = ax + (fx * cs - fy * sn);
  ay = ay + (fx * sn + fy * cs);
}

// A linear deflector from its raw slot.
template <typename T, typename S>
__device__ __forceinline__ void defl_g(int type, const S *p, const S &x, const S &y, S &ax, S &ay) {
  if (type == LENSIM_SHEAR) {
    const S dx = x - p[2], dy = y - p[3];
    ax = ax + (p[0] * dx + p[1] * dy);
    ay = ay + (p[1] * dx - p[0] * dy);
  } else if (type == LENSIM_CONVERGENCE) {  // convergence.py:34-46; p: kappa, ra_0, dec_0
    ax = ax + p[0] * (x - p[1]);
    ay = ay + p[0] * (y - p[2]);
  }
}

// Sersic kernel, sersic_utils.py:239-267 (R_sersic already max(0, .) for the ellipse)
template <typename T, typename S>
__device__ __forceinline__ S sersic_g(const S &R, const S &R_sersic, const S &n) {
  const S R_ = fmax(R, T(0.0001));
  const S Rs_ = fmax(R_sersic, T(0.0001));
  const S bn = fmax(T(1.9992) * n - T(0.3271), T(0.00001));
  const S frac = R_ / Rs_;
  if (!(val(frac) <= T(1000))) return lift(T(0), R);
  return exp(-bn * (exp(log(frac) / n) - T(1)));
}

// SERSIC_ELLIPSE at (x, y) with its derivatives in closed form: returns the
// flux, writes d flux / d(amp, R_sersic, n_sersic, e1, e2, center_x,
// center_y) to gp and d flux / d(x, y) to gx, gy.  Same expression, floors
// and window as light_g (sersic_ellipse.py:62-93, param_util.py:103-124,
// sersic_utils.py:239-267); a floor that binds passes no derivative, as
// fmax does for duals.  With u = frac^(1/n) and E = exp(-b_n (u - 1)):
//   d flux / d ln(frac) = -amp E b_n u / n,
//   d flux / dn = -(d flux / d ln frac) ln(frac) / n - amp E (u - 1) db_n/dn.
template <typename T>
__device__ __forceinline__ T sersic_ellipse_grad(const double *p, T x, T y, T *gp, T &gx, T &gy) {
  const T amp = T(p[0]), p1 = T(p[1]), n = T(p[2]), e1 = T(p[3]), e2 = T(p[4]);
  const T dx = x - T(p[5]), dy = y - T(p[6]);
  const T Rs = p1 >= T(0) ? p1 : T(0);
  const T v = T(1) - e1 * e1 - e2 * e2;
  const T sq = sqrt(v >= T(0) ? v : -v);
  const bool nfree = sq >= T(0.000001);
  const T norm = nfree ? sq : T(0.000001);
  const T inorm = T(1) / norm;
  const T xe = ((T(1) - e1) * dx - e2 * dy) * inorm;
  const T ye = ((T(1) + e1) * dy - e2 * dx) * inorm;
  const T R = sqrt(xe * xe + ye * ye);
  const bool rfree = R >= T(0.0001), sfree = Rs >= T(0.0001);
  const T R_ = rfree ? R : T(0.0001);
  const T Rs_ = sfree ? Rs : T(0.0001);
  const T bn0 = T(1.9992) * n - T(0.3271);
  const bool bfree = bn0 >= T(0.00001);
  const T bn = bfree ? bn0 : T(0.00001);
  const T frac = R_ / Rs_;
#pragma unroll
  for (int i = 0; i < 7; ++i) gp[i] = T(0);
  gx = gy = T(0);
  if (!(frac <= T(1000))) return T(0);
  const T lf = log(frac);
  const T u = exp(lf / n);
  const T E = exp(-bn * (u - T(1)));
  const T c = -amp * E * bn * u / n;  // d flux / d ln(frac)
  gp[0] = E;
  gp[1] = (sfree && p1 >= T(0)) ? -c / Rs_ : T(0);
  gp[2] = -c * lf / n - (bfree ? amp * E * (u - T(1)) * T(1.9992) : T(0));
  // d flux / d(xe, ye) through R = |(xe, ye)|
  const T gR = rfree ? c / (R_ * R) : T(0);
  const T gxe = gR * xe, gye = gR * ye;
  // d norm / d e_i = -sign(v) e_i / sq where the floor does not bind
  const T sg = v >= T(0) ? T(1) : T(-1);
  const T dn1 = nfree ? -sg * e1 / sq : T(0), dn2 = nfree ? -sg * e2 / sq : T(0);
  gp[3] = (gxe * (-dx - xe * dn1) + gye * (dy - ye * dn1)) * inorm;
  gp[4] = (gxe * (-dy - xe * dn2) + gye * (-dx - ye * dn2)) * inorm;
  gx = (gxe * (T(1) - e1) - gye * e2) * inorm;
  gy = (gye * (T(1) + e1) - gxe * e2) * inorm;
  gp[5] = -gx;
  gp[6] = -gy;
  return amp * E;
}

// ---- FP64 closed forms ----
// The float gradient kernels differentiate with duals; in double those took
// 3000 vector instructions a ray for the EPL (every dual division, root and
// logarithm on library functions).  The FP64 kernels use the derivatives
// written out below, on the records' constants, the library's own log2, exp2,
// atan and atanh and third-order reciprocals.

// The EPL's alpha at (x, y) and its derivatives by (theta_E, gamma, e1, e2,
// center_x, center_y).  With Z = q x + i y (major-axis frame), R = |Z|, z = -f
// Z / conj(Z), F = 2F1(1, t/2; 2 - t/2; z) and s = 2/(1+q) (b/R)^t, alpha = s Z F.
//  * F = 1 + delta, delta = (w P(w) + z/2) / (1 - z/2), w = z/(z - 2), P = sum_n>=1
//    F_n w^(n-1) (the Lopez-Temme series of epl_major_f64).  With its first
//    parameter 1, F obeys the first-order equation
//      z F' = [b z + (b z + 1 - c) delta] / (1 - z),  b = t/2, c = 2 - t/2,
//    so no second series is needed for dF/dz;
//  * d/dt: ln(b/R) alpha + s Z dF/dt, dF/dt = (sum dF_n/dt w^n) / (1 - z/2);
//  * d/dq at fixed frame: dZ = x dq, dz/z = df/f - 2 i x y dq / R^2, ds/s =
//    (-1/(1+q) + t (1/(2q) - q x^2/R^2)) dq;
//  * theta_E, the centre and the orientation as in epl_dalpha's comment, the
//    Hessian with 1/r^2 alone.
// epl_basis_f64 gives alpha, d/dt and d/dq of it, its derivative by the angle
// and by the centre (x and y components in ax[], ay[]); the kwargs' derivatives
// are linear in these with factors of the kwargs alone (EllKw, epl_kw): sums
// over rays are taken of the basis.
struct EllKw {
  double dp1, dp2, dq1, dq2;  // d phi and d q by e1 and e2
  double q0;                  // the unclamped q
  EllKw() = default;
  __device__ __forceinline__ EllKw(double e1, double e2) {
    const double c2 = e1 * e1 + e2 * e2, ce = ::sqrt(c2);
    const double cc = ce < 0.9999 ? ce : 0.9999, h = 0.5 / c2;
    q0 = (1.0 - cc) / (1.0 + cc);
    dp1 = -e2 * h;
    dp2 = e1 * h;
    const double dqdc = ce < 0.9999 ? -2.0 / ((1.0 + ce) * (1.0 + ce)) : 0.0;
    dq1 = dqdc * e1 / ce;
    dq2 = dqdc * e2 / ce;
  }
};
__device__ __forceinline__ void epl_kw(const EllKw &ek, const double *rd, const double *pk, double *v) {
  const double q = v[2], ph = v[3];
  v[0] *= pk[0] != 0.0 ? rd[EPL_T] / pk[0] : 0.0;
  v[2] = q * ek.dq1 + ph * ek.dp1;
  v[3] = q * ek.dq2 + ph * ek.dp2;
}
__device__ __forceinline__ void epl_basis_f64(const double *rd, const double *__restrict__ c,
                                              const double *__restrict__ dc, double x, double y, double *ax,
                                              double *ay) {
  const double q = rd[EPL_Q], t = rd[EPL_T], f = rd[EPL_F], cs = rd[EPL_C], sn = rd[EPL_S];
  const double dx = x - rd[R_CX], dy = y - rd[R_CY];
  const double xr = dx * cs + dy * sn, yr = dy * cs - dx * sn;
  const double Zr = q * xr, Zi = yr;
  const double R2 = Zr * Zr + Zi * Zi;
#pragma unroll
  for (int i = 0; i < 6; ++i) ax[i] = ay[i] = 0.0;
  if (R2 == 0.0) return;  // the reference's NaN at Z = 0 becomes 0 (epl.py:391-392)
  const bool rfree = R2 >= 1e-18;  // the floor R >= 1e-9 passes no derivative
  const double R2c = rfree ? R2 : 1e-18;
  const double iR2 = rcp_full(R2);
  double Fr = 1.0, Fi = 0.0, tr = 0.0, ti = 0.0, gr = 0.0, gi = 0.0;  // F, dF/dt, z F' (dz/dq)/z
  if (f != 0.0) {
    const double zr = -f * (Zr * Zr - Zi * Zi) * iR2, zi = -2.0 * f * (Zr * Zi) * iR2;
    const double er = fma(-0.5, zr, 1.0), ei = -0.5 * zi;
    const double ed = rcp_full(fma(er, er, ei * ei));
    const double vr = er * ed, vi = -ei * ed;  // 1 / (1 - z/2)
    const double wr = -0.5 * (zr * vr - zi * vi), wi = -0.5 * (zr * vi + zi * vr);
    const int n = (int)rd[EPL_NMAX];
    double Pr, Pi, Ur, Ui;
    real_poly_at_complex<double>(c + 1, n - 1, wr, wi, Pr, Pi);
    real_poly_at_complex<double>(dc + 1, n - 1, wr, wi, Ur, Ui);
    const double nr = fma(wr, Pr, fma(-wi, Pi, 0.5 * zr)), ni = fma(wr, Pi, fma(wi, Pr, 0.5 * zi));
    const double er2 = nr * vr - ni * vi, ei2 = nr * vi + ni * vr;  // delta
    Fr = 1.0 + er2;
    Fi = ei2;
    const double ur = wr * Ur - wi * Ui, ui = wr * Ui + wi * Ur;
    tr = ur * vr - ui * vi;
    ti = ur * vi + ui * vr;
    // z F'
    const double b = 0.5 * t, mr = fma(b, zr, b - 1.0), mi = b * zi;
    const double kr = fma(b, zr, mr * er2 - mi * ei2), ki = fma(b, zi, mr * ei2 + mi * er2);
    const double or_ = 1.0 - zr, od = rcp_full(fma(or_, or_, zi * zi));
    const double hr = (kr * or_ - ki * zi) * od, hi = (kr * zi + ki * or_) * od;
    // times (dz/dq) / z
    const double qr = -2.0 / ((1.0 + q) * (1.0 + q) * f), qi = -2.0 * xr * yr * iR2;
    gr = hr * qr - hi * qi;
    gi = hr * qi + hi * qr;
  }
  const double lb2 = rd[EPL_LB2] - 0.5 * log2_pos(R2c);  // log2(b / R)
  const double pw = exp2_fin(t * lb2), s = rd[EPL_PREF] * pw;
  const double sZr = s * Zr, sZi = s * Zi;
  const double fr = sZr * Fr - sZi * Fi, fi = sZr * Fi + sZi * Fr;
  const double lnbr = pw > 0.0 ? 0.6931471805599453 * lb2 : 0.0;
  const double atr = fma(lnbr, fr, sZr * tr - sZi * ti), ati = fma(lnbr, fi, sZr * ti + sZi * tr);
  const double ls = -1.0 / (1.0 + q) + t * (0.5 / q - (rfree ? q * xr * xr * iR2 : 0.0));
  const double sx = s * xr;
  const double aqr = fma(ls, fr, fma(sx, Fr, sZr * gr - sZi * gi)), aqi = fma(ls, fi, fma(sx, Fi, sZr * gi + sZi * gr));
  ax[0] = fr * cs - fi * sn;
  ay[0] = fr * sn + fi * cs;
  ax[1] = atr * cs - ati * sn;
  ay[1] = atr * sn + ati * cs;
  ax[2] = aqr * cs - aqi * sn;
  ay[2] = aqr * sn + aqi * cs;
  // Hessian: kappa and the shear of EPLMajorAxis.hessian, rotated back
  const double x2 = xr * xr, y2 = yr * yr, ir2 = rcp_full(x2 + y2);
  const double kappa = 0.5 * (2.0 - t) * pw;
  const double g1 = ((1.0 - t) * (fr * xr - fi * yr) - kappa * (x2 - y2)) * ir2;
  const double g2 = ((1.0 - t) * (fi * xr + fr * yr) - kappa * (2.0 * xr * yr)) * ir2;
  const double c2p = cs * cs - sn * sn, s2p = 2.0 * sn * cs;
  const double G1 = c2p * g1 - s2p * g2, fxy = s2p * g1 + c2p * g2;
  const double fxx = kappa + G1, fyy = kappa - G1;
  ax[3] = fxx * dy - fxy * dx - ay[0];
  ay[3] = fxy * dy - fyy * dx + ax[0];
  ax[4] = -fxx;
  ax[5] = ay[4] = -fxy;
  ay[5] = -fyy;
}
__device__ __forceinline__ void epl_dalpha_f64(const double *rd, const double *__restrict__ c,
                                               const double *__restrict__ dc, const double *pk, double x, double y,
                                               double &a_x, double &a_y, double *dax, double *day) {
  epl_basis_f64(rd, c, dc, x, y, dax, day);
  a_x = dax[0];
  a_y = day[0];
  const EllKw ek(pk[2], pk[3]);
  epl_kw(ek, rd, pk, dax);
  epl_kw(ek, rd, pk, day);
}

// The SIE / NIE's alpha at (x, y) and its derivatives by (theta_E, e1, e2[,
// s_scale], center_x, center_y).  In the major-axis frame alpha = k (A, B), k = b
// / sq, sq = sqrt(1 - q^2), A = arctan(sq x / D1), B = arctanh(sq y / D2), D1 =
// psi + s, D2 = psi + q^2 s, psi^2 = q^2 (s^2 + x^2) + y^2, with b = theta_E
// sqrt(q) and s = s_scale / sqrt(q) (nie.py:182-200, :280-295).
// nie_basis_f64: alpha, d/dq, the derivative by the angle, for a NIE by s, and
// by the centre; nie_kw as epl_kw.
template <int TYPE>
__device__ __forceinline__ void nie_kw(const EllKw &ek, const double *pk, double *v) {
  const double q = v[1], ph = v[2];
  v[0] *= pk[0] != 0.0 ? 1.0 / pk[0] : 0.0;
  v[1] = q * ek.dq1 + ph * ek.dp1;
  v[2] = q * ek.dq2 + ph * ek.dp2;
  if constexpr (TYPE == LENSIM_NIE) v[3] *= rsq_full(ek.q0);  // s = s_scale / sqrt(q)
}
template <int TYPE>
__device__ __forceinline__ void nie_basis_f64(const double *rd, double q0, double x, double y, double *ax,
                                              double *ay) {
  constexpr bool kNie = TYPE == LENSIM_NIE;
  constexpr int kc = kNie ? 4 : 3;  // the centre's slots
  const double q = rd[NIE_Q], q2 = rd[NIE_Q2], s = rd[NIE_SS], sq = rd[NIE_SQ], k = rd[NIE_BSQ], cs = rd[NIE_C],
               sn = rd[NIE_S];
  const bool qfree = q0 < 1.0;  // else the frame's q is a constant
  const double dx = x - rd[R_CX], dy = y - rd[R_CY];
  const double xr = dx * cs + dy * sn, yr = dy * cs - dx * sn;
  const double p2 = fma(q2, fma(s, s, xr * xr), yr * yr);
  const double ip = p2 > 0.0 ? rsq_full(p2) : 0.0, psi = p2 * ip;
  const double D1 = psi + s, D2 = fma(q2, s, psi);
  const double i1 = rcp_full(D1), i2 = rcp_full(D2);
  const double u1 = sq * xr * i1, u2 = sq * yr * i2;
  const double A = atan_dbl(u1), B = atanh_dbl(u2);
  const double fx = k * A, fy = k * B;
  ax[0] = fx * cs - fy * sn;
  ay[0] = fx * sn + fy * cs;
  // k dA = k1 d(x / D1 sq) and k dB = k2 d(y / D2 sq)
  const double k1 = k * rcp_full(fma(u1, u1, 1.0)), k2 = k * rcp_full(fma(-u2, u2, 1.0));
  const double px = q2 * xr * ip, py = yr * ip, ps = q2 * s * ip, pq = q * fma(s, s, xr * xr) * ip;
  const double w1 = k1 * sq * i1, w2 = k2 * sq * i2;
  const double axx = w1 * (1.0 - xr * px * i1), axy = -w1 * xr * py * i1;
  const double ayx = -w2 * yr * px * i2, ayy = w2 * (1.0 - yr * py * i2);
  const double axs = -w1 * xr * (ps + 1.0) * i1, ays = -w2 * yr * (ps + q2) * i2;
  // q: through k, sq and psi (the frame's q), and through b and s = s_scale / sqrt(q)
  const double isq2 = rcp_full(sq * sq), iq0 = 0.5 * rcp_full(q0);
  double qxr = iq0 * fma(-s, axs, fx), qyr = iq0 * fma(-s, ays, fy);
  if (qfree) {
    qxr += q * isq2 * (fx - w1 * xr) - w1 * xr * pq * i1;
    qyr += q * isq2 * (fy - w2 * yr) - w2 * yr * fma(2.0 * q, s, pq) * i2;
  }
  // H = R (d alpha / d(xr, yr)) R^T
  const double mxx = axx * cs - ayx * sn, mxy = axy * cs - ayy * sn, myx = axx * sn + ayx * cs,
               myy = axy * sn + ayy * cs;
  const double hxx = mxx * cs - mxy * sn, hxy = mxx * sn + mxy * cs, hyx = myx * cs - myy * sn,
               hyy = myx * sn + myy * cs;
  ax[1] = qxr * cs - qyr * sn;
  ay[1] = qxr * sn + qyr * cs;
  ax[2] = hxx * dy - hxy * dx - ay[0];
  ay[2] = hyx * dy - hyy * dx + ax[0];
  if constexpr (kNie) {
    ax[3] = axs * cs - ays * sn;
    ay[3] = axs * sn + ays * cs;
  }
  ax[kc] = -hxx;
  ay[kc] = -hyx;
  ax[kc + 1] = -hxy;
  ay[kc + 1] = -hyy;
}
template <int TYPE>
__device__ __forceinline__ void nie_dalpha_f64(const double *rd, const double *pk, double x, double y, double &a_x,
                                               double &a_y, double *dax, double *day) {
  const EllKw ek(pk[1], pk[2]);
  nie_basis_f64<TYPE>(rd, ek.q0, x, y, dax, day);
  a_x = dax[0];
  a_y = day[0];
  nie_kw<TYPE>(ek, pk, dax);
  nie_kw<TYPE>(ek, pk, day);
}

// The NFW's alpha = a (dx, dy) at (x, y), a = 4 rho0 Rs g / u, u = X^2, and its
// derivatives by (Rs, alpha_Rs, center_x, center_y): X dg/dX = 1 + X F' = u (1 -
// F) / (u - 1), so X da/dX = 4 rho0 Rs X dg/dX / u - 2 a, Rs da/dRs = -(a + X
// da/dX), and the Jacobian a I + (X da/dX / R^2) d d^T.  Floors as nfw.py:86-105
// (R >= 1e-8, X >= 1e-6 in g, Rs >= 1e-7), which pass no derivative.
__device__ __forceinline__ void nfw_dalpha_f64(const double *rd, const double *pk, double x, double y, double &a_x,
                                               double &a_y, double *dax, double *day) {
  const double dx = x - rd[R_CX], dy = y - rd[R_CY], irs = rd[NFW_IRS];
  const double R2 = fma(dx, dx, dy * dy);
  const bool rfree = R2 >= 1e-16;
  const double u = (rfree ? R2 : 1e-16) * irs * irs;
  const bool xfree = u >= 1e-12;
  const double uc = xfree ? u : 1e-12, rX = rsq_full(uc), iu = xfree ? rX * rX : 1.0 / u;
  const double F = halo_F(uc, rX);
  const double l = fma(0.34657359027997264, log2_pos(uc), -0.6931471805599453);  // ln(X / 2)
  double g = l + F;
  if (uc < 0.0025) {
    // the sum cancels to u: with F = arccosh(1 / X) / sqrt(1 - u) by its series,
    // g = -u (l P(u) + Q(u)) to 2e-16 here
    constexpr double kP[6] = {0.5, 0.375, 0.3125, 0.2734375, 0.24609375, 0.2255859375};
    constexpr double kQ[6] = {0.25, 0.21875, 0.19270833333333334, 0.17350260416666666, 0.15888671875,
                              0.14735514322916668};
    g = -uc * fma(l, poly(kP, uc), poly(kQ, uc));
  }
  const double e = uc - 1.0;
  const double xg = fabs(e) < 0.03 ? 1.0 + halo_XdF(uc, F) : uc * (1.0 - F) * rcp_full(e);
  const double A = rd[NFW_A], a = A * g * iu;
  const double aX = rfree ? fma(A * iu, xfree ? xg : 0.0, -2.0 * a) : 0.0;
  const double rs0 = pk[0];
  const double aR = rs0 >= 0.0000001 ? -(a + aX) * irs : -2.0 * a / rs0;
  const double aA = rd[NFW_RS] / (rs0 * rs0 * (1.0 + ::log(0.5))) * g * iu;
  const double q = aX * rcp_full(rfree ? R2 : 1.0);
  a_x = a * dx;
  a_y = a * dy;
  dax[0] = aR * dx;
  day[0] = aR * dy;
  dax[1] = aA * dx;
  day[1] = aA * dy;
  dax[2] = -fma(q * dx, dx, a);
  day[2] = dax[3] = -(q * dx) * dy;
  day[3] = -fma(q * dy, dy, a);
}

// sersic_ellipse_grad in double from the profile's record rd and kwargs p.
__device__ __forceinline__ double sersic_ellipse_grad_f64(const double *rd, const double *p, double x, double y,
                                                          double *gp, double &gx, double &gy) {
  const double amp = rd[SE_AMP], p1 = p[1], e1 = p[3], e2 = p[4], invn = rd[SE_INVN];
  const double dx = x - rd[R_CX], dy = y - rd[R_CY];
  const double v = 1.0 - e1 * e1 - e2 * e2, sq = ::sqrt(fabs(v));
  const bool nfree = sq >= 0.000001, sfree = p1 >= 0.0001, bfree = 1.9992 * p[2] - 0.3271 >= 0.00001;
  const double inorm = 1.0 / (nfree ? sq : 0.000001);
  const double sg = v >= 0.0 ? 1.0 : -1.0;
  const double dn1 = nfree ? -sg * e1 * inorm : 0.0, dn2 = nfree ? -sg * e2 * inorm : 0.0;
  const double xe = rd[SE_M00] * dx + rd[SE_M01] * dy, ye = rd[SE_M01] * dx + rd[SE_M11] * dy;
  const double R2 = fma(xe, xe, ye * ye);
  const bool rfree = R2 >= 1e-8;
  const double R2c = rfree ? R2 : 1e-8;
#pragma unroll
  for (int i = 0; i < 7; ++i) gp[i] = 0.0;
  gx = gy = 0.0;
  if (!(R2c <= rd[SE_R2MAX])) return 0.0;
  const double l2 = (0.5 * log2_pos(R2c) - rd[SE_LNRS] * 1.4426950408889634) * invn;  // log2(frac) / n
  const double u = exp2_fin(l2);
  const double E = exp2_fin(rd[SE_K2] * (1.0 - u)), aE = amp * E;
  const double c = -aE * rd[SE_BN] * u * invn;  // d flux / d ln(frac)
  gp[0] = E;
  gp[1] = sfree ? -c * rd[SE_IRS] : 0.0;
  gp[2] = -c * (0.6931471805599453 * l2) - (bfree ? aE * (u - 1.0) * 1.9992 : 0.0);
  const double k = rfree ? c * rcp_full(R2c) : 0.0;
  const double gxe = k * xe, gye = k * ye;
  gp[3] = (gxe * (-dx - xe * dn1) + gye * (dy - ye * dn1)) * inorm;
  gp[4] = (gxe * (-dy - xe * dn2) + gye * (-dx - ye * dn2)) * inorm;
  gx = gxe * rd[SE_M00] + gye * rd[SE_M01];
  gy = gye * rd[SE_M11] + gxe * rd[SE_M01];
  gp[5] = -gx;
  gp[6] = -gy;
  return aE;
}
// Sums over rays of w times sersic_ellipse_grad_f64's derivatives, from a
// profile's constants read once: with k = (d flux / d ln R) / R^2 the
// derivatives by e1, e2 and the centre are linear in the moments of k about the
// centre, and those by R_sersic and n in three sums, so a ray adds nine numbers
// and the kwargs' factors are applied to the sums (kwargs()).
struct SersicGrad {
  double cx, cy, m00, m01, m11, a, b, c, amp, lnrs, invn, k2, bnin, r2max;
  double se = 0.0, sc = 0.0, sl = 0.0, su = 0.0, kx = 0.0, ky = 0.0, kxx = 0.0, kxy = 0.0, kyy = 0.0;
  __device__ __forceinline__ explicit SersicGrad(const double *rd)
      : cx(wave_uniform(rd[R_CX])), cy(wave_uniform(rd[R_CY])), m00(wave_uniform(rd[SE_M00])),
        m01(wave_uniform(rd[SE_M01])), m11(wave_uniform(rd[SE_M11])), amp(wave_uniform(rd[SE_AMP])),
        lnrs(wave_uniform(rd[SE_LNRS] * 1.4426950408889634)), invn(wave_uniform(rd[SE_INVN])),
        k2(wave_uniform(rd[SE_K2])), bnin(wave_uniform(rd[SE_BN] * rd[SE_INVN])), r2max(wave_uniform(rd[SE_R2MAX])) {
    a = wave_uniform(m00 * m00 + m01 * m01);
    b = wave_uniform(m01 * (m00 + m11));
    c = wave_uniform(m01 * m01 + m11 * m11);
  }
  // the ray at (x, y) with weight w; (gx, gy): d flux / d(x, y)
  __device__ __forceinline__ void add(double x, double y, double w, double &gx, double &gy) {
    const double dx = x - cx, dy = y - cy;
    const double xe = m00 * dx + m01 * dy, ye = m01 * dx + m11 * dy;
    const double R2 = fma(xe, xe, ye * ye);
    const bool rfree = R2 >= 1e-8;
    const double R2c = rfree ? R2 : 1e-8;
    gx = gy = 0.0;
    if (!(R2c <= r2max)) return;
    const double l2 = fma(0.5, log2_pos(R2c), -lnrs) * invn;  // log2(frac) / n
    const double u = exp2_fin(l2);
    const double E = exp2_fin(k2 * (1.0 - u)), aE = amp * E;
    const double d = -aE * bnin * u, wd = w * d;  // d flux / d ln(frac)
    se = fma(w, E, se);
    sc += wd;
    sl = fma(wd, l2, sl);
    su = fma(w * aE, u - 1.0, su);
    const double k = rfree ? d * rcp_full(R2c) : 0.0, wx = w * k * dx, wy = w * k * dy;
    gx = k * fma(a, dx, b * dy);
    gy = k * fma(b, dx, c * dy);
    kx += wx;
    ky += wy;
    kxx = fma(wx, dx, kxx);
    kxy = fma(wx, dy, kxy);
    kyy = fma(wy, dy, kyy);
  }
  __device__ __forceinline__ void kwargs(const double *rd, const double *p, double *acc) const {
    const double e1 = p[3], e2 = p[4], v = 1.0 - e1 * e1 - e2 * e2, sq = ::sqrt(fabs(v));
    const bool nfree = sq >= 0.000001, sfree = p[1] >= 0.0001, bfree = 1.9992 * p[2] - 0.3271 >= 0.00001;
    const double inorm = 1.0 / (nfree ? sq : 0.000001), sg = v >= 0.0 ? 1.0 : -1.0;
    const double dn1 = nfree ? -sg * e1 * inorm : 0.0, dn2 = nfree ? -sg * e2 * inorm : 0.0;
    const double sr = a * kxx + 2.0 * b * kxy + c * kyy;  // sum of k R^2
    acc[0] = se;
    acc[1] = sfree ? -sc * rd[SE_IRS] : 0.0;
    acc[2] = -0.6931471805599453 * sl - (bfree ? 1.9992 * su : 0.0);
    acc[3] = (m11 * kyy - m00 * kxx - dn1 * sr) * inorm;
    acc[4] = (-(m00 * kxy + m01 * kyy) - (m01 * kxx + m11 * kxy) - dn2 * sr) * inorm;
    acc[5] = -(a * kx + b * ky);
    acc[6] = -(b * kx + c * ky);
    acc[7] = 0.0;
  }
};

template <typename T>
__device__ __forceinline__ T sersic_ellipse_grad_rec(const double *rd, const double *p, T x, T y, T *gp, T &gx, T &gy) {
  if constexpr (sizeof(T) == sizeof(double)) return sersic_ellipse_grad_f64(rd, p, x, y, gp, gx, gy);
  else return sersic_ellipse_grad<T>(p, x, y, gp, gx, gy);
}

// One light profile from its raw slot at (x, y).
template <typename T, typename S>
__device__ __forceinline__ S light_g(int type, const S *p, const S &x, const S &y) {
  switch (type) {
    case LENSIM_SERSIC_ELLIPSE: {
      // sersic_ellipse.py:62-93 with param_util.py:103-124 (product average)
      const S Rs = fmax(p[1], T(0));
      const S dx = x - p[5], dy = y - p[6];
      const S norm = fmax(sqrt(fabs(T(1) - p[3] * p[3] - p[4] * p[4])), T(0.000001));
      const S xe = ((T(1) - p[3]) * dx - p[4] * dy) / norm;
      const S ye = ((T(1) + p[3]) * dy - p[4] * dx) / norm;
      return p[0] * sersic_g<T>(sqrt(xe * xe + ye * ye), Rs, p[2]);
    }
    case LENSIM_SERSIC: {
      const S dx = x - p[3], dy = y - p[4];
      return p[0] * sersic_g<T>(sqrt(dx * dx + dy * dy), p[1], p[2]);
    }
    case LENSIM_GAUSSIAN: {
      // gaussian.py:27-42
      const S s2 = p[1] * p[1];
      const S dx = x - p[2], dy = y - p[3];
      return p[0] / (T(2 * M_PI) * s2) * exp(-(dx * dx / s2 + dy * dy / s2) * T(0.5));
    }
    default:
      return lift(T(0), x);
  }
}

}  // namespace gm
}  // namespace lensim
