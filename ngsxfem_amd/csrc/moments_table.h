// moments_table.h -- GENERATED by gen_moments.py; do not edit.
// Moment form of the H1 mass and stiffness element matrices (see gen_moments.py).
#pragma once
#ifndef XG_DEV  // host builds (tests) define XG_DEV themselves
#include "xg_device.hpp"
#endif
#include <math.h>
namespace xg {
template <int D, int P>
struct Moments;
#pragma clang fp contract(fast)
template <>
struct Moments<1, 1> {
  static constexpr int NM = 3;  // degree-2 moments
  static constexpr int NK = 1;  // degree-0 moments
  static constexpr int NQ = 2;  // degree-1 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    {
      const double wb = w * l[0];
      m[0] = fma(wb, l[0], m[0]);
      m[1] = fma(wb, l[1], m[1]);
    }
    {
      const double wb = w * l[1];
      m[2] = fma(wb, l[1], m[2]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.3333333333333333 - m[0];
    m[1] = 0.16666666666666666 - m[1];
    m[2] = 0.3333333333333333 - m[2];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + m[2];
  }
  static constexpr int NH = 2;  // h: coefficients of H_1 .. H_1
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/2))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    m[0] = fma(l[0], h[0], m[0]);
    m[1] = fma(l[1], h[0], fma(l[0], h[1], m[1]));
    m[2] = fma(l[1], h[1], m[2]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 2.0;
    m[2] *= 2.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 3;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0];
      const double K_ = Gs[0] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1];
      const double K_ = Gs[1] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[2] = v_;
    }
    {
      const double M_ = m[2];
      const double K_ = Gs[2] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[3] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1]));
    out[1] = (T)(s * (m[1] + m[2]));
  }
};  // 6 coefficient terms
template <>
struct Moments<1, 2> {
  static constexpr int NM = 5;  // degree-4 moments
  static constexpr int NK = 3;  // degree-2 moments
  static constexpr int NQ = 3;  // degree-2 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[1] * l[1];
    {
      const double wb = w * t0;
      m[0] = fma(wb, t0, m[0]);
      m[1] = fma(wb, t1, m[1]);
      m[2] = fma(wb, t2, m[2]);
    }
    {
      const double wb = w * t1;
      m[3] = fma(wb, t2, m[3]);
    }
    {
      const double wb = w * t2;
      m[4] = fma(wb, t2, m[4]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.2 - m[0];
    m[1] = 0.05 - m[1];
    m[2] = 0.03333333333333333 - m[2];
    m[3] = 0.05 - m[3];
    m[4] = 0.2 - m[4];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + m[2];
    mk[1] = m[1] + 2.0 * m[2] + m[3];
    mk[2] = m[2] + 2.0 * m[3] + m[4];
  }
  static constexpr int NH = 9;  // h: coefficients of H_1 .. H_3
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/4))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    h[2] = fma(l[0], h[0], h[2]);
    h[3] = fma(l[1], h[0], fma(l[0], h[1], h[3]));
    h[4] = fma(l[1], h[1], h[4]);
    h[5] = fma(l[0], h[2], h[5]);
    h[6] = fma(l[1], h[2], fma(l[0], h[3], h[6]));
    h[7] = fma(l[1], h[3], fma(l[0], h[4], h[7]));
    h[8] = fma(l[1], h[4], h[8]);
    m[0] = fma(l[0], h[5], m[0]);
    m[1] = fma(l[1], h[5], fma(l[0], h[6], m[1]));
    m[2] = fma(l[1], h[6], fma(l[0], h[7], m[2]));
    m[3] = fma(l[1], h[7], fma(l[0], h[8], m[3]));
    m[4] = fma(l[1], h[8], m[4]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 24.0;
    m[1] *= 6.0;
    m[2] *= 4.0;
    m[3] *= 6.0;
    m[4] *= 24.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 3;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    const double sm2_ = 2.0 * sm;
    const double sm4_ = 4.0 * sm;
    const double sk4_ = 4.0 * sk;
    const double Gd1 = 2.0 * Gs[1];
    // A = sm M^B + sk K^B (Bernstein basis, upper triangle)
    const double A0_0 = sm * m[0] + sk4_ * (Gs[0] * mk[0]);
    const double A0_1 = sm2_ * m[1] + sk4_ * (Gs[0] * mk[1] + Gs[1] * mk[0]);
    const double A0_2 = sm * m[2] + sk4_ * (Gs[1] * mk[1]);
    const double A1_1 = sm4_ * m[2] + sk4_ * (Gs[0] * mk[2] + Gd1 * mk[1] + Gs[2] * mk[0]);
    const double A1_2 = sm2_ * m[3] + sk4_ * (Gs[1] * mk[2] + Gs[2] * mk[1]);
    const double A2_2 = sm * m[4] + sk4_ * (Gs[2] * mk[2]);
    // L = T A T^T: a column b of X = A T^T where T's row b has several
    // entries, otherwise the entries of A directly
    {
      const double X0 = A0_0 - 0.5 * A0_1;
      const double X1 = A0_1 - 0.5 * A1_1;
      const double X2 = A0_2 - 0.5 * A1_2;
      const T v0_ = (T)(X0 - 0.5 * X1);
      out[0] = v0_;
    }
    {
      const double X0 = -0.5 * A0_1 + A0_2;
      const double X1 = -0.5 * A1_1 + A1_2;
      const double X2 = -0.5 * A1_2 + A2_2;
      const T v0_ = (T)(X0 - 0.5 * X1);
      out[1] = v0_;
      out[3] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X2);
      out[4] = v1_;
    }
    {
      const T v0_ = (T)(2.0 * A0_1 - A1_1);
      out[2] = v0_;
      out[6] = v0_;
      const T v1_ = (T)(-A1_1 + 2.0 * A1_2);
      out[5] = v1_;
      out[7] = v1_;
      const T v2_ = (T)(4.0 * A1_1);
      out[8] = v2_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1] - m[2] - m[3]));
    out[1] = (T)(s * (-m[1] - m[2] + m[3] + m[4]));
    out[2] = (T)(s * (4.0 * m[1] + 8.0 * m[2] + 4.0 * m[3]));
  }
};  // 39 coefficient terms
template <>
struct Moments<1, 3> {
  static constexpr int NM = 7;  // degree-6 moments
  static constexpr int NK = 5;  // degree-4 moments
  static constexpr int NQ = 4;  // degree-3 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[1] * l[1];
    const double t3 = t0 * l[0];
    const double t4 = t1 * l[0];
    const double t5 = t2 * l[0];
    const double t6 = t2 * l[1];
    {
      const double wb = w * t3;
      m[0] = fma(wb, t3, m[0]);
      m[1] = fma(wb, t4, m[1]);
      m[2] = fma(wb, t5, m[2]);
      m[3] = fma(wb, t6, m[3]);
    }
    {
      const double wb = w * t4;
      m[4] = fma(wb, t6, m[4]);
    }
    {
      const double wb = w * t5;
      m[5] = fma(wb, t6, m[5]);
    }
    {
      const double wb = w * t6;
      m[6] = fma(wb, t6, m[6]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.14285714285714285 - m[0];
    m[1] = 0.023809523809523808 - m[1];
    m[2] = 0.009523809523809525 - m[2];
    m[3] = 0.007142857142857143 - m[3];
    m[4] = 0.009523809523809525 - m[4];
    m[5] = 0.023809523809523808 - m[5];
    m[6] = 0.14285714285714285 - m[6];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + m[2];
    mk[1] = m[1] + 2.0 * m[2] + m[3];
    mk[2] = m[2] + 2.0 * m[3] + m[4];
    mk[3] = m[3] + 2.0 * m[4] + m[5];
    mk[4] = m[4] + 2.0 * m[5] + m[6];
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 3;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0] - 5.0 * m[1] + 8.25 * m[2] - 5.0 * m[3] + m[4];
      const double K_ = Gs[0] * (30.25 * mk[0] - 77.0 * mk[1] + 60.0 * mk[2] - 14.0 * mk[3] + mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1] - 5.0 * m[2] + 8.25 * m[3] - 5.0 * m[4] + m[5];
      const double K_ = Gs[1] * (5.5 * mk[0] - 45.5 * mk[1] + 80.25 * mk[2] - 45.5 * mk[3] + 5.5 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[4] = v_;
    }
    {
      const double M_ = 9.0 * m[1] - 27.0 * m[2] + 20.25 * m[3] - 4.5 * m[4];
      const double K_ = Gs[0] * (123.75 * mk[1] - 182.25 * mk[2] + 54.0 * mk[3] - 4.5 * mk[4]) + Gs[1] * (49.5 * mk[0] - 87.75 * mk[1] + 40.5 * mk[2] - 4.5 * mk[3]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[2] = v_;
      out[8] = v_;
    }
    {
      const double M_ = -4.5 * m[1] + 20.25 * m[2] - 27.0 * m[3] + 9.0 * m[4];
      const double K_ = Gs[0] * (-24.75 * mk[1] + 81.0 * mk[2] - 67.5 * mk[3] + 9.0 * mk[4]) + Gs[1] * (-24.75 * mk[0] + 155.25 * mk[1] - 162.0 * mk[2] + 22.5 * mk[3]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[3] = v_;
      out[12] = v_;
    }
    {
      const double M_ = m[2] - 5.0 * m[3] + 8.25 * m[4] - 5.0 * m[5] + m[6];
      const double K_ = Gs[2] * (mk[0] - 14.0 * mk[1] + 60.0 * mk[2] - 77.0 * mk[3] + 30.25 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[5] = v_;
    }
    {
      const double M_ = 9.0 * m[2] - 27.0 * m[3] + 20.25 * m[4] - 4.5 * m[5];
      const double K_ = Gs[1] * (22.5 * mk[1] - 162.0 * mk[2] + 155.25 * mk[3] - 24.75 * mk[4]) + Gs[2] * (9.0 * mk[0] - 67.5 * mk[1] + 81.0 * mk[2] - 24.75 * mk[3]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[6] = v_;
      out[9] = v_;
    }
    {
      const double M_ = -4.5 * m[2] + 20.25 * m[3] - 27.0 * m[4] + 9.0 * m[5];
      const double K_ = Gs[1] * (-4.5 * mk[1] + 40.5 * mk[2] - 87.75 * mk[3] + 49.5 * mk[4]) + Gs[2] * (-4.5 * mk[0] + 54.0 * mk[1] - 182.25 * mk[2] + 123.75 * mk[3]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[7] = v_;
      out[13] = v_;
    }
    {
      const double M_ = 81.0 * m[2] - 81.0 * m[3] + 20.25 * m[4];
      const double K_ = Gs[0] * (506.25 * mk[2] - 202.5 * mk[3] + 20.25 * mk[4]) + Gs[1] * (405.0 * mk[1] - 283.5 * mk[2] + 40.5 * mk[3]) + Gs[2] * (81.0 * mk[0] - 81.0 * mk[1] + 20.25 * mk[2]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[10] = v_;
    }
    {
      const double M_ = -40.5 * m[2] + 101.25 * m[3] - 40.5 * m[4];
      const double K_ = Gs[0] * (-101.25 * mk[2] + 222.75 * mk[3] - 40.5 * mk[4]) + Gs[1] * (-141.75 * mk[1] + 627.75 * mk[2] - 141.75 * mk[3]) + Gs[2] * (-40.5 * mk[0] + 222.75 * mk[1] - 101.25 * mk[2]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[11] = v_;
      out[14] = v_;
    }
    {
      const double M_ = 20.25 * m[2] - 81.0 * m[3] + 81.0 * m[4];
      const double K_ = Gs[0] * (20.25 * mk[2] - 81.0 * mk[3] + 81.0 * mk[4]) + Gs[1] * (40.5 * mk[1] - 283.5 * mk[2] + 405.0 * mk[3]) + Gs[2] * (20.25 * mk[0] - 202.5 * mk[1] + 506.25 * mk[2]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[15] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + 0.5 * m[1] - 3.5 * m[2] - 3.5 * m[3] + 0.5 * m[4] + m[5]));
    out[1] = (T)(s * (m[1] + 0.5 * m[2] - 3.5 * m[3] - 3.5 * m[4] + 0.5 * m[5] + m[6]));
    out[2] = (T)(s * (9.0 * m[1] + 22.5 * m[2] + 13.5 * m[3] - 4.5 * m[4] - 4.5 * m[5]));
    out[3] = (T)(s * (-4.5 * m[1] - 4.5 * m[2] + 13.5 * m[3] + 22.5 * m[4] + 9.0 * m[5]));
  }
};  // 114 coefficient terms
template <>
struct Moments<2, 1> {
  static constexpr int NM = 6;  // degree-2 moments
  static constexpr int NK = 1;  // degree-0 moments
  static constexpr int NQ = 3;  // degree-1 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    {
      const double wb = w * l[0];
      m[0] = fma(wb, l[0], m[0]);
      m[1] = fma(wb, l[1], m[1]);
      m[2] = fma(wb, l[2], m[2]);
    }
    {
      const double wb = w * l[1];
      m[3] = fma(wb, l[1], m[3]);
      m[4] = fma(wb, l[2], m[4]);
    }
    {
      const double wb = w * l[2];
      m[5] = fma(wb, l[2], m[5]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.08333333333333333 - m[0];
    m[1] = 0.041666666666666664 - m[1];
    m[2] = 0.041666666666666664 - m[2];
    m[3] = 0.08333333333333333 - m[3];
    m[4] = 0.041666666666666664 - m[4];
    m[5] = 0.08333333333333333 - m[5];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + m[3] + 2.0 * m[4] + m[5];
  }
  static constexpr int NH = 3;  // h: coefficients of H_1 .. H_1
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/2))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    h[2] = h[2] + l[2];
    m[0] = fma(l[0], h[0], m[0]);
    m[1] = fma(l[1], h[0], fma(l[0], h[1], m[1]));
    m[2] = fma(l[2], h[0], fma(l[0], h[2], m[2]));
    m[3] = fma(l[1], h[1], m[3]);
    m[4] = fma(l[2], h[1], fma(l[1], h[2], m[4]));
    m[5] = fma(l[2], h[2], m[5]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 2.0;
    m[3] *= 2.0;
    m[5] *= 2.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 6;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0];
      const double K_ = Gs[0] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1];
      const double K_ = Gs[1] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[3] = v_;
    }
    {
      const double M_ = m[2];
      const double K_ = Gs[2] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[2] = v_;
      out[6] = v_;
    }
    {
      const double M_ = m[3];
      const double K_ = Gs[3] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[4] = v_;
    }
    {
      const double M_ = m[4];
      const double K_ = Gs[4] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[5] = v_;
      out[7] = v_;
    }
    {
      const double M_ = m[5];
      const double K_ = Gs[5] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[8] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1] + m[2]));
    out[1] = (T)(s * (m[1] + m[3] + m[4]));
    out[2] = (T)(s * (m[2] + m[4] + m[5]));
  }
};  // 12 coefficient terms
template <>
struct Moments<2, 2> {
  static constexpr int NM = 15;  // degree-4 moments
  static constexpr int NK = 6;  // degree-2 moments
  static constexpr int NQ = 6;  // degree-2 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[2] * l[0];
    const double t3 = l[1] * l[1];
    const double t4 = l[2] * l[1];
    const double t5 = l[2] * l[2];
    {
      const double wb = w * t0;
      m[0] = fma(wb, t0, m[0]);
      m[1] = fma(wb, t1, m[1]);
      m[2] = fma(wb, t2, m[2]);
      m[3] = fma(wb, t3, m[3]);
      m[4] = fma(wb, t4, m[4]);
      m[5] = fma(wb, t5, m[5]);
    }
    {
      const double wb = w * t1;
      m[6] = fma(wb, t3, m[6]);
      m[7] = fma(wb, t4, m[7]);
      m[8] = fma(wb, t5, m[8]);
    }
    {
      const double wb = w * t2;
      m[9] = fma(wb, t5, m[9]);
    }
    {
      const double wb = w * t3;
      m[10] = fma(wb, t3, m[10]);
      m[11] = fma(wb, t4, m[11]);
      m[12] = fma(wb, t5, m[12]);
    }
    {
      const double wb = w * t4;
      m[13] = fma(wb, t5, m[13]);
    }
    {
      const double wb = w * t5;
      m[14] = fma(wb, t5, m[14]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.03333333333333333 - m[0];
    m[1] = 0.008333333333333333 - m[1];
    m[2] = 0.008333333333333333 - m[2];
    m[3] = 0.005555555555555556 - m[3];
    m[4] = 0.002777777777777778 - m[4];
    m[5] = 0.005555555555555556 - m[5];
    m[6] = 0.008333333333333333 - m[6];
    m[7] = 0.002777777777777778 - m[7];
    m[8] = 0.002777777777777778 - m[8];
    m[9] = 0.008333333333333333 - m[9];
    m[10] = 0.03333333333333333 - m[10];
    m[11] = 0.008333333333333333 - m[11];
    m[12] = 0.005555555555555556 - m[12];
    m[13] = 0.008333333333333333 - m[13];
    m[14] = 0.03333333333333333 - m[14];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + m[3] + 2.0 * m[4] + m[5];
    mk[1] = m[1] + 2.0 * m[3] + 2.0 * m[4] + m[6] + 2.0 * m[7] + m[8];
    mk[2] = m[2] + 2.0 * m[4] + 2.0 * m[5] + m[7] + 2.0 * m[8] + m[9];
    mk[3] = m[3] + 2.0 * m[6] + 2.0 * m[7] + m[10] + 2.0 * m[11] + m[12];
    mk[4] = m[4] + 2.0 * m[7] + 2.0 * m[8] + m[11] + 2.0 * m[12] + m[13];
    mk[5] = m[5] + 2.0 * m[8] + 2.0 * m[9] + m[12] + 2.0 * m[13] + m[14];
  }
  static constexpr int NH = 19;  // h: coefficients of H_1 .. H_3
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/4))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    h[2] = h[2] + l[2];
    h[3] = fma(l[0], h[0], h[3]);
    h[4] = fma(l[1], h[0], fma(l[0], h[1], h[4]));
    h[5] = fma(l[2], h[0], fma(l[0], h[2], h[5]));
    h[6] = fma(l[1], h[1], h[6]);
    h[7] = fma(l[2], h[1], fma(l[1], h[2], h[7]));
    h[8] = fma(l[2], h[2], h[8]);
    h[9] = fma(l[0], h[3], h[9]);
    h[10] = fma(l[1], h[3], fma(l[0], h[4], h[10]));
    h[11] = fma(l[2], h[3], fma(l[0], h[5], h[11]));
    h[12] = fma(l[1], h[4], fma(l[0], h[6], h[12]));
    h[13] = fma(l[2], h[4], fma(l[1], h[5], fma(l[0], h[7], h[13])));
    h[14] = fma(l[2], h[5], fma(l[0], h[8], h[14]));
    h[15] = fma(l[1], h[6], h[15]);
    h[16] = fma(l[2], h[6], fma(l[1], h[7], h[16]));
    h[17] = fma(l[2], h[7], fma(l[1], h[8], h[17]));
    h[18] = fma(l[2], h[8], h[18]);
    m[0] = fma(l[0], h[9], m[0]);
    m[1] = fma(l[1], h[9], fma(l[0], h[10], m[1]));
    m[2] = fma(l[2], h[9], fma(l[0], h[11], m[2]));
    m[3] = fma(l[1], h[10], fma(l[0], h[12], m[3]));
    m[4] = fma(l[2], h[10], fma(l[1], h[11], fma(l[0], h[13], m[4])));
    m[5] = fma(l[2], h[11], fma(l[0], h[14], m[5]));
    m[6] = fma(l[1], h[12], fma(l[0], h[15], m[6]));
    m[7] = fma(l[2], h[12], fma(l[1], h[13], fma(l[0], h[16], m[7])));
    m[8] = fma(l[2], h[13], fma(l[1], h[14], fma(l[0], h[17], m[8])));
    m[9] = fma(l[2], h[14], fma(l[0], h[18], m[9]));
    m[10] = fma(l[1], h[15], m[10]);
    m[11] = fma(l[2], h[15], fma(l[1], h[16], m[11]));
    m[12] = fma(l[2], h[16], fma(l[1], h[17], m[12]));
    m[13] = fma(l[2], h[17], fma(l[1], h[18], m[13]));
    m[14] = fma(l[2], h[18], m[14]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 24.0;
    m[1] *= 6.0;
    m[2] *= 6.0;
    m[3] *= 4.0;
    m[4] *= 2.0;
    m[5] *= 4.0;
    m[6] *= 6.0;
    m[7] *= 2.0;
    m[8] *= 2.0;
    m[9] *= 6.0;
    m[10] *= 24.0;
    m[11] *= 6.0;
    m[12] *= 4.0;
    m[13] *= 6.0;
    m[14] *= 24.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 6;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    const double sm2_ = 2.0 * sm;
    const double sm4_ = 4.0 * sm;
    const double sk4_ = 4.0 * sk;
    const double Gd1 = 2.0 * Gs[1];
    const double Gd2 = 2.0 * Gs[2];
    const double Gd4 = 2.0 * Gs[4];
    // A = sm M^B + sk K^B (Bernstein basis, upper triangle)
    const double A0_0 = sm * m[0] + sk4_ * (Gs[0] * mk[0]);
    const double A0_1 = sm2_ * m[1] + sk4_ * (Gs[0] * mk[1] + Gs[1] * mk[0]);
    const double A0_2 = sm2_ * m[2] + sk4_ * (Gs[0] * mk[2] + Gs[2] * mk[0]);
    const double A0_3 = sm * m[3] + sk4_ * (Gs[1] * mk[1]);
    const double A0_4 = sm2_ * m[4] + sk4_ * (Gs[1] * mk[2] + Gs[2] * mk[1]);
    const double A0_5 = sm * m[5] + sk4_ * (Gs[2] * mk[2]);
    const double A1_1 = sm4_ * m[3] + sk4_ * (Gs[0] * mk[3] + Gd1 * mk[1] + Gs[3] * mk[0]);
    const double A1_2 = sm4_ * m[4] + sk4_ * (Gs[0] * mk[4] + Gs[1] * mk[2] + Gs[2] * mk[1] + Gs[4] * mk[0]);
    const double A1_3 = sm2_ * m[6] + sk4_ * (Gs[1] * mk[3] + Gs[3] * mk[1]);
    const double A1_4 = sm4_ * m[7] + sk4_ * (Gs[1] * mk[4] + Gs[2] * mk[3] + Gs[3] * mk[2] + Gs[4] * mk[1]);
    const double A1_5 = sm2_ * m[8] + sk4_ * (Gs[2] * mk[4] + Gs[4] * mk[2]);
    const double A2_2 = sm4_ * m[5] + sk4_ * (Gs[0] * mk[5] + Gd2 * mk[2] + Gs[5] * mk[0]);
    const double A2_3 = sm2_ * m[7] + sk4_ * (Gs[1] * mk[4] + Gs[4] * mk[1]);
    const double A2_4 = sm4_ * m[8] + sk4_ * (Gs[1] * mk[5] + Gs[2] * mk[4] + Gs[4] * mk[2] + Gs[5] * mk[1]);
    const double A2_5 = sm2_ * m[9] + sk4_ * (Gs[2] * mk[5] + Gs[5] * mk[2]);
    const double A3_3 = sm * m[10] + sk4_ * (Gs[3] * mk[3]);
    const double A3_4 = sm2_ * m[11] + sk4_ * (Gs[3] * mk[4] + Gs[4] * mk[3]);
    const double A3_5 = sm * m[12] + sk4_ * (Gs[4] * mk[4]);
    const double A4_4 = sm4_ * m[12] + sk4_ * (Gs[3] * mk[5] + Gd4 * mk[4] + Gs[5] * mk[3]);
    const double A4_5 = sm2_ * m[13] + sk4_ * (Gs[4] * mk[5] + Gs[5] * mk[4]);
    const double A5_5 = sm * m[14] + sk4_ * (Gs[5] * mk[5]);
    // L = T A T^T: a column b of X = A T^T where T's row b has several
    // entries, otherwise the entries of A directly
    {
      const double X0 = A0_0 - 0.5 * A0_1 - 0.5 * A0_2;
      const double X1 = A0_1 - 0.5 * A1_1 - 0.5 * A1_2;
      const double X2 = A0_2 - 0.5 * A1_2 - 0.5 * A2_2;
      const double X3 = A0_3 - 0.5 * A1_3 - 0.5 * A2_3;
      const double X4 = A0_4 - 0.5 * A1_4 - 0.5 * A2_4;
      const double X5 = A0_5 - 0.5 * A1_5 - 0.5 * A2_5;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2);
      out[0] = v0_;
    }
    {
      const double X0 = -0.5 * A0_1 + A0_3 - 0.5 * A0_4;
      const double X1 = -0.5 * A1_1 + A1_3 - 0.5 * A1_4;
      const double X2 = -0.5 * A1_2 + A2_3 - 0.5 * A2_4;
      const double X3 = -0.5 * A1_3 + A3_3 - 0.5 * A3_4;
      const double X4 = -0.5 * A1_4 + A3_4 - 0.5 * A4_4;
      const double X5 = -0.5 * A1_5 + A3_5 - 0.5 * A4_5;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2);
      out[1] = v0_;
      out[6] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X3 - 0.5 * X4);
      out[7] = v1_;
    }
    {
      const double X0 = -0.5 * A0_2 - 0.5 * A0_4 + A0_5;
      const double X1 = -0.5 * A1_2 - 0.5 * A1_4 + A1_5;
      const double X2 = -0.5 * A2_2 - 0.5 * A2_4 + A2_5;
      const double X3 = -0.5 * A2_3 - 0.5 * A3_4 + A3_5;
      const double X4 = -0.5 * A2_4 - 0.5 * A4_4 + A4_5;
      const double X5 = -0.5 * A2_5 - 0.5 * A4_5 + A5_5;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2);
      out[2] = v0_;
      out[12] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X3 - 0.5 * X4);
      out[8] = v1_;
      out[13] = v1_;
      const T v2_ = (T)(-0.5 * X2 - 0.5 * X4 + X5);
      out[14] = v2_;
    }
    {
      const T v0_ = (T)(2.0 * A0_1 - A1_1 - A1_2);
      out[3] = v0_;
      out[18] = v0_;
      const T v1_ = (T)(-A1_1 + 2.0 * A1_3 - A1_4);
      out[9] = v1_;
      out[19] = v1_;
      const T v2_ = (T)(-A1_2 - A1_4 + 2.0 * A1_5);
      out[15] = v2_;
      out[20] = v2_;
      const T v3_ = (T)(4.0 * A1_1);
      out[21] = v3_;
    }
    {
      const T v0_ = (T)(2.0 * A0_2 - A1_2 - A2_2);
      out[4] = v0_;
      out[24] = v0_;
      const T v1_ = (T)(-A1_2 + 2.0 * A2_3 - A2_4);
      out[10] = v1_;
      out[25] = v1_;
      const T v2_ = (T)(-A2_2 - A2_4 + 2.0 * A2_5);
      out[16] = v2_;
      out[26] = v2_;
      const T v3_ = (T)(4.0 * A1_2);
      out[22] = v3_;
      out[27] = v3_;
      const T v4_ = (T)(4.0 * A2_2);
      out[28] = v4_;
    }
    {
      const T v0_ = (T)(2.0 * A0_4 - A1_4 - A2_4);
      out[5] = v0_;
      out[30] = v0_;
      const T v1_ = (T)(-A1_4 + 2.0 * A3_4 - A4_4);
      out[11] = v1_;
      out[31] = v1_;
      const T v2_ = (T)(-A2_4 - A4_4 + 2.0 * A4_5);
      out[17] = v2_;
      out[32] = v2_;
      const T v3_ = (T)(4.0 * A1_4);
      out[23] = v3_;
      out[33] = v3_;
      const T v4_ = (T)(4.0 * A2_4);
      out[29] = v4_;
      out[34] = v4_;
      const T v5_ = (T)(4.0 * A4_4);
      out[35] = v5_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1] + m[2] - m[3] - 2.0 * m[4] - m[5] - m[6] - 3.0 * m[7] - 3.0 * m[8] - m[9]));
    out[1] = (T)(s * (-m[1] - m[3] - 3.0 * m[4] + m[6] - 2.0 * m[7] - 3.0 * m[8] + m[10] + m[11] - m[12] - m[13]));
    out[2] = (T)(s * (-m[2] - 3.0 * m[4] - m[5] - 3.0 * m[7] - 2.0 * m[8] + m[9] - m[11] - m[12] + m[13] + m[14]));
    out[3] = (T)(s * (4.0 * m[1] + 8.0 * m[3] + 8.0 * m[4] + 4.0 * m[6] + 8.0 * m[7] + 4.0 * m[8]));
    out[4] = (T)(s * (4.0 * m[2] + 8.0 * m[4] + 8.0 * m[5] + 4.0 * m[7] + 8.0 * m[8] + 4.0 * m[9]));
    out[5] = (T)(s * (4.0 * m[4] + 8.0 * m[7] + 8.0 * m[8] + 4.0 * m[11] + 8.0 * m[12] + 4.0 * m[13]));
  }
};  // 171 coefficient terms
template <>
struct Moments<2, 3> {
  static constexpr int NM = 28;  // degree-6 moments
  static constexpr int NK = 15;  // degree-4 moments
  static constexpr int NQ = 10;  // degree-3 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[2] * l[0];
    const double t3 = l[1] * l[1];
    const double t4 = l[2] * l[1];
    const double t5 = l[2] * l[2];
    const double t6 = t0 * l[0];
    const double t7 = t1 * l[0];
    const double t8 = t2 * l[0];
    const double t9 = t3 * l[0];
    const double t10 = t4 * l[0];
    const double t11 = t5 * l[0];
    const double t12 = t3 * l[1];
    const double t13 = t4 * l[1];
    const double t14 = t5 * l[1];
    const double t15 = t5 * l[2];
    {
      const double wb = w * t6;
      m[0] = fma(wb, t6, m[0]);
      m[1] = fma(wb, t7, m[1]);
      m[2] = fma(wb, t8, m[2]);
      m[3] = fma(wb, t9, m[3]);
      m[4] = fma(wb, t10, m[4]);
      m[5] = fma(wb, t11, m[5]);
      m[6] = fma(wb, t12, m[6]);
      m[7] = fma(wb, t13, m[7]);
      m[8] = fma(wb, t14, m[8]);
      m[9] = fma(wb, t15, m[9]);
    }
    {
      const double wb = w * t7;
      m[10] = fma(wb, t12, m[10]);
      m[11] = fma(wb, t13, m[11]);
      m[12] = fma(wb, t14, m[12]);
      m[13] = fma(wb, t15, m[13]);
    }
    {
      const double wb = w * t8;
      m[14] = fma(wb, t15, m[14]);
    }
    {
      const double wb = w * t9;
      m[15] = fma(wb, t12, m[15]);
      m[16] = fma(wb, t13, m[16]);
      m[17] = fma(wb, t14, m[17]);
      m[18] = fma(wb, t15, m[18]);
    }
    {
      const double wb = w * t10;
      m[19] = fma(wb, t15, m[19]);
    }
    {
      const double wb = w * t11;
      m[20] = fma(wb, t15, m[20]);
    }
    {
      const double wb = w * t12;
      m[21] = fma(wb, t12, m[21]);
      m[22] = fma(wb, t13, m[22]);
      m[23] = fma(wb, t14, m[23]);
      m[24] = fma(wb, t15, m[24]);
    }
    {
      const double wb = w * t13;
      m[25] = fma(wb, t15, m[25]);
    }
    {
      const double wb = w * t14;
      m[26] = fma(wb, t15, m[26]);
    }
    {
      const double wb = w * t15;
      m[27] = fma(wb, t15, m[27]);
    }
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.017857142857142856 - m[0];
    m[1] = 0.002976190476190476 - m[1];
    m[2] = 0.002976190476190476 - m[2];
    m[3] = 0.0011904761904761906 - m[3];
    m[4] = 0.0005952380952380953 - m[4];
    m[5] = 0.0011904761904761906 - m[5];
    m[6] = 0.0008928571428571428 - m[6];
    m[7] = 0.00029761904761904765 - m[7];
    m[8] = 0.00029761904761904765 - m[8];
    m[9] = 0.0008928571428571428 - m[9];
    m[10] = 0.0011904761904761906 - m[10];
    m[11] = 0.00029761904761904765 - m[11];
    m[12] = 0.0001984126984126984 - m[12];
    m[13] = 0.00029761904761904765 - m[13];
    m[14] = 0.0011904761904761906 - m[14];
    m[15] = 0.002976190476190476 - m[15];
    m[16] = 0.0005952380952380953 - m[16];
    m[17] = 0.00029761904761904765 - m[17];
    m[18] = 0.00029761904761904765 - m[18];
    m[19] = 0.0005952380952380953 - m[19];
    m[20] = 0.002976190476190476 - m[20];
    m[21] = 0.017857142857142856 - m[21];
    m[22] = 0.002976190476190476 - m[22];
    m[23] = 0.0011904761904761906 - m[23];
    m[24] = 0.0008928571428571428 - m[24];
    m[25] = 0.0011904761904761906 - m[25];
    m[26] = 0.002976190476190476 - m[26];
    m[27] = 0.017857142857142856 - m[27];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + m[3] + 2.0 * m[4] + m[5];
    mk[1] = m[1] + 2.0 * m[3] + 2.0 * m[4] + m[6] + 2.0 * m[7] + m[8];
    mk[2] = m[2] + 2.0 * m[4] + 2.0 * m[5] + m[7] + 2.0 * m[8] + m[9];
    mk[3] = m[3] + 2.0 * m[6] + 2.0 * m[7] + m[10] + 2.0 * m[11] + m[12];
    mk[4] = m[4] + 2.0 * m[7] + 2.0 * m[8] + m[11] + 2.0 * m[12] + m[13];
    mk[5] = m[5] + 2.0 * m[8] + 2.0 * m[9] + m[12] + 2.0 * m[13] + m[14];
    mk[6] = m[6] + 2.0 * m[10] + 2.0 * m[11] + m[15] + 2.0 * m[16] + m[17];
    mk[7] = m[7] + 2.0 * m[11] + 2.0 * m[12] + m[16] + 2.0 * m[17] + m[18];
    mk[8] = m[8] + 2.0 * m[12] + 2.0 * m[13] + m[17] + 2.0 * m[18] + m[19];
    mk[9] = m[9] + 2.0 * m[13] + 2.0 * m[14] + m[18] + 2.0 * m[19] + m[20];
    mk[10] = m[10] + 2.0 * m[15] + 2.0 * m[16] + m[21] + 2.0 * m[22] + m[23];
    mk[11] = m[11] + 2.0 * m[16] + 2.0 * m[17] + m[22] + 2.0 * m[23] + m[24];
    mk[12] = m[12] + 2.0 * m[17] + 2.0 * m[18] + m[23] + 2.0 * m[24] + m[25];
    mk[13] = m[13] + 2.0 * m[18] + 2.0 * m[19] + m[24] + 2.0 * m[25] + m[26];
    mk[14] = m[14] + 2.0 * m[19] + 2.0 * m[20] + m[25] + 2.0 * m[26] + m[27];
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 6;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0] - 5.0 * m[1] - 5.0 * m[2] + 8.25 * m[3] + 16.5 * m[4] + 8.25 * m[5] - 5.0 * m[6] - 15.0 * m[7] - 15.0 * m[8] - 5.0 * m[9] + m[10] + 4.0 * m[11] + 6.0 * m[12] + 4.0 * m[13] + m[14];
      const double K_ = Gs[0] * (30.25 * mk[0] - 77.0 * mk[1] - 77.0 * mk[2] + 60.0 * mk[3] + 120.0 * mk[4] + 60.0 * mk[5] - 14.0 * mk[6] - 42.0 * mk[7] - 42.0 * mk[8] - 14.0 * mk[9] + mk[10] + 4.0 * mk[11] + 6.0 * mk[12] + 4.0 * mk[13] + mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1] - 5.0 * m[3] - 0.5 * m[4] + 8.25 * m[6] + 0.75 * m[7] - 3.0 * m[8] - 5.0 * m[10] + 0.75 * m[11] + 5.25 * m[12] - 0.5 * m[13] + m[15] - 0.5 * m[16] - 3.0 * m[17] - 0.5 * m[18] + m[19];
      const double K_ = Gs[1] * (5.5 * mk[0] - 45.5 * mk[1] + 4.0 * mk[2] + 80.25 * mk[3] - 1.5 * mk[4] - 7.5 * mk[5] - 45.5 * mk[6] - 1.5 * mk[7] + 39.0 * mk[8] - 5.0 * mk[9] + 5.5 * mk[10] + 4.0 * mk[11] - 7.5 * mk[12] - 5.0 * mk[13] + mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[10] = v_;
    }
    {
      const double M_ = m[2] - 0.5 * m[4] - 5.0 * m[5] - 3.0 * m[7] + 0.75 * m[8] + 8.25 * m[9] - 0.5 * m[11] + 5.25 * m[12] + 0.75 * m[13] - 5.0 * m[14] + m[16] - 0.5 * m[17] - 3.0 * m[18] - 0.5 * m[19] + m[20];
      const double K_ = Gs[2] * (5.5 * mk[0] + 4.0 * mk[1] - 45.5 * mk[2] - 7.5 * mk[3] - 1.5 * mk[4] + 80.25 * mk[5] - 5.0 * mk[6] + 39.0 * mk[7] - 1.5 * mk[8] - 45.5 * mk[9] + mk[10] - 5.0 * mk[11] - 7.5 * mk[12] + 4.0 * mk[13] + 5.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[2] = v_;
      out[20] = v_;
    }
    {
      const double M_ = 9.0 * m[1] - 27.0 * m[3] - 27.0 * m[4] + 20.25 * m[6] + 40.5 * m[7] + 20.25 * m[8] - 4.5 * m[10] - 13.5 * m[11] - 13.5 * m[12] - 4.5 * m[13];
      const double K_ = Gs[0] * (123.75 * mk[1] - 182.25 * mk[3] - 182.25 * mk[4] + 54.0 * mk[6] + 108.0 * mk[7] + 54.0 * mk[8] - 4.5 * mk[10] - 13.5 * mk[11] - 13.5 * mk[12] - 4.5 * mk[13]) + Gs[1] * (49.5 * mk[0] - 87.75 * mk[1] - 87.75 * mk[2] + 40.5 * mk[3] + 81.0 * mk[4] + 40.5 * mk[5] - 4.5 * mk[6] - 13.5 * mk[7] - 13.5 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[3] = v_;
      out[30] = v_;
    }
    {
      const double M_ = -4.5 * m[1] + 20.25 * m[3] + 6.75 * m[4] - 27.0 * m[6] - 20.25 * m[7] + 6.75 * m[8] + 9.0 * m[10] + 13.5 * m[11] - 4.5 * m[13];
      const double K_ = Gs[0] * (-24.75 * mk[1] + 81.0 * mk[3] + 6.75 * mk[4] - 67.5 * mk[6] - 40.5 * mk[7] + 27.0 * mk[8] + 9.0 * mk[10] + 13.5 * mk[11] - 4.5 * mk[13]) + Gs[1] * (-24.75 * mk[0] + 155.25 * mk[1] + 6.75 * mk[2] - 162.0 * mk[3] - 135.0 * mk[4] + 27.0 * mk[5] + 22.5 * mk[6] + 40.5 * mk[7] + 13.5 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[4] = v_;
      out[40] = v_;
    }
    {
      const double M_ = 9.0 * m[2] - 27.0 * m[4] - 27.0 * m[5] + 20.25 * m[7] + 40.5 * m[8] + 20.25 * m[9] - 4.5 * m[11] - 13.5 * m[12] - 13.5 * m[13] - 4.5 * m[14];
      const double K_ = Gs[0] * (123.75 * mk[2] - 182.25 * mk[4] - 182.25 * mk[5] + 54.0 * mk[7] + 108.0 * mk[8] + 54.0 * mk[9] - 4.5 * mk[11] - 13.5 * mk[12] - 13.5 * mk[13] - 4.5 * mk[14]) + Gs[2] * (49.5 * mk[0] - 87.75 * mk[1] - 87.75 * mk[2] + 40.5 * mk[3] + 81.0 * mk[4] + 40.5 * mk[5] - 4.5 * mk[6] - 13.5 * mk[7] - 13.5 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[5] = v_;
      out[50] = v_;
    }
    {
      const double M_ = -4.5 * m[2] + 6.75 * m[4] + 20.25 * m[5] + 6.75 * m[7] - 20.25 * m[8] - 27.0 * m[9] - 4.5 * m[11] + 13.5 * m[13] + 9.0 * m[14];
      const double K_ = Gs[0] * (-24.75 * mk[2] + 6.75 * mk[4] + 81.0 * mk[5] + 27.0 * mk[7] - 40.5 * mk[8] - 67.5 * mk[9] - 4.5 * mk[11] + 13.5 * mk[13] + 9.0 * mk[14]) + Gs[2] * (-24.75 * mk[0] + 6.75 * mk[1] + 155.25 * mk[2] + 27.0 * mk[3] - 135.0 * mk[4] - 162.0 * mk[5] - 4.5 * mk[6] + 13.5 * mk[7] + 40.5 * mk[8] + 22.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[6] = v_;
      out[60] = v_;
    }
    {
      const double M_ = -4.5 * m[4] + 20.25 * m[7] + 6.75 * m[8] - 27.0 * m[11] - 20.25 * m[12] + 6.75 * m[13] + 9.0 * m[16] + 13.5 * m[17] - 4.5 * m[19];
      const double K_ = Gs[1] * (-24.75 * mk[2] + 155.25 * mk[4] + 6.75 * mk[5] - 162.0 * mk[7] - 135.0 * mk[8] + 27.0 * mk[9] + 22.5 * mk[11] + 40.5 * mk[12] + 13.5 * mk[13] - 4.5 * mk[14]) + Gs[2] * (-24.75 * mk[1] + 81.0 * mk[3] + 6.75 * mk[4] - 67.5 * mk[6] - 40.5 * mk[7] + 27.0 * mk[8] + 9.0 * mk[10] + 13.5 * mk[11] - 4.5 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[7] = v_;
      out[70] = v_;
    }
    {
      const double M_ = -4.5 * m[4] + 6.75 * m[7] + 20.25 * m[8] + 6.75 * m[11] - 20.25 * m[12] - 27.0 * m[13] - 4.5 * m[16] + 13.5 * m[18] + 9.0 * m[19];
      const double K_ = Gs[1] * (-24.75 * mk[2] + 6.75 * mk[4] + 81.0 * mk[5] + 27.0 * mk[7] - 40.5 * mk[8] - 67.5 * mk[9] - 4.5 * mk[11] + 13.5 * mk[13] + 9.0 * mk[14]) + Gs[2] * (-24.75 * mk[1] + 6.75 * mk[3] + 155.25 * mk[4] + 27.0 * mk[6] - 135.0 * mk[7] - 162.0 * mk[8] - 4.5 * mk[10] + 13.5 * mk[11] + 40.5 * mk[12] + 22.5 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[8] = v_;
      out[80] = v_;
    }
    {
      const double M_ = 27.0 * m[4] - 67.5 * m[7] - 67.5 * m[8] + 27.0 * m[11] + 54.0 * m[12] + 27.0 * m[13];
      const double K_ = Gs[0] * (148.5 * mk[4] - 189.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] + 54.0 * mk[12] + 27.0 * mk[13]) + Gs[1] * (148.5 * mk[2] - 189.0 * mk[4] - 189.0 * mk[5] + 27.0 * mk[7] + 54.0 * mk[8] + 27.0 * mk[9]) + Gs[2] * (148.5 * mk[1] - 189.0 * mk[3] - 189.0 * mk[4] + 27.0 * mk[6] + 54.0 * mk[7] + 27.0 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[9] = v_;
      out[90] = v_;
    }
    {
      const double M_ = m[3] - 5.0 * m[6] + 4.0 * m[7] + 8.25 * m[10] - 15.0 * m[11] + 6.0 * m[12] - 5.0 * m[15] + 16.5 * m[16] - 15.0 * m[17] + 4.0 * m[18] + m[21] - 5.0 * m[22] + 8.25 * m[23] - 5.0 * m[24] + m[25];
      const double K_ = Gs[3] * (mk[0] - 14.0 * mk[1] + 4.0 * mk[2] + 60.0 * mk[3] - 42.0 * mk[4] + 6.0 * mk[5] - 77.0 * mk[6] + 120.0 * mk[7] - 42.0 * mk[8] + 4.0 * mk[9] + 30.25 * mk[10] - 77.0 * mk[11] + 60.0 * mk[12] - 14.0 * mk[13] + mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[11] = v_;
    }
    {
      const double M_ = m[4] - 0.5 * m[7] - 0.5 * m[8] - 3.0 * m[11] + 5.25 * m[12] - 3.0 * m[13] - 0.5 * m[16] + 0.75 * m[17] + 0.75 * m[18] - 0.5 * m[19] + m[22] - 5.0 * m[23] + 8.25 * m[24] - 5.0 * m[25] + m[26];
      const double K_ = Gs[4] * (mk[0] - 5.0 * mk[1] - 5.0 * mk[2] - 7.5 * mk[3] + 39.0 * mk[4] - 7.5 * mk[5] + 4.0 * mk[6] - 1.5 * mk[7] - 1.5 * mk[8] + 4.0 * mk[9] + 5.5 * mk[10] - 45.5 * mk[11] + 80.25 * mk[12] - 45.5 * mk[13] + 5.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[12] = v_;
      out[21] = v_;
    }
    {
      const double M_ = 9.0 * m[3] - 27.0 * m[6] + 13.5 * m[7] + 20.25 * m[10] - 20.25 * m[11] - 4.5 * m[15] + 6.75 * m[16] + 6.75 * m[17] - 4.5 * m[18];
      const double K_ = Gs[1] * (22.5 * mk[1] - 162.0 * mk[3] + 40.5 * mk[4] + 155.25 * mk[6] - 135.0 * mk[7] + 13.5 * mk[8] - 24.75 * mk[10] + 6.75 * mk[11] + 27.0 * mk[12] - 4.5 * mk[13]) + Gs[3] * (9.0 * mk[0] - 67.5 * mk[1] + 13.5 * mk[2] + 81.0 * mk[3] - 40.5 * mk[4] - 24.75 * mk[6] + 6.75 * mk[7] + 27.0 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[13] = v_;
      out[31] = v_;
    }
    {
      const double M_ = -4.5 * m[3] + 20.25 * m[6] - 13.5 * m[7] - 27.0 * m[10] + 40.5 * m[11] - 13.5 * m[12] + 9.0 * m[15] - 27.0 * m[16] + 20.25 * m[17] - 4.5 * m[18];
      const double K_ = Gs[1] * (-4.5 * mk[1] + 40.5 * mk[3] - 13.5 * mk[4] - 87.75 * mk[6] + 81.0 * mk[7] - 13.5 * mk[8] + 49.5 * mk[10] - 87.75 * mk[11] + 40.5 * mk[12] - 4.5 * mk[13]) + Gs[3] * (-4.5 * mk[0] + 54.0 * mk[1] - 13.5 * mk[2] - 182.25 * mk[3] + 108.0 * mk[4] - 13.5 * mk[5] + 123.75 * mk[6] - 182.25 * mk[7] + 54.0 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[14] = v_;
      out[41] = v_;
    }
    {
      const double M_ = 9.0 * m[4] - 27.0 * m[7] + 13.5 * m[8] + 20.25 * m[11] - 20.25 * m[12] - 4.5 * m[16] + 6.75 * m[17] + 6.75 * m[18] - 4.5 * m[19];
      const double K_ = Gs[1] * (22.5 * mk[2] - 162.0 * mk[4] + 40.5 * mk[5] + 155.25 * mk[7] - 135.0 * mk[8] + 13.5 * mk[9] - 24.75 * mk[11] + 6.75 * mk[12] + 27.0 * mk[13] - 4.5 * mk[14]) + Gs[4] * (9.0 * mk[0] - 67.5 * mk[1] + 13.5 * mk[2] + 81.0 * mk[3] - 40.5 * mk[4] - 24.75 * mk[6] + 6.75 * mk[7] + 27.0 * mk[8] - 4.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[15] = v_;
      out[51] = v_;
    }
    {
      const double M_ = -4.5 * m[4] + 6.75 * m[7] + 6.75 * m[11] - 20.25 * m[12] + 13.5 * m[13] - 4.5 * m[16] + 20.25 * m[17] - 27.0 * m[18] + 9.0 * m[19];
      const double K_ = Gs[1] * (-4.5 * mk[2] + 27.0 * mk[4] + 6.75 * mk[7] - 40.5 * mk[8] + 13.5 * mk[9] - 24.75 * mk[11] + 81.0 * mk[12] - 67.5 * mk[13] + 9.0 * mk[14]) + Gs[4] * (-4.5 * mk[0] + 27.0 * mk[1] + 13.5 * mk[2] + 6.75 * mk[3] - 135.0 * mk[4] + 40.5 * mk[5] - 24.75 * mk[6] + 155.25 * mk[7] - 162.0 * mk[8] + 22.5 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[16] = v_;
      out[61] = v_;
    }
    {
      const double M_ = -4.5 * m[7] + 20.25 * m[11] - 13.5 * m[12] - 27.0 * m[16] + 40.5 * m[17] - 13.5 * m[18] + 9.0 * m[22] - 27.0 * m[23] + 20.25 * m[24] - 4.5 * m[25];
      const double K_ = Gs[3] * (-4.5 * mk[2] + 54.0 * mk[4] - 13.5 * mk[5] - 182.25 * mk[7] + 108.0 * mk[8] - 13.5 * mk[9] + 123.75 * mk[11] - 182.25 * mk[12] + 54.0 * mk[13] - 4.5 * mk[14]) + Gs[4] * (-4.5 * mk[1] + 40.5 * mk[3] - 13.5 * mk[4] - 87.75 * mk[6] + 81.0 * mk[7] - 13.5 * mk[8] + 49.5 * mk[10] - 87.75 * mk[11] + 40.5 * mk[12] - 4.5 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[17] = v_;
      out[71] = v_;
    }
    {
      const double M_ = -4.5 * m[7] + 6.75 * m[11] + 6.75 * m[16] - 20.25 * m[17] + 13.5 * m[18] - 4.5 * m[22] + 20.25 * m[23] - 27.0 * m[24] + 9.0 * m[25];
      const double K_ = Gs[3] * (-4.5 * mk[2] + 27.0 * mk[4] + 6.75 * mk[7] - 40.5 * mk[8] + 13.5 * mk[9] - 24.75 * mk[11] + 81.0 * mk[12] - 67.5 * mk[13] + 9.0 * mk[14]) + Gs[4] * (-4.5 * mk[1] + 27.0 * mk[3] + 13.5 * mk[4] + 6.75 * mk[6] - 135.0 * mk[7] + 40.5 * mk[8] - 24.75 * mk[10] + 155.25 * mk[11] - 162.0 * mk[12] + 22.5 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[18] = v_;
      out[81] = v_;
    }
    {
      const double M_ = 27.0 * m[7] - 67.5 * m[11] + 54.0 * m[12] + 27.0 * m[16] - 67.5 * m[17] + 27.0 * m[18];
      const double K_ = Gs[1] * (27.0 * mk[4] - 189.0 * mk[7] + 54.0 * mk[8] + 148.5 * mk[11] - 189.0 * mk[12] + 27.0 * mk[13]) + Gs[3] * (27.0 * mk[2] - 189.0 * mk[4] + 54.0 * mk[5] + 148.5 * mk[7] - 189.0 * mk[8] + 27.0 * mk[9]) + Gs[4] * (27.0 * mk[1] - 189.0 * mk[3] + 54.0 * mk[4] + 148.5 * mk[6] - 189.0 * mk[7] + 27.0 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[19] = v_;
      out[91] = v_;
    }
    {
      const double M_ = m[5] + 4.0 * m[8] - 5.0 * m[9] + 6.0 * m[12] - 15.0 * m[13] + 8.25 * m[14] + 4.0 * m[17] - 15.0 * m[18] + 16.5 * m[19] - 5.0 * m[20] + m[23] - 5.0 * m[24] + 8.25 * m[25] - 5.0 * m[26] + m[27];
      const double K_ = Gs[5] * (mk[0] + 4.0 * mk[1] - 14.0 * mk[2] + 6.0 * mk[3] - 42.0 * mk[4] + 60.0 * mk[5] + 4.0 * mk[6] - 42.0 * mk[7] + 120.0 * mk[8] - 77.0 * mk[9] + mk[10] - 14.0 * mk[11] + 60.0 * mk[12] - 77.0 * mk[13] + 30.25 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[22] = v_;
    }
    {
      const double M_ = 9.0 * m[4] + 13.5 * m[7] - 27.0 * m[8] - 20.25 * m[12] + 20.25 * m[13] - 4.5 * m[16] + 6.75 * m[17] + 6.75 * m[18] - 4.5 * m[19];
      const double K_ = Gs[2] * (22.5 * mk[1] + 40.5 * mk[3] - 162.0 * mk[4] + 13.5 * mk[6] - 135.0 * mk[7] + 155.25 * mk[8] - 4.5 * mk[10] + 27.0 * mk[11] + 6.75 * mk[12] - 24.75 * mk[13]) + Gs[4] * (9.0 * mk[0] + 13.5 * mk[1] - 67.5 * mk[2] - 40.5 * mk[4] + 81.0 * mk[5] - 4.5 * mk[6] + 27.0 * mk[7] + 6.75 * mk[8] - 24.75 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[23] = v_;
      out[32] = v_;
    }
    {
      const double M_ = -4.5 * m[4] + 6.75 * m[8] + 13.5 * m[11] - 20.25 * m[12] + 6.75 * m[13] + 9.0 * m[16] - 27.0 * m[17] + 20.25 * m[18] - 4.5 * m[19];
      const double K_ = Gs[2] * (-4.5 * mk[1] + 27.0 * mk[4] + 13.5 * mk[6] - 40.5 * mk[7] + 6.75 * mk[8] + 9.0 * mk[10] - 67.5 * mk[11] + 81.0 * mk[12] - 24.75 * mk[13]) + Gs[4] * (-4.5 * mk[0] + 13.5 * mk[1] + 27.0 * mk[2] + 40.5 * mk[3] - 135.0 * mk[4] + 6.75 * mk[5] + 22.5 * mk[6] - 162.0 * mk[7] + 155.25 * mk[8] - 24.75 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[24] = v_;
      out[42] = v_;
    }
    {
      const double M_ = 9.0 * m[5] + 13.5 * m[8] - 27.0 * m[9] - 20.25 * m[13] + 20.25 * m[14] - 4.5 * m[17] + 6.75 * m[18] + 6.75 * m[19] - 4.5 * m[20];
      const double K_ = Gs[2] * (22.5 * mk[2] + 40.5 * mk[4] - 162.0 * mk[5] + 13.5 * mk[7] - 135.0 * mk[8] + 155.25 * mk[9] - 4.5 * mk[11] + 27.0 * mk[12] + 6.75 * mk[13] - 24.75 * mk[14]) + Gs[5] * (9.0 * mk[0] + 13.5 * mk[1] - 67.5 * mk[2] - 40.5 * mk[4] + 81.0 * mk[5] - 4.5 * mk[6] + 27.0 * mk[7] + 6.75 * mk[8] - 24.75 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[25] = v_;
      out[52] = v_;
    }
    {
      const double M_ = -4.5 * m[5] - 13.5 * m[8] + 20.25 * m[9] - 13.5 * m[12] + 40.5 * m[13] - 27.0 * m[14] - 4.5 * m[17] + 20.25 * m[18] - 27.0 * m[19] + 9.0 * m[20];
      const double K_ = Gs[2] * (-4.5 * mk[2] - 13.5 * mk[4] + 40.5 * mk[5] - 13.5 * mk[7] + 81.0 * mk[8] - 87.75 * mk[9] - 4.5 * mk[11] + 40.5 * mk[12] - 87.75 * mk[13] + 49.5 * mk[14]) + Gs[5] * (-4.5 * mk[0] - 13.5 * mk[1] + 54.0 * mk[2] - 13.5 * mk[3] + 108.0 * mk[4] - 182.25 * mk[5] - 4.5 * mk[6] + 54.0 * mk[7] - 182.25 * mk[8] + 123.75 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[26] = v_;
      out[62] = v_;
    }
    {
      const double M_ = -4.5 * m[8] + 6.75 * m[13] + 13.5 * m[17] - 20.25 * m[18] + 6.75 * m[19] + 9.0 * m[23] - 27.0 * m[24] + 20.25 * m[25] - 4.5 * m[26];
      const double K_ = Gs[4] * (-4.5 * mk[2] + 13.5 * mk[4] + 27.0 * mk[5] + 40.5 * mk[7] - 135.0 * mk[8] + 6.75 * mk[9] + 22.5 * mk[11] - 162.0 * mk[12] + 155.25 * mk[13] - 24.75 * mk[14]) + Gs[5] * (-4.5 * mk[1] + 27.0 * mk[4] + 13.5 * mk[6] - 40.5 * mk[7] + 6.75 * mk[8] + 9.0 * mk[10] - 67.5 * mk[11] + 81.0 * mk[12] - 24.75 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[27] = v_;
      out[72] = v_;
    }
    {
      const double M_ = -4.5 * m[8] - 13.5 * m[12] + 20.25 * m[13] - 13.5 * m[17] + 40.5 * m[18] - 27.0 * m[19] - 4.5 * m[23] + 20.25 * m[24] - 27.0 * m[25] + 9.0 * m[26];
      const double K_ = Gs[4] * (-4.5 * mk[2] - 13.5 * mk[4] + 40.5 * mk[5] - 13.5 * mk[7] + 81.0 * mk[8] - 87.75 * mk[9] - 4.5 * mk[11] + 40.5 * mk[12] - 87.75 * mk[13] + 49.5 * mk[14]) + Gs[5] * (-4.5 * mk[1] - 13.5 * mk[3] + 54.0 * mk[4] - 13.5 * mk[6] + 108.0 * mk[7] - 182.25 * mk[8] - 4.5 * mk[10] + 54.0 * mk[11] - 182.25 * mk[12] + 123.75 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[28] = v_;
      out[82] = v_;
    }
    {
      const double M_ = 27.0 * m[8] + 54.0 * m[12] - 67.5 * m[13] + 27.0 * m[17] - 67.5 * m[18] + 27.0 * m[19];
      const double K_ = Gs[2] * (27.0 * mk[4] + 54.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] - 189.0 * mk[12] + 148.5 * mk[13]) + Gs[4] * (27.0 * mk[2] + 54.0 * mk[4] - 189.0 * mk[5] + 27.0 * mk[7] - 189.0 * mk[8] + 148.5 * mk[9]) + Gs[5] * (27.0 * mk[1] + 54.0 * mk[3] - 189.0 * mk[4] + 27.0 * mk[6] - 189.0 * mk[7] + 148.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[29] = v_;
      out[92] = v_;
    }
    {
      const double M_ = 81.0 * m[3] - 81.0 * m[6] - 81.0 * m[7] + 20.25 * m[10] + 40.5 * m[11] + 20.25 * m[12];
      const double K_ = Gs[0] * (506.25 * mk[3] - 202.5 * mk[6] - 202.5 * mk[7] + 20.25 * mk[10] + 40.5 * mk[11] + 20.25 * mk[12]) + Gs[1] * (405.0 * mk[1] - 283.5 * mk[3] - 283.5 * mk[4] + 40.5 * mk[6] + 81.0 * mk[7] + 40.5 * mk[8]) + Gs[3] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] + 20.25 * mk[3] + 40.5 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[33] = v_;
    }
    {
      const double M_ = -40.5 * m[3] + 101.25 * m[6] - 20.25 * m[7] - 40.5 * m[10] - 20.25 * m[11] + 20.25 * m[12];
      const double K_ = Gs[0] * (-101.25 * mk[3] + 222.75 * mk[6] - 81.0 * mk[7] - 40.5 * mk[10] - 20.25 * mk[11] + 20.25 * mk[12]) + Gs[1] * (-141.75 * mk[1] + 627.75 * mk[3] - 101.25 * mk[4] - 141.75 * mk[6] - 101.25 * mk[7] + 40.5 * mk[8]) + Gs[3] * (-40.5 * mk[0] + 222.75 * mk[1] - 20.25 * mk[2] - 101.25 * mk[3] - 81.0 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[34] = v_;
      out[43] = v_;
    }
    {
      const double M_ = 81.0 * m[4] - 81.0 * m[7] - 81.0 * m[8] + 20.25 * m[11] + 40.5 * m[12] + 20.25 * m[13];
      const double K_ = Gs[0] * (506.25 * mk[4] - 202.5 * mk[7] - 202.5 * mk[8] + 20.25 * mk[11] + 40.5 * mk[12] + 20.25 * mk[13]) + Gs[1] * (202.5 * mk[2] - 141.75 * mk[4] - 141.75 * mk[5] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]) + Gs[2] * (202.5 * mk[1] - 141.75 * mk[3] - 141.75 * mk[4] + 20.25 * mk[6] + 40.5 * mk[7] + 20.25 * mk[8]) + Gs[4] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] + 20.25 * mk[3] + 40.5 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[35] = v_;
      out[53] = v_;
    }
    {
      const double M_ = -40.5 * m[4] - 20.25 * m[7] + 101.25 * m[8] + 20.25 * m[11] - 20.25 * m[12] - 40.5 * m[13];
      const double K_ = Gs[0] * (-101.25 * mk[4] - 81.0 * mk[7] + 222.75 * mk[8] + 20.25 * mk[11] - 20.25 * mk[12] - 40.5 * mk[13]) + Gs[1] * (-40.5 * mk[2] - 20.25 * mk[4] + 101.25 * mk[5] + 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[9]) + Gs[2] * (-101.25 * mk[1] - 81.0 * mk[3] + 526.5 * mk[4] + 20.25 * mk[6] - 81.0 * mk[7] - 101.25 * mk[8]) + Gs[4] * (-40.5 * mk[0] - 20.25 * mk[1] + 222.75 * mk[2] + 20.25 * mk[3] - 81.0 * mk[4] - 101.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[36] = v_;
      out[63] = v_;
    }
    {
      const double M_ = -40.5 * m[7] + 101.25 * m[11] - 20.25 * m[12] - 40.5 * m[16] - 20.25 * m[17] + 20.25 * m[18];
      const double K_ = Gs[1] * (-101.25 * mk[4] + 526.5 * mk[7] - 81.0 * mk[8] - 101.25 * mk[11] - 81.0 * mk[12] + 20.25 * mk[13]) + Gs[2] * (-101.25 * mk[3] + 222.75 * mk[6] - 81.0 * mk[7] - 40.5 * mk[10] - 20.25 * mk[11] + 20.25 * mk[12]) + Gs[3] * (-40.5 * mk[2] + 222.75 * mk[4] - 20.25 * mk[5] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]) + Gs[4] * (-40.5 * mk[1] + 101.25 * mk[3] - 20.25 * mk[4] - 40.5 * mk[6] - 20.25 * mk[7] + 20.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[37] = v_;
      out[73] = v_;
    }
    {
      const double M_ = -40.5 * m[7] - 20.25 * m[11] + 101.25 * m[12] + 20.25 * m[16] - 20.25 * m[17] - 40.5 * m[18];
      const double K_ = Gs[1] * (-101.25 * mk[4] - 81.0 * mk[7] + 222.75 * mk[8] + 20.25 * mk[11] - 20.25 * mk[12] - 40.5 * mk[13]) + Gs[2] * (-101.25 * mk[3] - 81.0 * mk[6] + 526.5 * mk[7] + 20.25 * mk[10] - 81.0 * mk[11] - 101.25 * mk[12]) + Gs[3] * (-40.5 * mk[2] - 20.25 * mk[4] + 101.25 * mk[5] + 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[9]) + Gs[4] * (-40.5 * mk[1] - 20.25 * mk[3] + 222.75 * mk[4] + 20.25 * mk[6] - 81.0 * mk[7] - 101.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[38] = v_;
      out[83] = v_;
    }
    {
      const double M_ = 243.0 * m[7] - 121.5 * m[11] - 121.5 * m[12];
      const double K_ = Gs[0] * (607.5 * mk[7] - 121.5 * mk[11] - 121.5 * mk[12]) + Gs[1] * (850.5 * mk[4] - 243.0 * mk[7] - 243.0 * mk[8]) + Gs[2] * (607.5 * mk[3] - 121.5 * mk[6] - 121.5 * mk[7]) + Gs[3] * (243.0 * mk[2] - 121.5 * mk[4] - 121.5 * mk[5]) + Gs[4] * (243.0 * mk[1] - 121.5 * mk[3] - 121.5 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[39] = v_;
      out[93] = v_;
    }
    {
      const double M_ = 20.25 * m[3] - 81.0 * m[6] + 40.5 * m[7] + 81.0 * m[10] - 81.0 * m[11] + 20.25 * m[12];
      const double K_ = Gs[0] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[10] - 81.0 * mk[11] + 20.25 * mk[12]) + Gs[1] * (40.5 * mk[1] - 283.5 * mk[3] + 81.0 * mk[4] + 405.0 * mk[6] - 283.5 * mk[7] + 40.5 * mk[8]) + Gs[3] * (20.25 * mk[0] - 202.5 * mk[1] + 40.5 * mk[2] + 506.25 * mk[3] - 202.5 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[44] = v_;
    }
    {
      const double M_ = -40.5 * m[4] + 101.25 * m[7] - 20.25 * m[8] - 40.5 * m[11] - 20.25 * m[12] + 20.25 * m[13];
      const double K_ = Gs[0] * (-101.25 * mk[4] + 222.75 * mk[7] - 81.0 * mk[8] - 40.5 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13]) + Gs[1] * (-101.25 * mk[2] + 526.5 * mk[4] - 81.0 * mk[5] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]) + Gs[2] * (-40.5 * mk[1] + 101.25 * mk[3] - 20.25 * mk[4] - 40.5 * mk[6] - 20.25 * mk[7] + 20.25 * mk[8]) + Gs[4] * (-40.5 * mk[0] + 222.75 * mk[1] - 20.25 * mk[2] - 101.25 * mk[3] - 81.0 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[45] = v_;
      out[54] = v_;
    }
    {
      const double M_ = 20.25 * m[4] - 20.25 * m[7] - 20.25 * m[8] - 40.5 * m[11] + 101.25 * m[12] - 40.5 * m[13];
      const double K_ = Gs[0] * (20.25 * mk[4] - 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[11] + 101.25 * mk[12] - 40.5 * mk[13]) + Gs[1] * (20.25 * mk[2] - 81.0 * mk[4] - 20.25 * mk[5] - 101.25 * mk[7] + 222.75 * mk[8] - 40.5 * mk[9]) + Gs[2] * (20.25 * mk[1] - 20.25 * mk[3] - 81.0 * mk[4] - 40.5 * mk[6] + 222.75 * mk[7] - 101.25 * mk[8]) + Gs[4] * (20.25 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 101.25 * mk[3] + 526.5 * mk[4] - 101.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[46] = v_;
      out[64] = v_;
    }
    {
      const double M_ = 20.25 * m[7] - 81.0 * m[11] + 40.5 * m[12] + 81.0 * m[16] - 81.0 * m[17] + 20.25 * m[18];
      const double K_ = Gs[1] * (20.25 * mk[4] - 141.75 * mk[7] + 40.5 * mk[8] + 202.5 * mk[11] - 141.75 * mk[12] + 20.25 * mk[13]) + Gs[2] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[10] - 81.0 * mk[11] + 20.25 * mk[12]) + Gs[3] * (20.25 * mk[2] - 202.5 * mk[4] + 40.5 * mk[5] + 506.25 * mk[7] - 202.5 * mk[8] + 20.25 * mk[9]) + Gs[4] * (20.25 * mk[1] - 141.75 * mk[3] + 40.5 * mk[4] + 202.5 * mk[6] - 141.75 * mk[7] + 20.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[47] = v_;
      out[74] = v_;
    }
    {
      const double M_ = 20.25 * m[7] - 20.25 * m[11] - 20.25 * m[12] - 40.5 * m[16] + 101.25 * m[17] - 40.5 * m[18];
      const double K_ = Gs[1] * (20.25 * mk[4] - 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[11] + 101.25 * mk[12] - 40.5 * mk[13]) + Gs[2] * (20.25 * mk[3] - 20.25 * mk[6] - 81.0 * mk[7] - 40.5 * mk[10] + 222.75 * mk[11] - 101.25 * mk[12]) + Gs[3] * (20.25 * mk[2] - 81.0 * mk[4] - 20.25 * mk[5] - 101.25 * mk[7] + 222.75 * mk[8] - 40.5 * mk[9]) + Gs[4] * (20.25 * mk[1] - 81.0 * mk[3] - 81.0 * mk[4] - 101.25 * mk[6] + 526.5 * mk[7] - 101.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[48] = v_;
      out[84] = v_;
    }
    {
      const double M_ = -121.5 * m[7] + 243.0 * m[11] - 121.5 * m[12];
      const double K_ = Gs[0] * (-121.5 * mk[7] + 243.0 * mk[11] - 121.5 * mk[12]) + Gs[1] * (-243.0 * mk[4] + 850.5 * mk[7] - 243.0 * mk[8]) + Gs[2] * (-121.5 * mk[3] + 243.0 * mk[6] - 121.5 * mk[7]) + Gs[3] * (-121.5 * mk[2] + 607.5 * mk[4] - 121.5 * mk[5]) + Gs[4] * (-121.5 * mk[1] + 607.5 * mk[3] - 121.5 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[49] = v_;
      out[94] = v_;
    }
    {
      const double M_ = 81.0 * m[5] - 81.0 * m[8] - 81.0 * m[9] + 20.25 * m[12] + 40.5 * m[13] + 20.25 * m[14];
      const double K_ = Gs[0] * (506.25 * mk[5] - 202.5 * mk[8] - 202.5 * mk[9] + 20.25 * mk[12] + 40.5 * mk[13] + 20.25 * mk[14]) + Gs[2] * (405.0 * mk[2] - 283.5 * mk[4] - 283.5 * mk[5] + 40.5 * mk[7] + 81.0 * mk[8] + 40.5 * mk[9]) + Gs[5] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] + 20.25 * mk[3] + 40.5 * mk[4] + 20.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[55] = v_;
    }
    {
      const double M_ = -40.5 * m[5] - 20.25 * m[8] + 101.25 * m[9] + 20.25 * m[12] - 20.25 * m[13] - 40.5 * m[14];
      const double K_ = Gs[0] * (-101.25 * mk[5] - 81.0 * mk[8] + 222.75 * mk[9] + 20.25 * mk[12] - 20.25 * mk[13] - 40.5 * mk[14]) + Gs[2] * (-141.75 * mk[2] - 101.25 * mk[4] + 627.75 * mk[5] + 40.5 * mk[7] - 101.25 * mk[8] - 141.75 * mk[9]) + Gs[5] * (-40.5 * mk[0] - 20.25 * mk[1] + 222.75 * mk[2] + 20.25 * mk[3] - 81.0 * mk[4] - 101.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[56] = v_;
      out[65] = v_;
    }
    {
      const double M_ = -40.5 * m[8] + 101.25 * m[12] - 20.25 * m[13] - 40.5 * m[17] - 20.25 * m[18] + 20.25 * m[19];
      const double K_ = Gs[1] * (-101.25 * mk[5] + 526.5 * mk[8] - 81.0 * mk[9] - 101.25 * mk[12] - 81.0 * mk[13] + 20.25 * mk[14]) + Gs[2] * (-101.25 * mk[4] + 222.75 * mk[7] - 81.0 * mk[8] - 40.5 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13]) + Gs[4] * (-40.5 * mk[2] + 222.75 * mk[4] - 20.25 * mk[5] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]) + Gs[5] * (-40.5 * mk[1] + 101.25 * mk[3] - 20.25 * mk[4] - 40.5 * mk[6] - 20.25 * mk[7] + 20.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[57] = v_;
      out[75] = v_;
    }
    {
      const double M_ = -40.5 * m[8] - 20.25 * m[12] + 101.25 * m[13] + 20.25 * m[17] - 20.25 * m[18] - 40.5 * m[19];
      const double K_ = Gs[1] * (-101.25 * mk[5] - 81.0 * mk[8] + 222.75 * mk[9] + 20.25 * mk[12] - 20.25 * mk[13] - 40.5 * mk[14]) + Gs[2] * (-101.25 * mk[4] - 81.0 * mk[7] + 526.5 * mk[8] + 20.25 * mk[11] - 81.0 * mk[12] - 101.25 * mk[13]) + Gs[4] * (-40.5 * mk[2] - 20.25 * mk[4] + 101.25 * mk[5] + 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[9]) + Gs[5] * (-40.5 * mk[1] - 20.25 * mk[3] + 222.75 * mk[4] + 20.25 * mk[6] - 81.0 * mk[7] - 101.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[58] = v_;
      out[85] = v_;
    }
    {
      const double M_ = 243.0 * m[8] - 121.5 * m[12] - 121.5 * m[13];
      const double K_ = Gs[0] * (607.5 * mk[8] - 121.5 * mk[12] - 121.5 * mk[13]) + Gs[1] * (607.5 * mk[5] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[2] * (850.5 * mk[4] - 243.0 * mk[7] - 243.0 * mk[8]) + Gs[4] * (243.0 * mk[2] - 121.5 * mk[4] - 121.5 * mk[5]) + Gs[5] * (243.0 * mk[1] - 121.5 * mk[3] - 121.5 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[59] = v_;
      out[95] = v_;
    }
    {
      const double M_ = 20.25 * m[5] + 40.5 * m[8] - 81.0 * m[9] + 20.25 * m[12] - 81.0 * m[13] + 81.0 * m[14];
      const double K_ = Gs[0] * (20.25 * mk[5] + 40.5 * mk[8] - 81.0 * mk[9] + 20.25 * mk[12] - 81.0 * mk[13] + 81.0 * mk[14]) + Gs[2] * (40.5 * mk[2] + 81.0 * mk[4] - 283.5 * mk[5] + 40.5 * mk[7] - 283.5 * mk[8] + 405.0 * mk[9]) + Gs[5] * (20.25 * mk[0] + 40.5 * mk[1] - 202.5 * mk[2] + 20.25 * mk[3] - 202.5 * mk[4] + 506.25 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[66] = v_;
    }
    {
      const double M_ = 20.25 * m[8] - 20.25 * m[12] - 20.25 * m[13] - 40.5 * m[17] + 101.25 * m[18] - 40.5 * m[19];
      const double K_ = Gs[1] * (20.25 * mk[5] - 81.0 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] + 222.75 * mk[13] - 40.5 * mk[14]) + Gs[2] * (20.25 * mk[4] - 20.25 * mk[7] - 20.25 * mk[8] - 40.5 * mk[11] + 101.25 * mk[12] - 40.5 * mk[13]) + Gs[4] * (20.25 * mk[2] - 81.0 * mk[4] - 81.0 * mk[5] - 101.25 * mk[7] + 526.5 * mk[8] - 101.25 * mk[9]) + Gs[5] * (20.25 * mk[1] - 20.25 * mk[3] - 81.0 * mk[4] - 40.5 * mk[6] + 222.75 * mk[7] - 101.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[67] = v_;
      out[76] = v_;
    }
    {
      const double M_ = 20.25 * m[8] + 40.5 * m[12] - 81.0 * m[13] + 20.25 * m[17] - 81.0 * m[18] + 81.0 * m[19];
      const double K_ = Gs[1] * (20.25 * mk[5] + 40.5 * mk[8] - 81.0 * mk[9] + 20.25 * mk[12] - 81.0 * mk[13] + 81.0 * mk[14]) + Gs[2] * (20.25 * mk[4] + 40.5 * mk[7] - 141.75 * mk[8] + 20.25 * mk[11] - 141.75 * mk[12] + 202.5 * mk[13]) + Gs[4] * (20.25 * mk[2] + 40.5 * mk[4] - 141.75 * mk[5] + 20.25 * mk[7] - 141.75 * mk[8] + 202.5 * mk[9]) + Gs[5] * (20.25 * mk[1] + 40.5 * mk[3] - 202.5 * mk[4] + 20.25 * mk[6] - 202.5 * mk[7] + 506.25 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[68] = v_;
      out[86] = v_;
    }
    {
      const double M_ = -121.5 * m[8] - 121.5 * m[12] + 243.0 * m[13];
      const double K_ = Gs[0] * (-121.5 * mk[8] - 121.5 * mk[12] + 243.0 * mk[13]) + Gs[1] * (-121.5 * mk[5] - 121.5 * mk[8] + 243.0 * mk[9]) + Gs[2] * (-243.0 * mk[4] - 243.0 * mk[7] + 850.5 * mk[8]) + Gs[4] * (-121.5 * mk[2] - 121.5 * mk[4] + 607.5 * mk[5]) + Gs[5] * (-121.5 * mk[1] - 121.5 * mk[3] + 607.5 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[69] = v_;
      out[96] = v_;
    }
    {
      const double M_ = 20.25 * m[12] - 81.0 * m[17] + 40.5 * m[18] + 81.0 * m[23] - 81.0 * m[24] + 20.25 * m[25];
      const double K_ = Gs[3] * (20.25 * mk[5] - 202.5 * mk[8] + 40.5 * mk[9] + 506.25 * mk[12] - 202.5 * mk[13] + 20.25 * mk[14]) + Gs[4] * (40.5 * mk[4] - 283.5 * mk[7] + 81.0 * mk[8] + 405.0 * mk[11] - 283.5 * mk[12] + 40.5 * mk[13]) + Gs[5] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[10] - 81.0 * mk[11] + 20.25 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[77] = v_;
    }
    {
      const double M_ = 20.25 * m[12] - 20.25 * m[17] - 20.25 * m[18] - 40.5 * m[23] + 101.25 * m[24] - 40.5 * m[25];
      const double K_ = Gs[3] * (20.25 * mk[5] - 81.0 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] + 222.75 * mk[13] - 40.5 * mk[14]) + Gs[4] * (40.5 * mk[4] - 101.25 * mk[7] - 101.25 * mk[8] - 141.75 * mk[11] + 627.75 * mk[12] - 141.75 * mk[13]) + Gs[5] * (20.25 * mk[3] - 20.25 * mk[6] - 81.0 * mk[7] - 40.5 * mk[10] + 222.75 * mk[11] - 101.25 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[78] = v_;
      out[87] = v_;
    }
    {
      const double M_ = -121.5 * m[12] + 243.0 * m[17] - 121.5 * m[18];
      const double K_ = Gs[1] * (-121.5 * mk[8] + 607.5 * mk[12] - 121.5 * mk[13]) + Gs[2] * (-121.5 * mk[7] + 243.0 * mk[11] - 121.5 * mk[12]) + Gs[3] * (-121.5 * mk[5] + 607.5 * mk[8] - 121.5 * mk[9]) + Gs[4] * (-243.0 * mk[4] + 850.5 * mk[7] - 243.0 * mk[8]) + Gs[5] * (-121.5 * mk[3] + 243.0 * mk[6] - 121.5 * mk[7]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[79] = v_;
      out[97] = v_;
    }
    {
      const double M_ = 20.25 * m[12] + 40.5 * m[17] - 81.0 * m[18] + 20.25 * m[23] - 81.0 * m[24] + 81.0 * m[25];
      const double K_ = Gs[3] * (20.25 * mk[5] + 40.5 * mk[8] - 81.0 * mk[9] + 20.25 * mk[12] - 81.0 * mk[13] + 81.0 * mk[14]) + Gs[4] * (40.5 * mk[4] + 81.0 * mk[7] - 283.5 * mk[8] + 40.5 * mk[11] - 283.5 * mk[12] + 405.0 * mk[13]) + Gs[5] * (20.25 * mk[3] + 40.5 * mk[6] - 202.5 * mk[7] + 20.25 * mk[10] - 202.5 * mk[11] + 506.25 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[88] = v_;
    }
    {
      const double M_ = -121.5 * m[12] - 121.5 * m[17] + 243.0 * m[18];
      const double K_ = Gs[1] * (-121.5 * mk[8] - 121.5 * mk[12] + 243.0 * mk[13]) + Gs[2] * (-121.5 * mk[7] - 121.5 * mk[11] + 607.5 * mk[12]) + Gs[3] * (-121.5 * mk[5] - 121.5 * mk[8] + 243.0 * mk[9]) + Gs[4] * (-243.0 * mk[4] - 243.0 * mk[7] + 850.5 * mk[8]) + Gs[5] * (-121.5 * mk[3] - 121.5 * mk[6] + 607.5 * mk[7]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[89] = v_;
      out[98] = v_;
    }
    {
      const double M_ = 729.0 * m[12];
      const double K_ = Gs[0] * (729.0 * mk[12]) + Gs[1] * (1458.0 * mk[8]) + Gs[2] * (1458.0 * mk[7]) + Gs[3] * (729.0 * mk[5]) + Gs[4] * (1458.0 * mk[4]) + Gs[5] * (729.0 * mk[3]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[99] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + 0.5 * m[1] + 0.5 * m[2] - 3.5 * m[3] - 7.0 * m[4] - 3.5 * m[5] - 3.5 * m[6] - 10.5 * m[7] - 10.5 * m[8] - 3.5 * m[9] + 0.5 * m[10] + 2.0 * m[11] + 3.0 * m[12] + 2.0 * m[13] + 0.5 * m[14] + m[15] + 5.0 * m[16] + 10.0 * m[17] + 10.0 * m[18] + 5.0 * m[19] + m[20]));
    out[1] = (T)(s * (m[1] + 0.5 * m[3] + 5.0 * m[4] - 3.5 * m[6] + 2.0 * m[7] + 10.0 * m[8] - 3.5 * m[10] - 10.5 * m[11] + 3.0 * m[12] + 10.0 * m[13] + 0.5 * m[15] - 7.0 * m[16] - 10.5 * m[17] + 2.0 * m[18] + 5.0 * m[19] + m[21] + 0.5 * m[22] - 3.5 * m[23] - 3.5 * m[24] + 0.5 * m[25] + m[26]));
    out[2] = (T)(s * (m[2] + 5.0 * m[4] + 0.5 * m[5] + 10.0 * m[7] + 2.0 * m[8] - 3.5 * m[9] + 10.0 * m[11] + 3.0 * m[12] - 10.5 * m[13] - 3.5 * m[14] + 5.0 * m[16] + 2.0 * m[17] - 10.5 * m[18] - 7.0 * m[19] + 0.5 * m[20] + m[22] + 0.5 * m[23] - 3.5 * m[24] - 3.5 * m[25] + 0.5 * m[26] + m[27]));
    out[3] = (T)(s * (9.0 * m[1] + 22.5 * m[3] + 22.5 * m[4] + 13.5 * m[6] + 27.0 * m[7] + 13.5 * m[8] - 4.5 * m[10] - 13.5 * m[11] - 13.5 * m[12] - 4.5 * m[13] - 4.5 * m[15] - 18.0 * m[16] - 27.0 * m[17] - 18.0 * m[18] - 4.5 * m[19]));
    out[4] = (T)(s * (-4.5 * m[1] - 4.5 * m[3] - 18.0 * m[4] + 13.5 * m[6] - 13.5 * m[7] - 27.0 * m[8] + 22.5 * m[10] + 27.0 * m[11] - 13.5 * m[12] - 18.0 * m[13] + 9.0 * m[15] + 22.5 * m[16] + 13.5 * m[17] - 4.5 * m[18] - 4.5 * m[19]));
    out[5] = (T)(s * (9.0 * m[2] + 22.5 * m[4] + 22.5 * m[5] + 13.5 * m[7] + 27.0 * m[8] + 13.5 * m[9] - 4.5 * m[11] - 13.5 * m[12] - 13.5 * m[13] - 4.5 * m[14] - 4.5 * m[16] - 18.0 * m[17] - 27.0 * m[18] - 18.0 * m[19] - 4.5 * m[20]));
    out[6] = (T)(s * (-4.5 * m[2] - 18.0 * m[4] - 4.5 * m[5] - 27.0 * m[7] - 13.5 * m[8] + 13.5 * m[9] - 18.0 * m[11] - 13.5 * m[12] + 27.0 * m[13] + 22.5 * m[14] - 4.5 * m[16] - 4.5 * m[17] + 13.5 * m[18] + 22.5 * m[19] + 9.0 * m[20]));
    out[7] = (T)(s * (-4.5 * m[4] - 4.5 * m[7] - 18.0 * m[8] + 13.5 * m[11] - 13.5 * m[12] - 27.0 * m[13] + 22.5 * m[16] + 27.0 * m[17] - 13.5 * m[18] - 18.0 * m[19] + 9.0 * m[22] + 22.5 * m[23] + 13.5 * m[24] - 4.5 * m[25] - 4.5 * m[26]));
    out[8] = (T)(s * (-4.5 * m[4] - 18.0 * m[7] - 4.5 * m[8] - 27.0 * m[11] - 13.5 * m[12] + 13.5 * m[13] - 18.0 * m[16] - 13.5 * m[17] + 27.0 * m[18] + 22.5 * m[19] - 4.5 * m[22] - 4.5 * m[23] + 13.5 * m[24] + 22.5 * m[25] + 9.0 * m[26]));
    out[9] = (T)(s * (27.0 * m[4] + 81.0 * m[7] + 81.0 * m[8] + 81.0 * m[11] + 162.0 * m[12] + 81.0 * m[13] + 27.0 * m[16] + 81.0 * m[17] + 81.0 * m[18] + 27.0 * m[19]));
  }
};  // 1459 coefficient terms
template <>
struct Moments<3, 1> {
  static constexpr int NM = 10;  // degree-2 moments
  static constexpr int NK = 1;  // degree-0 moments
  static constexpr int NQ = 4;  // degree-1 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    {
      const double wb = w * l[0];
      m[0] = fma(wb, l[0], m[0]);
      m[1] = fma(wb, l[1], m[1]);
      m[2] = fma(wb, l[2], m[2]);
      m[3] = fma(wb, l[3], m[3]);
    }
    {
      const double wb = w * l[1];
      m[4] = fma(wb, l[1], m[4]);
      m[5] = fma(wb, l[2], m[5]);
      m[6] = fma(wb, l[3], m[6]);
    }
    {
      const double wb = w * l[2];
      m[7] = fma(wb, l[2], m[7]);
      m[8] = fma(wb, l[3], m[8]);
    }
    {
      const double wb = w * l[3];
      m[9] = fma(wb, l[3], m[9]);
    }
  }
  // h = (w - <z, v>) / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_first(const double *y, double w, const double *v, double *h) {
    h[9] = w;
    h[3] = fma(y[0], h[9], -v[0]);
    h[6] = fma(y[1], h[9], -v[1]);
    h[8] = fma(y[2], h[9], -v[2]);
    h[0] = y[0] * h[3];
    h[1] = fma(y[1], h[3], y[0] * h[6]);
    h[2] = fma(y[2], h[3], y[0] * h[8]);
    h[4] = y[1] * h[6];
    h[5] = fma(y[2], h[6], y[1] * h[8]);
    h[7] = y[2] * h[8];
  }
  // h <- h / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_step(const double *y, double *h) {
    h[3] = fma(y[0], h[9], h[3]);
    h[6] = fma(y[1], h[9], h[6]);
    h[8] = fma(y[2], h[9], h[8]);
    h[0] = fma(y[0], h[3], h[0]);
    h[1] = fma(y[1], h[3], fma(y[0], h[6], h[1]));
    h[2] = fma(y[2], h[3], fma(y[0], h[8], h[2]));
    h[4] = fma(y[1], h[6], h[4]);
    h[5] = fma(y[2], h[6], fma(y[1], h[8], h[5]));
    h[7] = fma(y[2], h[8], h[7]);
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.016666666666666666 - m[0];
    m[1] = 0.008333333333333333 - m[1];
    m[2] = 0.008333333333333333 - m[2];
    m[3] = 0.008333333333333333 - m[3];
    m[4] = 0.016666666666666666 - m[4];
    m[5] = 0.008333333333333333 - m[5];
    m[6] = 0.008333333333333333 - m[6];
    m[7] = 0.016666666666666666 - m[7];
    m[8] = 0.008333333333333333 - m[8];
    m[9] = 0.016666666666666666 - m[9];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + 2.0 * m[3] + m[4] + 2.0 * m[5] + 2.0 * m[6] + m[7] + 2.0 * m[8] + m[9];
  }
  static constexpr int NH = 4;  // h: coefficients of H_1 .. H_1
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/2))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    h[2] = h[2] + l[2];
    h[3] = h[3] + l[3];
    m[0] = fma(l[0], h[0], m[0]);
    m[1] = fma(l[1], h[0], fma(l[0], h[1], m[1]));
    m[2] = fma(l[2], h[0], fma(l[0], h[2], m[2]));
    m[3] = fma(l[3], h[0], fma(l[0], h[3], m[3]));
    m[4] = fma(l[1], h[1], m[4]);
    m[5] = fma(l[2], h[1], fma(l[1], h[2], m[5]));
    m[6] = fma(l[3], h[1], fma(l[1], h[3], m[6]));
    m[7] = fma(l[2], h[2], m[7]);
    m[8] = fma(l[3], h[2], fma(l[2], h[3], m[8]));
    m[9] = fma(l[3], h[3], m[9]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 2.0;
    m[4] *= 2.0;
    m[7] *= 2.0;
    m[9] *= 2.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 10;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0];
      const double K_ = Gs[0] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1];
      const double K_ = Gs[1] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[4] = v_;
    }
    {
      const double M_ = m[2];
      const double K_ = Gs[2] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[2] = v_;
      out[8] = v_;
    }
    {
      const double M_ = m[3];
      const double K_ = Gs[3] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[3] = v_;
      out[12] = v_;
    }
    {
      const double M_ = m[4];
      const double K_ = Gs[4] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[5] = v_;
    }
    {
      const double M_ = m[5];
      const double K_ = Gs[5] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[6] = v_;
      out[9] = v_;
    }
    {
      const double M_ = m[6];
      const double K_ = Gs[6] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[7] = v_;
      out[13] = v_;
    }
    {
      const double M_ = m[7];
      const double K_ = Gs[7] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[10] = v_;
    }
    {
      const double M_ = m[8];
      const double K_ = Gs[8] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[11] = v_;
      out[14] = v_;
    }
    {
      const double M_ = m[9];
      const double K_ = Gs[9] * (mk[0]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[15] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1] + m[2] + m[3]));
    out[1] = (T)(s * (m[1] + m[4] + m[5] + m[6]));
    out[2] = (T)(s * (m[2] + m[5] + m[7] + m[8]));
    out[3] = (T)(s * (m[3] + m[6] + m[8] + m[9]));
  }
};  // 20 coefficient terms
template <>
struct Moments<3, 2> {
  static constexpr int NM = 35;  // degree-4 moments
  static constexpr int NK = 10;  // degree-2 moments
  static constexpr int NQ = 10;  // degree-2 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[2] * l[0];
    const double t3 = l[3] * l[0];
    const double t4 = l[1] * l[1];
    const double t5 = l[2] * l[1];
    const double t6 = l[3] * l[1];
    const double t7 = l[2] * l[2];
    const double t8 = l[3] * l[2];
    const double t9 = l[3] * l[3];
    {
      const double wb = w * t0;
      m[0] = fma(wb, t0, m[0]);
      m[1] = fma(wb, t1, m[1]);
      m[2] = fma(wb, t2, m[2]);
      m[3] = fma(wb, t3, m[3]);
      m[4] = fma(wb, t4, m[4]);
      m[5] = fma(wb, t5, m[5]);
      m[6] = fma(wb, t6, m[6]);
      m[7] = fma(wb, t7, m[7]);
      m[8] = fma(wb, t8, m[8]);
      m[9] = fma(wb, t9, m[9]);
    }
    {
      const double wb = w * t1;
      m[10] = fma(wb, t4, m[10]);
      m[11] = fma(wb, t5, m[11]);
      m[12] = fma(wb, t6, m[12]);
      m[13] = fma(wb, t7, m[13]);
      m[14] = fma(wb, t8, m[14]);
      m[15] = fma(wb, t9, m[15]);
    }
    {
      const double wb = w * t2;
      m[16] = fma(wb, t7, m[16]);
      m[17] = fma(wb, t8, m[17]);
      m[18] = fma(wb, t9, m[18]);
    }
    {
      const double wb = w * t3;
      m[19] = fma(wb, t9, m[19]);
    }
    {
      const double wb = w * t4;
      m[20] = fma(wb, t4, m[20]);
      m[21] = fma(wb, t5, m[21]);
      m[22] = fma(wb, t6, m[22]);
      m[23] = fma(wb, t7, m[23]);
      m[24] = fma(wb, t8, m[24]);
      m[25] = fma(wb, t9, m[25]);
    }
    {
      const double wb = w * t5;
      m[26] = fma(wb, t7, m[26]);
      m[27] = fma(wb, t8, m[27]);
      m[28] = fma(wb, t9, m[28]);
    }
    {
      const double wb = w * t6;
      m[29] = fma(wb, t9, m[29]);
    }
    {
      const double wb = w * t7;
      m[30] = fma(wb, t7, m[30]);
      m[31] = fma(wb, t8, m[31]);
      m[32] = fma(wb, t9, m[32]);
    }
    {
      const double wb = w * t8;
      m[33] = fma(wb, t9, m[33]);
    }
    {
      const double wb = w * t9;
      m[34] = fma(wb, t9, m[34]);
    }
  }
  // h = (w - <z, v>) / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_first(const double *y, double w, const double *v, double *h) {
    h[34] = w;
    h[19] = fma(y[0], h[34], -v[0]);
    h[29] = fma(y[1], h[34], -v[1]);
    h[33] = fma(y[2], h[34], -v[2]);
    h[9] = y[0] * h[19];
    h[15] = fma(y[1], h[19], y[0] * h[29]);
    h[18] = fma(y[2], h[19], y[0] * h[33]);
    h[25] = y[1] * h[29];
    h[28] = fma(y[2], h[29], y[1] * h[33]);
    h[32] = y[2] * h[33];
    h[3] = y[0] * h[9];
    h[6] = fma(y[1], h[9], y[0] * h[15]);
    h[8] = fma(y[2], h[9], y[0] * h[18]);
    h[12] = fma(y[1], h[15], y[0] * h[25]);
    h[14] = fma(y[2], h[15], fma(y[1], h[18], y[0] * h[28]));
    h[17] = fma(y[2], h[18], y[0] * h[32]);
    h[22] = y[1] * h[25];
    h[24] = fma(y[2], h[25], y[1] * h[28]);
    h[27] = fma(y[2], h[28], y[1] * h[32]);
    h[31] = y[2] * h[32];
    h[0] = y[0] * h[3];
    h[1] = fma(y[1], h[3], y[0] * h[6]);
    h[2] = fma(y[2], h[3], y[0] * h[8]);
    h[4] = fma(y[1], h[6], y[0] * h[12]);
    h[5] = fma(y[2], h[6], fma(y[1], h[8], y[0] * h[14]));
    h[7] = fma(y[2], h[8], y[0] * h[17]);
    h[10] = fma(y[1], h[12], y[0] * h[22]);
    h[11] = fma(y[2], h[12], fma(y[1], h[14], y[0] * h[24]));
    h[13] = fma(y[2], h[14], fma(y[1], h[17], y[0] * h[27]));
    h[16] = fma(y[2], h[17], y[0] * h[31]);
    h[20] = y[1] * h[22];
    h[21] = fma(y[2], h[22], y[1] * h[24]);
    h[23] = fma(y[2], h[24], y[1] * h[27]);
    h[26] = fma(y[2], h[27], y[1] * h[31]);
    h[30] = y[2] * h[31];
  }
  // h <- h / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_step(const double *y, double *h) {
    h[19] = fma(y[0], h[34], h[19]);
    h[29] = fma(y[1], h[34], h[29]);
    h[33] = fma(y[2], h[34], h[33]);
    h[9] = fma(y[0], h[19], h[9]);
    h[15] = fma(y[1], h[19], fma(y[0], h[29], h[15]));
    h[18] = fma(y[2], h[19], fma(y[0], h[33], h[18]));
    h[25] = fma(y[1], h[29], h[25]);
    h[28] = fma(y[2], h[29], fma(y[1], h[33], h[28]));
    h[32] = fma(y[2], h[33], h[32]);
    h[3] = fma(y[0], h[9], h[3]);
    h[6] = fma(y[1], h[9], fma(y[0], h[15], h[6]));
    h[8] = fma(y[2], h[9], fma(y[0], h[18], h[8]));
    h[12] = fma(y[1], h[15], fma(y[0], h[25], h[12]));
    h[14] = fma(y[2], h[15], fma(y[1], h[18], fma(y[0], h[28], h[14])));
    h[17] = fma(y[2], h[18], fma(y[0], h[32], h[17]));
    h[22] = fma(y[1], h[25], h[22]);
    h[24] = fma(y[2], h[25], fma(y[1], h[28], h[24]));
    h[27] = fma(y[2], h[28], fma(y[1], h[32], h[27]));
    h[31] = fma(y[2], h[32], h[31]);
    h[0] = fma(y[0], h[3], h[0]);
    h[1] = fma(y[1], h[3], fma(y[0], h[6], h[1]));
    h[2] = fma(y[2], h[3], fma(y[0], h[8], h[2]));
    h[4] = fma(y[1], h[6], fma(y[0], h[12], h[4]));
    h[5] = fma(y[2], h[6], fma(y[1], h[8], fma(y[0], h[14], h[5])));
    h[7] = fma(y[2], h[8], fma(y[0], h[17], h[7]));
    h[10] = fma(y[1], h[12], fma(y[0], h[22], h[10]));
    h[11] = fma(y[2], h[12], fma(y[1], h[14], fma(y[0], h[24], h[11])));
    h[13] = fma(y[2], h[14], fma(y[1], h[17], fma(y[0], h[27], h[13])));
    h[16] = fma(y[2], h[17], fma(y[0], h[31], h[16]));
    h[20] = fma(y[1], h[22], h[20]);
    h[21] = fma(y[2], h[22], fma(y[1], h[24], h[21]));
    h[23] = fma(y[2], h[24], fma(y[1], h[27], h[23]));
    h[26] = fma(y[2], h[27], fma(y[1], h[31], h[26]));
    h[30] = fma(y[2], h[31], h[30]);
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.004761904761904762 - m[0];
    m[1] = 0.0011904761904761906 - m[1];
    m[2] = 0.0011904761904761906 - m[2];
    m[3] = 0.0011904761904761906 - m[3];
    m[4] = 0.0007936507936507937 - m[4];
    m[5] = 0.0003968253968253968 - m[5];
    m[6] = 0.0003968253968253968 - m[6];
    m[7] = 0.0007936507936507937 - m[7];
    m[8] = 0.0003968253968253968 - m[8];
    m[9] = 0.0007936507936507937 - m[9];
    m[10] = 0.0011904761904761906 - m[10];
    m[11] = 0.0003968253968253968 - m[11];
    m[12] = 0.0003968253968253968 - m[12];
    m[13] = 0.0003968253968253968 - m[13];
    m[14] = 0.0001984126984126984 - m[14];
    m[15] = 0.0003968253968253968 - m[15];
    m[16] = 0.0011904761904761906 - m[16];
    m[17] = 0.0003968253968253968 - m[17];
    m[18] = 0.0003968253968253968 - m[18];
    m[19] = 0.0011904761904761906 - m[19];
    m[20] = 0.004761904761904762 - m[20];
    m[21] = 0.0011904761904761906 - m[21];
    m[22] = 0.0011904761904761906 - m[22];
    m[23] = 0.0007936507936507937 - m[23];
    m[24] = 0.0003968253968253968 - m[24];
    m[25] = 0.0007936507936507937 - m[25];
    m[26] = 0.0011904761904761906 - m[26];
    m[27] = 0.0003968253968253968 - m[27];
    m[28] = 0.0003968253968253968 - m[28];
    m[29] = 0.0011904761904761906 - m[29];
    m[30] = 0.004761904761904762 - m[30];
    m[31] = 0.0011904761904761906 - m[31];
    m[32] = 0.0007936507936507937 - m[32];
    m[33] = 0.0011904761904761906 - m[33];
    m[34] = 0.004761904761904762 - m[34];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + 2.0 * m[3] + m[4] + 2.0 * m[5] + 2.0 * m[6] + m[7] + 2.0 * m[8] + m[9];
    mk[1] = m[1] + 2.0 * m[4] + 2.0 * m[5] + 2.0 * m[6] + m[10] + 2.0 * m[11] + 2.0 * m[12] + m[13] + 2.0 * m[14] + m[15];
    mk[2] = m[2] + 2.0 * m[5] + 2.0 * m[7] + 2.0 * m[8] + m[11] + 2.0 * m[13] + 2.0 * m[14] + m[16] + 2.0 * m[17] + m[18];
    mk[3] = m[3] + 2.0 * m[6] + 2.0 * m[8] + 2.0 * m[9] + m[12] + 2.0 * m[14] + 2.0 * m[15] + m[17] + 2.0 * m[18] + m[19];
    mk[4] = m[4] + 2.0 * m[10] + 2.0 * m[11] + 2.0 * m[12] + m[20] + 2.0 * m[21] + 2.0 * m[22] + m[23] + 2.0 * m[24] + m[25];
    mk[5] = m[5] + 2.0 * m[11] + 2.0 * m[13] + 2.0 * m[14] + m[21] + 2.0 * m[23] + 2.0 * m[24] + m[26] + 2.0 * m[27] + m[28];
    mk[6] = m[6] + 2.0 * m[12] + 2.0 * m[14] + 2.0 * m[15] + m[22] + 2.0 * m[24] + 2.0 * m[25] + m[27] + 2.0 * m[28] + m[29];
    mk[7] = m[7] + 2.0 * m[13] + 2.0 * m[16] + 2.0 * m[17] + m[23] + 2.0 * m[26] + 2.0 * m[27] + m[30] + 2.0 * m[31] + m[32];
    mk[8] = m[8] + 2.0 * m[14] + 2.0 * m[17] + 2.0 * m[18] + m[24] + 2.0 * m[27] + 2.0 * m[28] + m[31] + 2.0 * m[32] + m[33];
    mk[9] = m[9] + 2.0 * m[15] + 2.0 * m[18] + 2.0 * m[19] + m[25] + 2.0 * m[28] + 2.0 * m[29] + m[32] + 2.0 * m[33] + m[34];
  }
  static constexpr int NH = 34;  // h: coefficients of H_1 .. H_3
  // one vertex of the complete homogeneous recursion (l: barycentrics scaled by s^(1/4))
  XG_DEV static void hstep(const double *l, double *h, double *m) {
    h[0] = h[0] + l[0];
    h[1] = h[1] + l[1];
    h[2] = h[2] + l[2];
    h[3] = h[3] + l[3];
    h[4] = fma(l[0], h[0], h[4]);
    h[5] = fma(l[1], h[0], fma(l[0], h[1], h[5]));
    h[6] = fma(l[2], h[0], fma(l[0], h[2], h[6]));
    h[7] = fma(l[3], h[0], fma(l[0], h[3], h[7]));
    h[8] = fma(l[1], h[1], h[8]);
    h[9] = fma(l[2], h[1], fma(l[1], h[2], h[9]));
    h[10] = fma(l[3], h[1], fma(l[1], h[3], h[10]));
    h[11] = fma(l[2], h[2], h[11]);
    h[12] = fma(l[3], h[2], fma(l[2], h[3], h[12]));
    h[13] = fma(l[3], h[3], h[13]);
    h[14] = fma(l[0], h[4], h[14]);
    h[15] = fma(l[1], h[4], fma(l[0], h[5], h[15]));
    h[16] = fma(l[2], h[4], fma(l[0], h[6], h[16]));
    h[17] = fma(l[3], h[4], fma(l[0], h[7], h[17]));
    h[18] = fma(l[1], h[5], fma(l[0], h[8], h[18]));
    h[19] = fma(l[2], h[5], fma(l[1], h[6], fma(l[0], h[9], h[19])));
    h[20] = fma(l[3], h[5], fma(l[1], h[7], fma(l[0], h[10], h[20])));
    h[21] = fma(l[2], h[6], fma(l[0], h[11], h[21]));
    h[22] = fma(l[3], h[6], fma(l[2], h[7], fma(l[0], h[12], h[22])));
    h[23] = fma(l[3], h[7], fma(l[0], h[13], h[23]));
    h[24] = fma(l[1], h[8], h[24]);
    h[25] = fma(l[2], h[8], fma(l[1], h[9], h[25]));
    h[26] = fma(l[3], h[8], fma(l[1], h[10], h[26]));
    h[27] = fma(l[2], h[9], fma(l[1], h[11], h[27]));
    h[28] = fma(l[3], h[9], fma(l[2], h[10], fma(l[1], h[12], h[28])));
    h[29] = fma(l[3], h[10], fma(l[1], h[13], h[29]));
    h[30] = fma(l[2], h[11], h[30]);
    h[31] = fma(l[3], h[11], fma(l[2], h[12], h[31]));
    h[32] = fma(l[3], h[12], fma(l[2], h[13], h[32]));
    h[33] = fma(l[3], h[13], h[33]);
    m[0] = fma(l[0], h[14], m[0]);
    m[1] = fma(l[1], h[14], fma(l[0], h[15], m[1]));
    m[2] = fma(l[2], h[14], fma(l[0], h[16], m[2]));
    m[3] = fma(l[3], h[14], fma(l[0], h[17], m[3]));
    m[4] = fma(l[1], h[15], fma(l[0], h[18], m[4]));
    m[5] = fma(l[2], h[15], fma(l[1], h[16], fma(l[0], h[19], m[5])));
    m[6] = fma(l[3], h[15], fma(l[1], h[17], fma(l[0], h[20], m[6])));
    m[7] = fma(l[2], h[16], fma(l[0], h[21], m[7]));
    m[8] = fma(l[3], h[16], fma(l[2], h[17], fma(l[0], h[22], m[8])));
    m[9] = fma(l[3], h[17], fma(l[0], h[23], m[9]));
    m[10] = fma(l[1], h[18], fma(l[0], h[24], m[10]));
    m[11] = fma(l[2], h[18], fma(l[1], h[19], fma(l[0], h[25], m[11])));
    m[12] = fma(l[3], h[18], fma(l[1], h[20], fma(l[0], h[26], m[12])));
    m[13] = fma(l[2], h[19], fma(l[1], h[21], fma(l[0], h[27], m[13])));
    m[14] = fma(l[3], h[19], fma(l[2], h[20], fma(l[1], h[22], fma(l[0], h[28], m[14]))));
    m[15] = fma(l[3], h[20], fma(l[1], h[23], fma(l[0], h[29], m[15])));
    m[16] = fma(l[2], h[21], fma(l[0], h[30], m[16]));
    m[17] = fma(l[3], h[21], fma(l[2], h[22], fma(l[0], h[31], m[17])));
    m[18] = fma(l[3], h[22], fma(l[2], h[23], fma(l[0], h[32], m[18])));
    m[19] = fma(l[3], h[23], fma(l[0], h[33], m[19]));
    m[20] = fma(l[1], h[24], m[20]);
    m[21] = fma(l[2], h[24], fma(l[1], h[25], m[21]));
    m[22] = fma(l[3], h[24], fma(l[1], h[26], m[22]));
    m[23] = fma(l[2], h[25], fma(l[1], h[27], m[23]));
    m[24] = fma(l[3], h[25], fma(l[2], h[26], fma(l[1], h[28], m[24])));
    m[25] = fma(l[3], h[26], fma(l[1], h[29], m[25]));
    m[26] = fma(l[2], h[27], fma(l[1], h[30], m[26]));
    m[27] = fma(l[3], h[27], fma(l[2], h[28], fma(l[1], h[31], m[27])));
    m[28] = fma(l[3], h[28], fma(l[2], h[29], fma(l[1], h[32], m[28])));
    m[29] = fma(l[3], h[29], fma(l[1], h[33], m[29]));
    m[30] = fma(l[2], h[30], m[30]);
    m[31] = fma(l[3], h[30], fma(l[2], h[31], m[31]));
    m[32] = fma(l[3], h[31], fma(l[2], h[32], m[32]));
    m[33] = fma(l[3], h[32], fma(l[2], h[33], m[33]));
    m[34] = fma(l[3], h[33], m[34]);
  }
  XG_DEV static void hfinish(double *m) {
    m[0] *= 24.0;
    m[1] *= 6.0;
    m[2] *= 6.0;
    m[3] *= 6.0;
    m[4] *= 4.0;
    m[5] *= 2.0;
    m[6] *= 2.0;
    m[7] *= 4.0;
    m[8] *= 2.0;
    m[9] *= 4.0;
    m[10] *= 6.0;
    m[11] *= 2.0;
    m[12] *= 2.0;
    m[13] *= 2.0;
    m[15] *= 2.0;
    m[16] *= 6.0;
    m[17] *= 2.0;
    m[18] *= 2.0;
    m[19] *= 6.0;
    m[20] *= 24.0;
    m[21] *= 6.0;
    m[22] *= 6.0;
    m[23] *= 4.0;
    m[24] *= 2.0;
    m[25] *= 4.0;
    m[26] *= 6.0;
    m[27] *= 2.0;
    m[28] *= 2.0;
    m[29] *= 6.0;
    m[30] *= 24.0;
    m[31] *= 6.0;
    m[32] *= 4.0;
    m[33] *= 6.0;
    m[34] *= 24.0;
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 10;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    const double sm2_ = 2.0 * sm;
    const double sm4_ = 4.0 * sm;
    const double sk4_ = 4.0 * sk;
    const double Gd1 = 2.0 * Gs[1];
    const double Gd2 = 2.0 * Gs[2];
    const double Gd3 = 2.0 * Gs[3];
    const double Gd5 = 2.0 * Gs[5];
    const double Gd6 = 2.0 * Gs[6];
    const double Gd8 = 2.0 * Gs[8];
    // A = sm M^B + sk K^B (Bernstein basis, upper triangle)
    const double A0_0 = sm * m[0] + sk4_ * (Gs[0] * mk[0]);
    const double A0_1 = sm2_ * m[1] + sk4_ * (Gs[0] * mk[1] + Gs[1] * mk[0]);
    const double A0_2 = sm2_ * m[2] + sk4_ * (Gs[0] * mk[2] + Gs[2] * mk[0]);
    const double A0_3 = sm2_ * m[3] + sk4_ * (Gs[0] * mk[3] + Gs[3] * mk[0]);
    const double A0_4 = sm * m[4] + sk4_ * (Gs[1] * mk[1]);
    const double A0_5 = sm2_ * m[5] + sk4_ * (Gs[1] * mk[2] + Gs[2] * mk[1]);
    const double A0_6 = sm2_ * m[6] + sk4_ * (Gs[1] * mk[3] + Gs[3] * mk[1]);
    const double A0_7 = sm * m[7] + sk4_ * (Gs[2] * mk[2]);
    const double A0_8 = sm2_ * m[8] + sk4_ * (Gs[2] * mk[3] + Gs[3] * mk[2]);
    const double A0_9 = sm * m[9] + sk4_ * (Gs[3] * mk[3]);
    const double A1_1 = sm4_ * m[4] + sk4_ * (Gs[0] * mk[4] + Gd1 * mk[1] + Gs[4] * mk[0]);
    const double A1_2 = sm4_ * m[5] + sk4_ * (Gs[0] * mk[5] + Gs[1] * mk[2] + Gs[2] * mk[1] + Gs[5] * mk[0]);
    const double A1_3 = sm4_ * m[6] + sk4_ * (Gs[0] * mk[6] + Gs[1] * mk[3] + Gs[3] * mk[1] + Gs[6] * mk[0]);
    const double A1_4 = sm2_ * m[10] + sk4_ * (Gs[1] * mk[4] + Gs[4] * mk[1]);
    const double A1_5 = sm4_ * m[11] + sk4_ * (Gs[1] * mk[5] + Gs[2] * mk[4] + Gs[4] * mk[2] + Gs[5] * mk[1]);
    const double A1_6 = sm4_ * m[12] + sk4_ * (Gs[1] * mk[6] + Gs[3] * mk[4] + Gs[4] * mk[3] + Gs[6] * mk[1]);
    const double A1_7 = sm2_ * m[13] + sk4_ * (Gs[2] * mk[5] + Gs[5] * mk[2]);
    const double A1_8 = sm4_ * m[14] + sk4_ * (Gs[2] * mk[6] + Gs[3] * mk[5] + Gs[5] * mk[3] + Gs[6] * mk[2]);
    const double A1_9 = sm2_ * m[15] + sk4_ * (Gs[3] * mk[6] + Gs[6] * mk[3]);
    const double A2_2 = sm4_ * m[7] + sk4_ * (Gs[0] * mk[7] + Gd2 * mk[2] + Gs[7] * mk[0]);
    const double A2_3 = sm4_ * m[8] + sk4_ * (Gs[0] * mk[8] + Gs[2] * mk[3] + Gs[3] * mk[2] + Gs[8] * mk[0]);
    const double A2_4 = sm2_ * m[11] + sk4_ * (Gs[1] * mk[5] + Gs[5] * mk[1]);
    const double A2_5 = sm4_ * m[13] + sk4_ * (Gs[1] * mk[7] + Gs[2] * mk[5] + Gs[5] * mk[2] + Gs[7] * mk[1]);
    const double A2_6 = sm4_ * m[14] + sk4_ * (Gs[1] * mk[8] + Gs[3] * mk[5] + Gs[5] * mk[3] + Gs[8] * mk[1]);
    const double A2_7 = sm2_ * m[16] + sk4_ * (Gs[2] * mk[7] + Gs[7] * mk[2]);
    const double A2_8 = sm4_ * m[17] + sk4_ * (Gs[2] * mk[8] + Gs[3] * mk[7] + Gs[7] * mk[3] + Gs[8] * mk[2]);
    const double A2_9 = sm2_ * m[18] + sk4_ * (Gs[3] * mk[8] + Gs[8] * mk[3]);
    const double A3_3 = sm4_ * m[9] + sk4_ * (Gs[0] * mk[9] + Gd3 * mk[3] + Gs[9] * mk[0]);
    const double A3_4 = sm2_ * m[12] + sk4_ * (Gs[1] * mk[6] + Gs[6] * mk[1]);
    const double A3_5 = sm4_ * m[14] + sk4_ * (Gs[1] * mk[8] + Gs[2] * mk[6] + Gs[6] * mk[2] + Gs[8] * mk[1]);
    const double A3_6 = sm4_ * m[15] + sk4_ * (Gs[1] * mk[9] + Gs[3] * mk[6] + Gs[6] * mk[3] + Gs[9] * mk[1]);
    const double A3_7 = sm2_ * m[17] + sk4_ * (Gs[2] * mk[8] + Gs[8] * mk[2]);
    const double A3_8 = sm4_ * m[18] + sk4_ * (Gs[2] * mk[9] + Gs[3] * mk[8] + Gs[8] * mk[3] + Gs[9] * mk[2]);
    const double A3_9 = sm2_ * m[19] + sk4_ * (Gs[3] * mk[9] + Gs[9] * mk[3]);
    const double A4_4 = sm * m[20] + sk4_ * (Gs[4] * mk[4]);
    const double A4_5 = sm2_ * m[21] + sk4_ * (Gs[4] * mk[5] + Gs[5] * mk[4]);
    const double A4_6 = sm2_ * m[22] + sk4_ * (Gs[4] * mk[6] + Gs[6] * mk[4]);
    const double A4_7 = sm * m[23] + sk4_ * (Gs[5] * mk[5]);
    const double A4_8 = sm2_ * m[24] + sk4_ * (Gs[5] * mk[6] + Gs[6] * mk[5]);
    const double A4_9 = sm * m[25] + sk4_ * (Gs[6] * mk[6]);
    const double A5_5 = sm4_ * m[23] + sk4_ * (Gs[4] * mk[7] + Gd5 * mk[5] + Gs[7] * mk[4]);
    const double A5_6 = sm4_ * m[24] + sk4_ * (Gs[4] * mk[8] + Gs[5] * mk[6] + Gs[6] * mk[5] + Gs[8] * mk[4]);
    const double A5_7 = sm2_ * m[26] + sk4_ * (Gs[5] * mk[7] + Gs[7] * mk[5]);
    const double A5_8 = sm4_ * m[27] + sk4_ * (Gs[5] * mk[8] + Gs[6] * mk[7] + Gs[7] * mk[6] + Gs[8] * mk[5]);
    const double A5_9 = sm2_ * m[28] + sk4_ * (Gs[6] * mk[8] + Gs[8] * mk[6]);
    const double A6_6 = sm4_ * m[25] + sk4_ * (Gs[4] * mk[9] + Gd6 * mk[6] + Gs[9] * mk[4]);
    const double A6_7 = sm2_ * m[27] + sk4_ * (Gs[5] * mk[8] + Gs[8] * mk[5]);
    const double A6_8 = sm4_ * m[28] + sk4_ * (Gs[5] * mk[9] + Gs[6] * mk[8] + Gs[8] * mk[6] + Gs[9] * mk[5]);
    const double A6_9 = sm2_ * m[29] + sk4_ * (Gs[6] * mk[9] + Gs[9] * mk[6]);
    const double A7_7 = sm * m[30] + sk4_ * (Gs[7] * mk[7]);
    const double A7_8 = sm2_ * m[31] + sk4_ * (Gs[7] * mk[8] + Gs[8] * mk[7]);
    const double A7_9 = sm * m[32] + sk4_ * (Gs[8] * mk[8]);
    const double A8_8 = sm4_ * m[32] + sk4_ * (Gs[7] * mk[9] + Gd8 * mk[8] + Gs[9] * mk[7]);
    const double A8_9 = sm2_ * m[33] + sk4_ * (Gs[8] * mk[9] + Gs[9] * mk[8]);
    const double A9_9 = sm * m[34] + sk4_ * (Gs[9] * mk[9]);
    // L = T A T^T: a column b of X = A T^T where T's row b has several
    // entries, otherwise the entries of A directly
    {
      const double X0 = A0_0 - 0.5 * A0_1 - 0.5 * A0_2 - 0.5 * A0_3;
      const double X1 = A0_1 - 0.5 * A1_1 - 0.5 * A1_2 - 0.5 * A1_3;
      const double X2 = A0_2 - 0.5 * A1_2 - 0.5 * A2_2 - 0.5 * A2_3;
      const double X3 = A0_3 - 0.5 * A1_3 - 0.5 * A2_3 - 0.5 * A3_3;
      const double X4 = A0_4 - 0.5 * A1_4 - 0.5 * A2_4 - 0.5 * A3_4;
      const double X5 = A0_5 - 0.5 * A1_5 - 0.5 * A2_5 - 0.5 * A3_5;
      const double X6 = A0_6 - 0.5 * A1_6 - 0.5 * A2_6 - 0.5 * A3_6;
      const double X7 = A0_7 - 0.5 * A1_7 - 0.5 * A2_7 - 0.5 * A3_7;
      const double X8 = A0_8 - 0.5 * A1_8 - 0.5 * A2_8 - 0.5 * A3_8;
      const double X9 = A0_9 - 0.5 * A1_9 - 0.5 * A2_9 - 0.5 * A3_9;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2 - 0.5 * X3);
      out[0] = v0_;
    }
    {
      const double X0 = -0.5 * A0_1 + A0_4 - 0.5 * A0_5 - 0.5 * A0_6;
      const double X1 = -0.5 * A1_1 + A1_4 - 0.5 * A1_5 - 0.5 * A1_6;
      const double X2 = -0.5 * A1_2 + A2_4 - 0.5 * A2_5 - 0.5 * A2_6;
      const double X3 = -0.5 * A1_3 + A3_4 - 0.5 * A3_5 - 0.5 * A3_6;
      const double X4 = -0.5 * A1_4 + A4_4 - 0.5 * A4_5 - 0.5 * A4_6;
      const double X5 = -0.5 * A1_5 + A4_5 - 0.5 * A5_5 - 0.5 * A5_6;
      const double X6 = -0.5 * A1_6 + A4_6 - 0.5 * A5_6 - 0.5 * A6_6;
      const double X7 = -0.5 * A1_7 + A4_7 - 0.5 * A5_7 - 0.5 * A6_7;
      const double X8 = -0.5 * A1_8 + A4_8 - 0.5 * A5_8 - 0.5 * A6_8;
      const double X9 = -0.5 * A1_9 + A4_9 - 0.5 * A5_9 - 0.5 * A6_9;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2 - 0.5 * X3);
      out[1] = v0_;
      out[10] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X4 - 0.5 * X5 - 0.5 * X6);
      out[11] = v1_;
    }
    {
      const double X0 = -0.5 * A0_2 - 0.5 * A0_5 + A0_7 - 0.5 * A0_8;
      const double X1 = -0.5 * A1_2 - 0.5 * A1_5 + A1_7 - 0.5 * A1_8;
      const double X2 = -0.5 * A2_2 - 0.5 * A2_5 + A2_7 - 0.5 * A2_8;
      const double X3 = -0.5 * A2_3 - 0.5 * A3_5 + A3_7 - 0.5 * A3_8;
      const double X4 = -0.5 * A2_4 - 0.5 * A4_5 + A4_7 - 0.5 * A4_8;
      const double X5 = -0.5 * A2_5 - 0.5 * A5_5 + A5_7 - 0.5 * A5_8;
      const double X6 = -0.5 * A2_6 - 0.5 * A5_6 + A6_7 - 0.5 * A6_8;
      const double X7 = -0.5 * A2_7 - 0.5 * A5_7 + A7_7 - 0.5 * A7_8;
      const double X8 = -0.5 * A2_8 - 0.5 * A5_8 + A7_8 - 0.5 * A8_8;
      const double X9 = -0.5 * A2_9 - 0.5 * A5_9 + A7_9 - 0.5 * A8_9;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2 - 0.5 * X3);
      out[2] = v0_;
      out[20] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X4 - 0.5 * X5 - 0.5 * X6);
      out[12] = v1_;
      out[21] = v1_;
      const T v2_ = (T)(-0.5 * X2 - 0.5 * X5 + X7 - 0.5 * X8);
      out[22] = v2_;
    }
    {
      const double X0 = -0.5 * A0_3 - 0.5 * A0_6 - 0.5 * A0_8 + A0_9;
      const double X1 = -0.5 * A1_3 - 0.5 * A1_6 - 0.5 * A1_8 + A1_9;
      const double X2 = -0.5 * A2_3 - 0.5 * A2_6 - 0.5 * A2_8 + A2_9;
      const double X3 = -0.5 * A3_3 - 0.5 * A3_6 - 0.5 * A3_8 + A3_9;
      const double X4 = -0.5 * A3_4 - 0.5 * A4_6 - 0.5 * A4_8 + A4_9;
      const double X5 = -0.5 * A3_5 - 0.5 * A5_6 - 0.5 * A5_8 + A5_9;
      const double X6 = -0.5 * A3_6 - 0.5 * A6_6 - 0.5 * A6_8 + A6_9;
      const double X7 = -0.5 * A3_7 - 0.5 * A6_7 - 0.5 * A7_8 + A7_9;
      const double X8 = -0.5 * A3_8 - 0.5 * A6_8 - 0.5 * A8_8 + A8_9;
      const double X9 = -0.5 * A3_9 - 0.5 * A6_9 - 0.5 * A8_9 + A9_9;
      const T v0_ = (T)(X0 - 0.5 * X1 - 0.5 * X2 - 0.5 * X3);
      out[3] = v0_;
      out[30] = v0_;
      const T v1_ = (T)(-0.5 * X1 + X4 - 0.5 * X5 - 0.5 * X6);
      out[13] = v1_;
      out[31] = v1_;
      const T v2_ = (T)(-0.5 * X2 - 0.5 * X5 + X7 - 0.5 * X8);
      out[23] = v2_;
      out[32] = v2_;
      const T v3_ = (T)(-0.5 * X3 - 0.5 * X6 - 0.5 * X8 + X9);
      out[33] = v3_;
    }
    {
      const T v0_ = (T)(2.0 * A0_1 - A1_1 - A1_2 - A1_3);
      out[4] = v0_;
      out[40] = v0_;
      const T v1_ = (T)(-A1_1 + 2.0 * A1_4 - A1_5 - A1_6);
      out[14] = v1_;
      out[41] = v1_;
      const T v2_ = (T)(-A1_2 - A1_5 + 2.0 * A1_7 - A1_8);
      out[24] = v2_;
      out[42] = v2_;
      const T v3_ = (T)(-A1_3 - A1_6 - A1_8 + 2.0 * A1_9);
      out[34] = v3_;
      out[43] = v3_;
      const T v4_ = (T)(4.0 * A1_1);
      out[44] = v4_;
    }
    {
      const T v0_ = (T)(2.0 * A0_2 - A1_2 - A2_2 - A2_3);
      out[5] = v0_;
      out[50] = v0_;
      const T v1_ = (T)(-A1_2 + 2.0 * A2_4 - A2_5 - A2_6);
      out[15] = v1_;
      out[51] = v1_;
      const T v2_ = (T)(-A2_2 - A2_5 + 2.0 * A2_7 - A2_8);
      out[25] = v2_;
      out[52] = v2_;
      const T v3_ = (T)(-A2_3 - A2_6 - A2_8 + 2.0 * A2_9);
      out[35] = v3_;
      out[53] = v3_;
      const T v4_ = (T)(4.0 * A1_2);
      out[45] = v4_;
      out[54] = v4_;
      const T v5_ = (T)(4.0 * A2_2);
      out[55] = v5_;
    }
    {
      const T v0_ = (T)(2.0 * A0_3 - A1_3 - A2_3 - A3_3);
      out[6] = v0_;
      out[60] = v0_;
      const T v1_ = (T)(-A1_3 + 2.0 * A3_4 - A3_5 - A3_6);
      out[16] = v1_;
      out[61] = v1_;
      const T v2_ = (T)(-A2_3 - A3_5 + 2.0 * A3_7 - A3_8);
      out[26] = v2_;
      out[62] = v2_;
      const T v3_ = (T)(-A3_3 - A3_6 - A3_8 + 2.0 * A3_9);
      out[36] = v3_;
      out[63] = v3_;
      const T v4_ = (T)(4.0 * A1_3);
      out[46] = v4_;
      out[64] = v4_;
      const T v5_ = (T)(4.0 * A2_3);
      out[56] = v5_;
      out[65] = v5_;
      const T v6_ = (T)(4.0 * A3_3);
      out[66] = v6_;
    }
    {
      const T v0_ = (T)(2.0 * A0_5 - A1_5 - A2_5 - A3_5);
      out[7] = v0_;
      out[70] = v0_;
      const T v1_ = (T)(-A1_5 + 2.0 * A4_5 - A5_5 - A5_6);
      out[17] = v1_;
      out[71] = v1_;
      const T v2_ = (T)(-A2_5 - A5_5 + 2.0 * A5_7 - A5_8);
      out[27] = v2_;
      out[72] = v2_;
      const T v3_ = (T)(-A3_5 - A5_6 - A5_8 + 2.0 * A5_9);
      out[37] = v3_;
      out[73] = v3_;
      const T v4_ = (T)(4.0 * A1_5);
      out[47] = v4_;
      out[74] = v4_;
      const T v5_ = (T)(4.0 * A2_5);
      out[57] = v5_;
      out[75] = v5_;
      const T v6_ = (T)(4.0 * A3_5);
      out[67] = v6_;
      out[76] = v6_;
      const T v7_ = (T)(4.0 * A5_5);
      out[77] = v7_;
    }
    {
      const T v0_ = (T)(2.0 * A0_6 - A1_6 - A2_6 - A3_6);
      out[8] = v0_;
      out[80] = v0_;
      const T v1_ = (T)(-A1_6 + 2.0 * A4_6 - A5_6 - A6_6);
      out[18] = v1_;
      out[81] = v1_;
      const T v2_ = (T)(-A2_6 - A5_6 + 2.0 * A6_7 - A6_8);
      out[28] = v2_;
      out[82] = v2_;
      const T v3_ = (T)(-A3_6 - A6_6 - A6_8 + 2.0 * A6_9);
      out[38] = v3_;
      out[83] = v3_;
      const T v4_ = (T)(4.0 * A1_6);
      out[48] = v4_;
      out[84] = v4_;
      const T v5_ = (T)(4.0 * A2_6);
      out[58] = v5_;
      out[85] = v5_;
      const T v6_ = (T)(4.0 * A3_6);
      out[68] = v6_;
      out[86] = v6_;
      const T v7_ = (T)(4.0 * A5_6);
      out[78] = v7_;
      out[87] = v7_;
      const T v8_ = (T)(4.0 * A6_6);
      out[88] = v8_;
    }
    {
      const T v0_ = (T)(2.0 * A0_8 - A1_8 - A2_8 - A3_8);
      out[9] = v0_;
      out[90] = v0_;
      const T v1_ = (T)(-A1_8 + 2.0 * A4_8 - A5_8 - A6_8);
      out[19] = v1_;
      out[91] = v1_;
      const T v2_ = (T)(-A2_8 - A5_8 + 2.0 * A7_8 - A8_8);
      out[29] = v2_;
      out[92] = v2_;
      const T v3_ = (T)(-A3_8 - A6_8 - A8_8 + 2.0 * A8_9);
      out[39] = v3_;
      out[93] = v3_;
      const T v4_ = (T)(4.0 * A1_8);
      out[49] = v4_;
      out[94] = v4_;
      const T v5_ = (T)(4.0 * A2_8);
      out[59] = v5_;
      out[95] = v5_;
      const T v6_ = (T)(4.0 * A3_8);
      out[69] = v6_;
      out[96] = v6_;
      const T v7_ = (T)(4.0 * A5_8);
      out[79] = v7_;
      out[97] = v7_;
      const T v8_ = (T)(4.0 * A6_8);
      out[89] = v8_;
      out[98] = v8_;
      const T v9_ = (T)(4.0 * A8_8);
      out[99] = v9_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + m[1] + m[2] + m[3] - m[4] - 2.0 * m[5] - 2.0 * m[6] - m[7] - 2.0 * m[8] - m[9] - m[10] - 3.0 * m[11] - 3.0 * m[12] - 3.0 * m[13] - 6.0 * m[14] - 3.0 * m[15] - m[16] - 3.0 * m[17] - 3.0 * m[18] - m[19]));
    out[1] = (T)(s * (-m[1] - m[4] - 3.0 * m[5] - 3.0 * m[6] + m[10] - 2.0 * m[11] - 2.0 * m[12] - 3.0 * m[13] - 6.0 * m[14] - 3.0 * m[15] + m[20] + m[21] + m[22] - m[23] - 2.0 * m[24] - m[25] - m[26] - 3.0 * m[27] - 3.0 * m[28] - m[29]));
    out[2] = (T)(s * (-m[2] - 3.0 * m[5] - m[7] - 3.0 * m[8] - 3.0 * m[11] - 2.0 * m[13] - 6.0 * m[14] + m[16] - 2.0 * m[17] - 3.0 * m[18] - m[21] - m[23] - 3.0 * m[24] + m[26] - 2.0 * m[27] - 3.0 * m[28] + m[30] + m[31] - m[32] - m[33]));
    out[3] = (T)(s * (-m[3] - 3.0 * m[6] - 3.0 * m[8] - m[9] - 3.0 * m[12] - 6.0 * m[14] - 2.0 * m[15] - 3.0 * m[17] - 2.0 * m[18] + m[19] - m[22] - 3.0 * m[24] - m[25] - 3.0 * m[27] - 2.0 * m[28] + m[29] - m[31] - m[32] + m[33] + m[34]));
    out[4] = (T)(s * (4.0 * m[1] + 8.0 * m[4] + 8.0 * m[5] + 8.0 * m[6] + 4.0 * m[10] + 8.0 * m[11] + 8.0 * m[12] + 4.0 * m[13] + 8.0 * m[14] + 4.0 * m[15]));
    out[5] = (T)(s * (4.0 * m[2] + 8.0 * m[5] + 8.0 * m[7] + 8.0 * m[8] + 4.0 * m[11] + 8.0 * m[13] + 8.0 * m[14] + 4.0 * m[16] + 8.0 * m[17] + 4.0 * m[18]));
    out[6] = (T)(s * (4.0 * m[3] + 8.0 * m[6] + 8.0 * m[8] + 8.0 * m[9] + 4.0 * m[12] + 8.0 * m[14] + 8.0 * m[15] + 4.0 * m[17] + 8.0 * m[18] + 4.0 * m[19]));
    out[7] = (T)(s * (4.0 * m[5] + 8.0 * m[11] + 8.0 * m[13] + 8.0 * m[14] + 4.0 * m[21] + 8.0 * m[23] + 8.0 * m[24] + 4.0 * m[26] + 8.0 * m[27] + 4.0 * m[28]));
    out[8] = (T)(s * (4.0 * m[6] + 8.0 * m[12] + 8.0 * m[14] + 8.0 * m[15] + 4.0 * m[22] + 8.0 * m[24] + 8.0 * m[25] + 4.0 * m[27] + 8.0 * m[28] + 4.0 * m[29]));
    out[9] = (T)(s * (4.0 * m[8] + 8.0 * m[14] + 8.0 * m[17] + 8.0 * m[18] + 4.0 * m[24] + 8.0 * m[27] + 8.0 * m[28] + 4.0 * m[31] + 8.0 * m[32] + 4.0 * m[33]));
  }
};  // 508 coefficient terms
template <>
struct Moments<3, 3> {
  static constexpr int NM = 84;  // degree-6 moments
  static constexpr int NK = 35;  // degree-4 moments
  static constexpr int NQ = 20;  // degree-3 monomials per point
  XG_DEV static void accum(const double *l, double w, double *m) {
    const double t0 = l[0] * l[0];
    const double t1 = l[1] * l[0];
    const double t2 = l[2] * l[0];
    const double t3 = l[3] * l[0];
    const double t4 = l[1] * l[1];
    const double t5 = l[2] * l[1];
    const double t6 = l[3] * l[1];
    const double t7 = l[2] * l[2];
    const double t8 = l[3] * l[2];
    const double t9 = l[3] * l[3];
    const double t10 = t0 * l[0];
    const double t11 = t1 * l[0];
    const double t12 = t2 * l[0];
    const double t13 = t3 * l[0];
    const double t14 = t4 * l[0];
    const double t15 = t5 * l[0];
    const double t16 = t6 * l[0];
    const double t17 = t7 * l[0];
    const double t18 = t8 * l[0];
    const double t19 = t9 * l[0];
    const double t20 = t4 * l[1];
    const double t21 = t5 * l[1];
    const double t22 = t6 * l[1];
    const double t23 = t7 * l[1];
    const double t24 = t8 * l[1];
    const double t25 = t9 * l[1];
    const double t26 = t7 * l[2];
    const double t27 = t8 * l[2];
    const double t28 = t9 * l[2];
    const double t29 = t9 * l[3];
    {
      const double wb = w * t10;
      m[0] = fma(wb, t10, m[0]);
      m[1] = fma(wb, t11, m[1]);
      m[2] = fma(wb, t12, m[2]);
      m[3] = fma(wb, t13, m[3]);
      m[4] = fma(wb, t14, m[4]);
      m[5] = fma(wb, t15, m[5]);
      m[6] = fma(wb, t16, m[6]);
      m[7] = fma(wb, t17, m[7]);
      m[8] = fma(wb, t18, m[8]);
      m[9] = fma(wb, t19, m[9]);
      m[10] = fma(wb, t20, m[10]);
      m[11] = fma(wb, t21, m[11]);
      m[12] = fma(wb, t22, m[12]);
      m[13] = fma(wb, t23, m[13]);
      m[14] = fma(wb, t24, m[14]);
      m[15] = fma(wb, t25, m[15]);
      m[16] = fma(wb, t26, m[16]);
      m[17] = fma(wb, t27, m[17]);
      m[18] = fma(wb, t28, m[18]);
      m[19] = fma(wb, t29, m[19]);
    }
    {
      const double wb = w * t11;
      m[20] = fma(wb, t20, m[20]);
      m[21] = fma(wb, t21, m[21]);
      m[22] = fma(wb, t22, m[22]);
      m[23] = fma(wb, t23, m[23]);
      m[24] = fma(wb, t24, m[24]);
      m[25] = fma(wb, t25, m[25]);
      m[26] = fma(wb, t26, m[26]);
      m[27] = fma(wb, t27, m[27]);
      m[28] = fma(wb, t28, m[28]);
      m[29] = fma(wb, t29, m[29]);
    }
    {
      const double wb = w * t12;
      m[30] = fma(wb, t26, m[30]);
      m[31] = fma(wb, t27, m[31]);
      m[32] = fma(wb, t28, m[32]);
      m[33] = fma(wb, t29, m[33]);
    }
    {
      const double wb = w * t13;
      m[34] = fma(wb, t29, m[34]);
    }
    {
      const double wb = w * t14;
      m[35] = fma(wb, t20, m[35]);
      m[36] = fma(wb, t21, m[36]);
      m[37] = fma(wb, t22, m[37]);
      m[38] = fma(wb, t23, m[38]);
      m[39] = fma(wb, t24, m[39]);
      m[40] = fma(wb, t25, m[40]);
      m[41] = fma(wb, t26, m[41]);
      m[42] = fma(wb, t27, m[42]);
      m[43] = fma(wb, t28, m[43]);
      m[44] = fma(wb, t29, m[44]);
    }
    {
      const double wb = w * t15;
      m[45] = fma(wb, t26, m[45]);
      m[46] = fma(wb, t27, m[46]);
      m[47] = fma(wb, t28, m[47]);
      m[48] = fma(wb, t29, m[48]);
    }
    {
      const double wb = w * t16;
      m[49] = fma(wb, t29, m[49]);
    }
    {
      const double wb = w * t17;
      m[50] = fma(wb, t26, m[50]);
      m[51] = fma(wb, t27, m[51]);
      m[52] = fma(wb, t28, m[52]);
      m[53] = fma(wb, t29, m[53]);
    }
    {
      const double wb = w * t18;
      m[54] = fma(wb, t29, m[54]);
    }
    {
      const double wb = w * t19;
      m[55] = fma(wb, t29, m[55]);
    }
    {
      const double wb = w * t20;
      m[56] = fma(wb, t20, m[56]);
      m[57] = fma(wb, t21, m[57]);
      m[58] = fma(wb, t22, m[58]);
      m[59] = fma(wb, t23, m[59]);
      m[60] = fma(wb, t24, m[60]);
      m[61] = fma(wb, t25, m[61]);
      m[62] = fma(wb, t26, m[62]);
      m[63] = fma(wb, t27, m[63]);
      m[64] = fma(wb, t28, m[64]);
      m[65] = fma(wb, t29, m[65]);
    }
    {
      const double wb = w * t21;
      m[66] = fma(wb, t26, m[66]);
      m[67] = fma(wb, t27, m[67]);
      m[68] = fma(wb, t28, m[68]);
      m[69] = fma(wb, t29, m[69]);
    }
    {
      const double wb = w * t22;
      m[70] = fma(wb, t29, m[70]);
    }
    {
      const double wb = w * t23;
      m[71] = fma(wb, t26, m[71]);
      m[72] = fma(wb, t27, m[72]);
      m[73] = fma(wb, t28, m[73]);
      m[74] = fma(wb, t29, m[74]);
    }
    {
      const double wb = w * t24;
      m[75] = fma(wb, t29, m[75]);
    }
    {
      const double wb = w * t25;
      m[76] = fma(wb, t29, m[76]);
    }
    {
      const double wb = w * t26;
      m[77] = fma(wb, t26, m[77]);
      m[78] = fma(wb, t27, m[78]);
      m[79] = fma(wb, t28, m[79]);
      m[80] = fma(wb, t29, m[80]);
    }
    {
      const double wb = w * t27;
      m[81] = fma(wb, t29, m[81]);
    }
    {
      const double wb = w * t28;
      m[82] = fma(wb, t29, m[82]);
    }
    {
      const double wb = w * t29;
      m[83] = fma(wb, t29, m[83]);
    }
  }
  // h = (w - <z, v>) / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_first(const double *y, double w, const double *v, double *h) {
    h[83] = w;
    h[55] = fma(y[0], h[83], -v[0]);
    h[76] = fma(y[1], h[83], -v[1]);
    h[82] = fma(y[2], h[83], -v[2]);
    h[34] = y[0] * h[55];
    h[49] = fma(y[1], h[55], y[0] * h[76]);
    h[54] = fma(y[2], h[55], y[0] * h[82]);
    h[70] = y[1] * h[76];
    h[75] = fma(y[2], h[76], y[1] * h[82]);
    h[81] = y[2] * h[82];
    h[19] = y[0] * h[34];
    h[29] = fma(y[1], h[34], y[0] * h[49]);
    h[33] = fma(y[2], h[34], y[0] * h[54]);
    h[44] = fma(y[1], h[49], y[0] * h[70]);
    h[48] = fma(y[2], h[49], fma(y[1], h[54], y[0] * h[75]));
    h[53] = fma(y[2], h[54], y[0] * h[81]);
    h[65] = y[1] * h[70];
    h[69] = fma(y[2], h[70], y[1] * h[75]);
    h[74] = fma(y[2], h[75], y[1] * h[81]);
    h[80] = y[2] * h[81];
    h[9] = y[0] * h[19];
    h[15] = fma(y[1], h[19], y[0] * h[29]);
    h[18] = fma(y[2], h[19], y[0] * h[33]);
    h[25] = fma(y[1], h[29], y[0] * h[44]);
    h[28] = fma(y[2], h[29], fma(y[1], h[33], y[0] * h[48]));
    h[32] = fma(y[2], h[33], y[0] * h[53]);
    h[40] = fma(y[1], h[44], y[0] * h[65]);
    h[43] = fma(y[2], h[44], fma(y[1], h[48], y[0] * h[69]));
    h[47] = fma(y[2], h[48], fma(y[1], h[53], y[0] * h[74]));
    h[52] = fma(y[2], h[53], y[0] * h[80]);
    h[61] = y[1] * h[65];
    h[64] = fma(y[2], h[65], y[1] * h[69]);
    h[68] = fma(y[2], h[69], y[1] * h[74]);
    h[73] = fma(y[2], h[74], y[1] * h[80]);
    h[79] = y[2] * h[80];
    h[3] = y[0] * h[9];
    h[6] = fma(y[1], h[9], y[0] * h[15]);
    h[8] = fma(y[2], h[9], y[0] * h[18]);
    h[12] = fma(y[1], h[15], y[0] * h[25]);
    h[14] = fma(y[2], h[15], fma(y[1], h[18], y[0] * h[28]));
    h[17] = fma(y[2], h[18], y[0] * h[32]);
    h[22] = fma(y[1], h[25], y[0] * h[40]);
    h[24] = fma(y[2], h[25], fma(y[1], h[28], y[0] * h[43]));
    h[27] = fma(y[2], h[28], fma(y[1], h[32], y[0] * h[47]));
    h[31] = fma(y[2], h[32], y[0] * h[52]);
    h[37] = fma(y[1], h[40], y[0] * h[61]);
    h[39] = fma(y[2], h[40], fma(y[1], h[43], y[0] * h[64]));
    h[42] = fma(y[2], h[43], fma(y[1], h[47], y[0] * h[68]));
    h[46] = fma(y[2], h[47], fma(y[1], h[52], y[0] * h[73]));
    h[51] = fma(y[2], h[52], y[0] * h[79]);
    h[58] = y[1] * h[61];
    h[60] = fma(y[2], h[61], y[1] * h[64]);
    h[63] = fma(y[2], h[64], y[1] * h[68]);
    h[67] = fma(y[2], h[68], y[1] * h[73]);
    h[72] = fma(y[2], h[73], y[1] * h[79]);
    h[78] = y[2] * h[79];
    h[0] = y[0] * h[3];
    h[1] = fma(y[1], h[3], y[0] * h[6]);
    h[2] = fma(y[2], h[3], y[0] * h[8]);
    h[4] = fma(y[1], h[6], y[0] * h[12]);
    h[5] = fma(y[2], h[6], fma(y[1], h[8], y[0] * h[14]));
    h[7] = fma(y[2], h[8], y[0] * h[17]);
    h[10] = fma(y[1], h[12], y[0] * h[22]);
    h[11] = fma(y[2], h[12], fma(y[1], h[14], y[0] * h[24]));
    h[13] = fma(y[2], h[14], fma(y[1], h[17], y[0] * h[27]));
    h[16] = fma(y[2], h[17], y[0] * h[31]);
    h[20] = fma(y[1], h[22], y[0] * h[37]);
    h[21] = fma(y[2], h[22], fma(y[1], h[24], y[0] * h[39]));
    h[23] = fma(y[2], h[24], fma(y[1], h[27], y[0] * h[42]));
    h[26] = fma(y[2], h[27], fma(y[1], h[31], y[0] * h[46]));
    h[30] = fma(y[2], h[31], y[0] * h[51]);
    h[35] = fma(y[1], h[37], y[0] * h[58]);
    h[36] = fma(y[2], h[37], fma(y[1], h[39], y[0] * h[60]));
    h[38] = fma(y[2], h[39], fma(y[1], h[42], y[0] * h[63]));
    h[41] = fma(y[2], h[42], fma(y[1], h[46], y[0] * h[67]));
    h[45] = fma(y[2], h[46], fma(y[1], h[51], y[0] * h[72]));
    h[50] = fma(y[2], h[51], y[0] * h[78]);
    h[56] = y[1] * h[58];
    h[57] = fma(y[2], h[58], y[1] * h[60]);
    h[59] = fma(y[2], h[60], y[1] * h[63]);
    h[62] = fma(y[2], h[63], y[1] * h[67]);
    h[66] = fma(y[2], h[67], y[1] * h[72]);
    h[71] = fma(y[2], h[72], y[1] * h[78]);
    h[77] = y[2] * h[78];
  }
  // h <- h / (1 - <z, y>), truncated at degree 2P
  XG_DEV static void aser_step(const double *y, double *h) {
    h[55] = fma(y[0], h[83], h[55]);
    h[76] = fma(y[1], h[83], h[76]);
    h[82] = fma(y[2], h[83], h[82]);
    h[34] = fma(y[0], h[55], h[34]);
    h[49] = fma(y[1], h[55], fma(y[0], h[76], h[49]));
    h[54] = fma(y[2], h[55], fma(y[0], h[82], h[54]));
    h[70] = fma(y[1], h[76], h[70]);
    h[75] = fma(y[2], h[76], fma(y[1], h[82], h[75]));
    h[81] = fma(y[2], h[82], h[81]);
    h[19] = fma(y[0], h[34], h[19]);
    h[29] = fma(y[1], h[34], fma(y[0], h[49], h[29]));
    h[33] = fma(y[2], h[34], fma(y[0], h[54], h[33]));
    h[44] = fma(y[1], h[49], fma(y[0], h[70], h[44]));
    h[48] = fma(y[2], h[49], fma(y[1], h[54], fma(y[0], h[75], h[48])));
    h[53] = fma(y[2], h[54], fma(y[0], h[81], h[53]));
    h[65] = fma(y[1], h[70], h[65]);
    h[69] = fma(y[2], h[70], fma(y[1], h[75], h[69]));
    h[74] = fma(y[2], h[75], fma(y[1], h[81], h[74]));
    h[80] = fma(y[2], h[81], h[80]);
    h[9] = fma(y[0], h[19], h[9]);
    h[15] = fma(y[1], h[19], fma(y[0], h[29], h[15]));
    h[18] = fma(y[2], h[19], fma(y[0], h[33], h[18]));
    h[25] = fma(y[1], h[29], fma(y[0], h[44], h[25]));
    h[28] = fma(y[2], h[29], fma(y[1], h[33], fma(y[0], h[48], h[28])));
    h[32] = fma(y[2], h[33], fma(y[0], h[53], h[32]));
    h[40] = fma(y[1], h[44], fma(y[0], h[65], h[40]));
    h[43] = fma(y[2], h[44], fma(y[1], h[48], fma(y[0], h[69], h[43])));
    h[47] = fma(y[2], h[48], fma(y[1], h[53], fma(y[0], h[74], h[47])));
    h[52] = fma(y[2], h[53], fma(y[0], h[80], h[52]));
    h[61] = fma(y[1], h[65], h[61]);
    h[64] = fma(y[2], h[65], fma(y[1], h[69], h[64]));
    h[68] = fma(y[2], h[69], fma(y[1], h[74], h[68]));
    h[73] = fma(y[2], h[74], fma(y[1], h[80], h[73]));
    h[79] = fma(y[2], h[80], h[79]);
    h[3] = fma(y[0], h[9], h[3]);
    h[6] = fma(y[1], h[9], fma(y[0], h[15], h[6]));
    h[8] = fma(y[2], h[9], fma(y[0], h[18], h[8]));
    h[12] = fma(y[1], h[15], fma(y[0], h[25], h[12]));
    h[14] = fma(y[2], h[15], fma(y[1], h[18], fma(y[0], h[28], h[14])));
    h[17] = fma(y[2], h[18], fma(y[0], h[32], h[17]));
    h[22] = fma(y[1], h[25], fma(y[0], h[40], h[22]));
    h[24] = fma(y[2], h[25], fma(y[1], h[28], fma(y[0], h[43], h[24])));
    h[27] = fma(y[2], h[28], fma(y[1], h[32], fma(y[0], h[47], h[27])));
    h[31] = fma(y[2], h[32], fma(y[0], h[52], h[31]));
    h[37] = fma(y[1], h[40], fma(y[0], h[61], h[37]));
    h[39] = fma(y[2], h[40], fma(y[1], h[43], fma(y[0], h[64], h[39])));
    h[42] = fma(y[2], h[43], fma(y[1], h[47], fma(y[0], h[68], h[42])));
    h[46] = fma(y[2], h[47], fma(y[1], h[52], fma(y[0], h[73], h[46])));
    h[51] = fma(y[2], h[52], fma(y[0], h[79], h[51]));
    h[58] = fma(y[1], h[61], h[58]);
    h[60] = fma(y[2], h[61], fma(y[1], h[64], h[60]));
    h[63] = fma(y[2], h[64], fma(y[1], h[68], h[63]));
    h[67] = fma(y[2], h[68], fma(y[1], h[73], h[67]));
    h[72] = fma(y[2], h[73], fma(y[1], h[79], h[72]));
    h[78] = fma(y[2], h[79], h[78]);
    h[0] = fma(y[0], h[3], h[0]);
    h[1] = fma(y[1], h[3], fma(y[0], h[6], h[1]));
    h[2] = fma(y[2], h[3], fma(y[0], h[8], h[2]));
    h[4] = fma(y[1], h[6], fma(y[0], h[12], h[4]));
    h[5] = fma(y[2], h[6], fma(y[1], h[8], fma(y[0], h[14], h[5])));
    h[7] = fma(y[2], h[8], fma(y[0], h[17], h[7]));
    h[10] = fma(y[1], h[12], fma(y[0], h[22], h[10]));
    h[11] = fma(y[2], h[12], fma(y[1], h[14], fma(y[0], h[24], h[11])));
    h[13] = fma(y[2], h[14], fma(y[1], h[17], fma(y[0], h[27], h[13])));
    h[16] = fma(y[2], h[17], fma(y[0], h[31], h[16]));
    h[20] = fma(y[1], h[22], fma(y[0], h[37], h[20]));
    h[21] = fma(y[2], h[22], fma(y[1], h[24], fma(y[0], h[39], h[21])));
    h[23] = fma(y[2], h[24], fma(y[1], h[27], fma(y[0], h[42], h[23])));
    h[26] = fma(y[2], h[27], fma(y[1], h[31], fma(y[0], h[46], h[26])));
    h[30] = fma(y[2], h[31], fma(y[0], h[51], h[30]));
    h[35] = fma(y[1], h[37], fma(y[0], h[58], h[35]));
    h[36] = fma(y[2], h[37], fma(y[1], h[39], fma(y[0], h[60], h[36])));
    h[38] = fma(y[2], h[39], fma(y[1], h[42], fma(y[0], h[63], h[38])));
    h[41] = fma(y[2], h[42], fma(y[1], h[46], fma(y[0], h[67], h[41])));
    h[45] = fma(y[2], h[46], fma(y[1], h[51], fma(y[0], h[72], h[45])));
    h[50] = fma(y[2], h[51], fma(y[0], h[78], h[50]));
    h[56] = fma(y[1], h[58], h[56]);
    h[57] = fma(y[2], h[58], fma(y[1], h[60], h[57]));
    h[59] = fma(y[2], h[60], fma(y[1], h[63], h[59]));
    h[62] = fma(y[2], h[63], fma(y[1], h[67], h[62]));
    h[66] = fma(y[2], h[67], fma(y[1], h[72], h[66]));
    h[71] = fma(y[2], h[72], fma(y[1], h[78], h[71]));
    h[77] = fma(y[2], h[78], h[77]);
  }
  // m_alpha <- int_T lam^alpha - m_alpha over the whole reference simplex T
  XG_DEV static void complement(double *m) {
    m[0] = 0.001984126984126984 - m[0];
    m[1] = 0.00033068783068783067 - m[1];
    m[2] = 0.00033068783068783067 - m[2];
    m[3] = 0.00033068783068783067 - m[3];
    m[4] = 0.00013227513227513228 - m[4];
    m[5] = 6.613756613756614e-05 - m[5];
    m[6] = 6.613756613756614e-05 - m[6];
    m[7] = 0.00013227513227513228 - m[7];
    m[8] = 6.613756613756614e-05 - m[8];
    m[9] = 0.00013227513227513228 - m[9];
    m[10] = 9.92063492063492e-05 - m[10];
    m[11] = 3.306878306878307e-05 - m[11];
    m[12] = 3.306878306878307e-05 - m[12];
    m[13] = 3.306878306878307e-05 - m[13];
    m[14] = 1.6534391534391536e-05 - m[14];
    m[15] = 3.306878306878307e-05 - m[15];
    m[16] = 9.92063492063492e-05 - m[16];
    m[17] = 3.306878306878307e-05 - m[17];
    m[18] = 3.306878306878307e-05 - m[18];
    m[19] = 9.92063492063492e-05 - m[19];
    m[20] = 0.00013227513227513228 - m[20];
    m[21] = 3.306878306878307e-05 - m[21];
    m[22] = 3.306878306878307e-05 - m[22];
    m[23] = 2.2045855379188714e-05 - m[23];
    m[24] = 1.1022927689594357e-05 - m[24];
    m[25] = 2.2045855379188714e-05 - m[25];
    m[26] = 3.306878306878307e-05 - m[26];
    m[27] = 1.1022927689594357e-05 - m[27];
    m[28] = 1.1022927689594357e-05 - m[28];
    m[29] = 3.306878306878307e-05 - m[29];
    m[30] = 0.00013227513227513228 - m[30];
    m[31] = 3.306878306878307e-05 - m[31];
    m[32] = 2.2045855379188714e-05 - m[32];
    m[33] = 3.306878306878307e-05 - m[33];
    m[34] = 0.00013227513227513228 - m[34];
    m[35] = 0.00033068783068783067 - m[35];
    m[36] = 6.613756613756614e-05 - m[36];
    m[37] = 6.613756613756614e-05 - m[37];
    m[38] = 3.306878306878307e-05 - m[38];
    m[39] = 1.6534391534391536e-05 - m[39];
    m[40] = 3.306878306878307e-05 - m[40];
    m[41] = 3.306878306878307e-05 - m[41];
    m[42] = 1.1022927689594357e-05 - m[42];
    m[43] = 1.1022927689594357e-05 - m[43];
    m[44] = 3.306878306878307e-05 - m[44];
    m[45] = 6.613756613756614e-05 - m[45];
    m[46] = 1.6534391534391536e-05 - m[46];
    m[47] = 1.1022927689594357e-05 - m[47];
    m[48] = 1.6534391534391536e-05 - m[48];
    m[49] = 6.613756613756614e-05 - m[49];
    m[50] = 0.00033068783068783067 - m[50];
    m[51] = 6.613756613756614e-05 - m[51];
    m[52] = 3.306878306878307e-05 - m[52];
    m[53] = 3.306878306878307e-05 - m[53];
    m[54] = 6.613756613756614e-05 - m[54];
    m[55] = 0.00033068783068783067 - m[55];
    m[56] = 0.001984126984126984 - m[56];
    m[57] = 0.00033068783068783067 - m[57];
    m[58] = 0.00033068783068783067 - m[58];
    m[59] = 0.00013227513227513228 - m[59];
    m[60] = 6.613756613756614e-05 - m[60];
    m[61] = 0.00013227513227513228 - m[61];
    m[62] = 9.92063492063492e-05 - m[62];
    m[63] = 3.306878306878307e-05 - m[63];
    m[64] = 3.306878306878307e-05 - m[64];
    m[65] = 9.92063492063492e-05 - m[65];
    m[66] = 0.00013227513227513228 - m[66];
    m[67] = 3.306878306878307e-05 - m[67];
    m[68] = 2.2045855379188714e-05 - m[68];
    m[69] = 3.306878306878307e-05 - m[69];
    m[70] = 0.00013227513227513228 - m[70];
    m[71] = 0.00033068783068783067 - m[71];
    m[72] = 6.613756613756614e-05 - m[72];
    m[73] = 3.306878306878307e-05 - m[73];
    m[74] = 3.306878306878307e-05 - m[74];
    m[75] = 6.613756613756614e-05 - m[75];
    m[76] = 0.00033068783068783067 - m[76];
    m[77] = 0.001984126984126984 - m[77];
    m[78] = 0.00033068783068783067 - m[78];
    m[79] = 0.00013227513227513228 - m[79];
    m[80] = 9.92063492063492e-05 - m[80];
    m[81] = 0.00013227513227513228 - m[81];
    m[82] = 0.00033068783068783067 - m[82];
    m[83] = 0.001984126984126984 - m[83];
  }
  XG_DEV static void lower(const double *m, double *mk) {
    mk[0] = m[0] + 2.0 * m[1] + 2.0 * m[2] + 2.0 * m[3] + m[4] + 2.0 * m[5] + 2.0 * m[6] + m[7] + 2.0 * m[8] + m[9];
    mk[1] = m[1] + 2.0 * m[4] + 2.0 * m[5] + 2.0 * m[6] + m[10] + 2.0 * m[11] + 2.0 * m[12] + m[13] + 2.0 * m[14] + m[15];
    mk[2] = m[2] + 2.0 * m[5] + 2.0 * m[7] + 2.0 * m[8] + m[11] + 2.0 * m[13] + 2.0 * m[14] + m[16] + 2.0 * m[17] + m[18];
    mk[3] = m[3] + 2.0 * m[6] + 2.0 * m[8] + 2.0 * m[9] + m[12] + 2.0 * m[14] + 2.0 * m[15] + m[17] + 2.0 * m[18] + m[19];
    mk[4] = m[4] + 2.0 * m[10] + 2.0 * m[11] + 2.0 * m[12] + m[20] + 2.0 * m[21] + 2.0 * m[22] + m[23] + 2.0 * m[24] + m[25];
    mk[5] = m[5] + 2.0 * m[11] + 2.0 * m[13] + 2.0 * m[14] + m[21] + 2.0 * m[23] + 2.0 * m[24] + m[26] + 2.0 * m[27] + m[28];
    mk[6] = m[6] + 2.0 * m[12] + 2.0 * m[14] + 2.0 * m[15] + m[22] + 2.0 * m[24] + 2.0 * m[25] + m[27] + 2.0 * m[28] + m[29];
    mk[7] = m[7] + 2.0 * m[13] + 2.0 * m[16] + 2.0 * m[17] + m[23] + 2.0 * m[26] + 2.0 * m[27] + m[30] + 2.0 * m[31] + m[32];
    mk[8] = m[8] + 2.0 * m[14] + 2.0 * m[17] + 2.0 * m[18] + m[24] + 2.0 * m[27] + 2.0 * m[28] + m[31] + 2.0 * m[32] + m[33];
    mk[9] = m[9] + 2.0 * m[15] + 2.0 * m[18] + 2.0 * m[19] + m[25] + 2.0 * m[28] + 2.0 * m[29] + m[32] + 2.0 * m[33] + m[34];
    mk[10] = m[10] + 2.0 * m[20] + 2.0 * m[21] + 2.0 * m[22] + m[35] + 2.0 * m[36] + 2.0 * m[37] + m[38] + 2.0 * m[39] + m[40];
    mk[11] = m[11] + 2.0 * m[21] + 2.0 * m[23] + 2.0 * m[24] + m[36] + 2.0 * m[38] + 2.0 * m[39] + m[41] + 2.0 * m[42] + m[43];
    mk[12] = m[12] + 2.0 * m[22] + 2.0 * m[24] + 2.0 * m[25] + m[37] + 2.0 * m[39] + 2.0 * m[40] + m[42] + 2.0 * m[43] + m[44];
    mk[13] = m[13] + 2.0 * m[23] + 2.0 * m[26] + 2.0 * m[27] + m[38] + 2.0 * m[41] + 2.0 * m[42] + m[45] + 2.0 * m[46] + m[47];
    mk[14] = m[14] + 2.0 * m[24] + 2.0 * m[27] + 2.0 * m[28] + m[39] + 2.0 * m[42] + 2.0 * m[43] + m[46] + 2.0 * m[47] + m[48];
    mk[15] = m[15] + 2.0 * m[25] + 2.0 * m[28] + 2.0 * m[29] + m[40] + 2.0 * m[43] + 2.0 * m[44] + m[47] + 2.0 * m[48] + m[49];
    mk[16] = m[16] + 2.0 * m[26] + 2.0 * m[30] + 2.0 * m[31] + m[41] + 2.0 * m[45] + 2.0 * m[46] + m[50] + 2.0 * m[51] + m[52];
    mk[17] = m[17] + 2.0 * m[27] + 2.0 * m[31] + 2.0 * m[32] + m[42] + 2.0 * m[46] + 2.0 * m[47] + m[51] + 2.0 * m[52] + m[53];
    mk[18] = m[18] + 2.0 * m[28] + 2.0 * m[32] + 2.0 * m[33] + m[43] + 2.0 * m[47] + 2.0 * m[48] + m[52] + 2.0 * m[53] + m[54];
    mk[19] = m[19] + 2.0 * m[29] + 2.0 * m[33] + 2.0 * m[34] + m[44] + 2.0 * m[48] + 2.0 * m[49] + m[53] + 2.0 * m[54] + m[55];
    mk[20] = m[20] + 2.0 * m[35] + 2.0 * m[36] + 2.0 * m[37] + m[56] + 2.0 * m[57] + 2.0 * m[58] + m[59] + 2.0 * m[60] + m[61];
    mk[21] = m[21] + 2.0 * m[36] + 2.0 * m[38] + 2.0 * m[39] + m[57] + 2.0 * m[59] + 2.0 * m[60] + m[62] + 2.0 * m[63] + m[64];
    mk[22] = m[22] + 2.0 * m[37] + 2.0 * m[39] + 2.0 * m[40] + m[58] + 2.0 * m[60] + 2.0 * m[61] + m[63] + 2.0 * m[64] + m[65];
    mk[23] = m[23] + 2.0 * m[38] + 2.0 * m[41] + 2.0 * m[42] + m[59] + 2.0 * m[62] + 2.0 * m[63] + m[66] + 2.0 * m[67] + m[68];
    mk[24] = m[24] + 2.0 * m[39] + 2.0 * m[42] + 2.0 * m[43] + m[60] + 2.0 * m[63] + 2.0 * m[64] + m[67] + 2.0 * m[68] + m[69];
    mk[25] = m[25] + 2.0 * m[40] + 2.0 * m[43] + 2.0 * m[44] + m[61] + 2.0 * m[64] + 2.0 * m[65] + m[68] + 2.0 * m[69] + m[70];
    mk[26] = m[26] + 2.0 * m[41] + 2.0 * m[45] + 2.0 * m[46] + m[62] + 2.0 * m[66] + 2.0 * m[67] + m[71] + 2.0 * m[72] + m[73];
    mk[27] = m[27] + 2.0 * m[42] + 2.0 * m[46] + 2.0 * m[47] + m[63] + 2.0 * m[67] + 2.0 * m[68] + m[72] + 2.0 * m[73] + m[74];
    mk[28] = m[28] + 2.0 * m[43] + 2.0 * m[47] + 2.0 * m[48] + m[64] + 2.0 * m[68] + 2.0 * m[69] + m[73] + 2.0 * m[74] + m[75];
    mk[29] = m[29] + 2.0 * m[44] + 2.0 * m[48] + 2.0 * m[49] + m[65] + 2.0 * m[69] + 2.0 * m[70] + m[74] + 2.0 * m[75] + m[76];
    mk[30] = m[30] + 2.0 * m[45] + 2.0 * m[50] + 2.0 * m[51] + m[66] + 2.0 * m[71] + 2.0 * m[72] + m[77] + 2.0 * m[78] + m[79];
    mk[31] = m[31] + 2.0 * m[46] + 2.0 * m[51] + 2.0 * m[52] + m[67] + 2.0 * m[72] + 2.0 * m[73] + m[78] + 2.0 * m[79] + m[80];
    mk[32] = m[32] + 2.0 * m[47] + 2.0 * m[52] + 2.0 * m[53] + m[68] + 2.0 * m[73] + 2.0 * m[74] + m[79] + 2.0 * m[80] + m[81];
    mk[33] = m[33] + 2.0 * m[48] + 2.0 * m[53] + 2.0 * m[54] + m[69] + 2.0 * m[74] + 2.0 * m[75] + m[80] + 2.0 * m[81] + m[82];
    mk[34] = m[34] + 2.0 * m[49] + 2.0 * m[54] + 2.0 * m[55] + m[70] + 2.0 * m[75] + 2.0 * m[76] + m[81] + 2.0 * m[82] + m[83];
  }
  // out[a*N+b] = sm * M_ab + sk * K_ab; Gs = grad lam_i . grad lam_j, i <= j (row-major upper)
  static constexpr int NG = 10;
  template <typename T>
  XG_DEV static void forms(const double *m, const double *mk, const double *Gs, double sm, double sk,
                           T *out) {
    {
      const double M_ = m[0] - 5.0 * m[1] - 5.0 * m[2] - 5.0 * m[3] + 8.25 * m[4] + 16.5 * m[5] + 16.5 * m[6] + 8.25 * m[7] + 16.5 * m[8] + 8.25 * m[9] - 5.0 * m[10] - 15.0 * m[11] - 15.0 * m[12] - 15.0 * m[13] - 30.0 * m[14] - 15.0 * m[15] - 5.0 * m[16] - 15.0 * m[17] - 15.0 * m[18] - 5.0 * m[19] + m[20] + 4.0 * m[21] + 4.0 * m[22] + 6.0 * m[23] + 12.0 * m[24] + 6.0 * m[25] + 4.0 * m[26] + 12.0 * m[27] + 12.0 * m[28] + 4.0 * m[29] + m[30] + 4.0 * m[31] + 6.0 * m[32] + 4.0 * m[33] + m[34];
      const double K_ = Gs[0] * (30.25 * mk[0] - 77.0 * mk[1] - 77.0 * mk[2] - 77.0 * mk[3] + 60.0 * mk[4] + 120.0 * mk[5] + 120.0 * mk[6] + 60.0 * mk[7] + 120.0 * mk[8] + 60.0 * mk[9] - 14.0 * mk[10] - 42.0 * mk[11] - 42.0 * mk[12] - 42.0 * mk[13] - 84.0 * mk[14] - 42.0 * mk[15] - 14.0 * mk[16] - 42.0 * mk[17] - 42.0 * mk[18] - 14.0 * mk[19] + mk[20] + 4.0 * mk[21] + 4.0 * mk[22] + 6.0 * mk[23] + 12.0 * mk[24] + 6.0 * mk[25] + 4.0 * mk[26] + 12.0 * mk[27] + 12.0 * mk[28] + 4.0 * mk[29] + mk[30] + 4.0 * mk[31] + 6.0 * mk[32] + 4.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[0] = v_;
    }
    {
      const double M_ = m[1] - 5.0 * m[4] - 0.5 * m[5] - 0.5 * m[6] + 8.25 * m[10] + 0.75 * m[11] + 0.75 * m[12] - 3.0 * m[13] - 6.0 * m[14] - 3.0 * m[15] - 5.0 * m[20] + 0.75 * m[21] + 0.75 * m[22] + 5.25 * m[23] + 10.5 * m[24] + 5.25 * m[25] - 0.5 * m[26] - 1.5 * m[27] - 1.5 * m[28] - 0.5 * m[29] + m[35] - 0.5 * m[36] - 0.5 * m[37] - 3.0 * m[38] - 6.0 * m[39] - 3.0 * m[40] - 0.5 * m[41] - 1.5 * m[42] - 1.5 * m[43] - 0.5 * m[44] + m[45] + 4.0 * m[46] + 6.0 * m[47] + 4.0 * m[48] + m[49];
      const double K_ = Gs[1] * (5.5 * mk[0] - 45.5 * mk[1] + 4.0 * mk[2] + 4.0 * mk[3] + 80.25 * mk[4] - 1.5 * mk[5] - 1.5 * mk[6] - 7.5 * mk[7] - 15.0 * mk[8] - 7.5 * mk[9] - 45.5 * mk[10] - 1.5 * mk[11] - 1.5 * mk[12] + 39.0 * mk[13] + 78.0 * mk[14] + 39.0 * mk[15] - 5.0 * mk[16] - 15.0 * mk[17] - 15.0 * mk[18] - 5.0 * mk[19] + 5.5 * mk[20] + 4.0 * mk[21] + 4.0 * mk[22] - 7.5 * mk[23] - 15.0 * mk[24] - 7.5 * mk[25] - 5.0 * mk[26] - 15.0 * mk[27] - 15.0 * mk[28] - 5.0 * mk[29] + mk[30] + 4.0 * mk[31] + 6.0 * mk[32] + 4.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[1] = v_;
      out[20] = v_;
    }
    {
      const double M_ = m[2] - 0.5 * m[5] - 5.0 * m[7] - 0.5 * m[8] - 3.0 * m[11] + 0.75 * m[13] - 6.0 * m[14] + 8.25 * m[16] + 0.75 * m[17] - 3.0 * m[18] - 0.5 * m[21] + 5.25 * m[23] - 1.5 * m[24] + 0.75 * m[26] + 10.5 * m[27] - 1.5 * m[28] - 5.0 * m[30] + 0.75 * m[31] + 5.25 * m[32] - 0.5 * m[33] + m[36] - 0.5 * m[38] + 4.0 * m[39] - 3.0 * m[41] - 1.5 * m[42] + 6.0 * m[43] - 0.5 * m[45] - 6.0 * m[46] - 1.5 * m[47] + 4.0 * m[48] + m[50] - 0.5 * m[51] - 3.0 * m[52] - 0.5 * m[53] + m[54];
      const double K_ = Gs[2] * (5.5 * mk[0] + 4.0 * mk[1] - 45.5 * mk[2] + 4.0 * mk[3] - 7.5 * mk[4] - 1.5 * mk[5] - 15.0 * mk[6] + 80.25 * mk[7] - 1.5 * mk[8] - 7.5 * mk[9] - 5.0 * mk[10] + 39.0 * mk[11] - 15.0 * mk[12] - 1.5 * mk[13] + 78.0 * mk[14] - 15.0 * mk[15] - 45.5 * mk[16] - 1.5 * mk[17] + 39.0 * mk[18] - 5.0 * mk[19] + mk[20] - 5.0 * mk[21] + 4.0 * mk[22] - 7.5 * mk[23] - 15.0 * mk[24] + 6.0 * mk[25] + 4.0 * mk[26] - 15.0 * mk[27] - 15.0 * mk[28] + 4.0 * mk[29] + 5.5 * mk[30] + 4.0 * mk[31] - 7.5 * mk[32] - 5.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[2] = v_;
      out[40] = v_;
    }
    {
      const double M_ = m[3] - 0.5 * m[6] - 0.5 * m[8] - 5.0 * m[9] - 3.0 * m[12] - 6.0 * m[14] + 0.75 * m[15] - 3.0 * m[17] + 0.75 * m[18] + 8.25 * m[19] - 0.5 * m[22] - 1.5 * m[24] + 5.25 * m[25] - 1.5 * m[27] + 10.5 * m[28] + 0.75 * m[29] - 0.5 * m[31] + 5.25 * m[32] + 0.75 * m[33] - 5.0 * m[34] + m[37] + 4.0 * m[39] - 0.5 * m[40] + 6.0 * m[42] - 1.5 * m[43] - 3.0 * m[44] + 4.0 * m[46] - 1.5 * m[47] - 6.0 * m[48] - 0.5 * m[49] + m[51] - 0.5 * m[52] - 3.0 * m[53] - 0.5 * m[54] + m[55];
      const double K_ = Gs[3] * (5.5 * mk[0] + 4.0 * mk[1] + 4.0 * mk[2] - 45.5 * mk[3] - 7.5 * mk[4] - 15.0 * mk[5] - 1.5 * mk[6] - 7.5 * mk[7] - 1.5 * mk[8] + 80.25 * mk[9] - 5.0 * mk[10] - 15.0 * mk[11] + 39.0 * mk[12] - 15.0 * mk[13] + 78.0 * mk[14] - 1.5 * mk[15] - 5.0 * mk[16] + 39.0 * mk[17] - 1.5 * mk[18] - 45.5 * mk[19] + mk[20] + 4.0 * mk[21] - 5.0 * mk[22] + 6.0 * mk[23] - 15.0 * mk[24] - 7.5 * mk[25] + 4.0 * mk[26] - 15.0 * mk[27] - 15.0 * mk[28] + 4.0 * mk[29] + mk[30] - 5.0 * mk[31] - 7.5 * mk[32] + 4.0 * mk[33] + 5.5 * mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[3] = v_;
      out[60] = v_;
    }
    {
      const double M_ = 9.0 * m[1] - 27.0 * m[4] - 27.0 * m[5] - 27.0 * m[6] + 20.25 * m[10] + 40.5 * m[11] + 40.5 * m[12] + 20.25 * m[13] + 40.5 * m[14] + 20.25 * m[15] - 4.5 * m[20] - 13.5 * m[21] - 13.5 * m[22] - 13.5 * m[23] - 27.0 * m[24] - 13.5 * m[25] - 4.5 * m[26] - 13.5 * m[27] - 13.5 * m[28] - 4.5 * m[29];
      const double K_ = Gs[0] * (123.75 * mk[1] - 182.25 * mk[4] - 182.25 * mk[5] - 182.25 * mk[6] + 54.0 * mk[10] + 108.0 * mk[11] + 108.0 * mk[12] + 54.0 * mk[13] + 108.0 * mk[14] + 54.0 * mk[15] - 4.5 * mk[20] - 13.5 * mk[21] - 13.5 * mk[22] - 13.5 * mk[23] - 27.0 * mk[24] - 13.5 * mk[25] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]) + Gs[1] * (49.5 * mk[0] - 87.75 * mk[1] - 87.75 * mk[2] - 87.75 * mk[3] + 40.5 * mk[4] + 81.0 * mk[5] + 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[8] + 40.5 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] - 13.5 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[4] = v_;
      out[80] = v_;
    }
    {
      const double M_ = -4.5 * m[1] + 20.25 * m[4] + 6.75 * m[5] + 6.75 * m[6] - 27.0 * m[10] - 20.25 * m[11] - 20.25 * m[12] + 6.75 * m[13] + 13.5 * m[14] + 6.75 * m[15] + 9.0 * m[20] + 13.5 * m[21] + 13.5 * m[22] - 4.5 * m[26] - 13.5 * m[27] - 13.5 * m[28] - 4.5 * m[29];
      const double K_ = Gs[0] * (-24.75 * mk[1] + 81.0 * mk[4] + 6.75 * mk[5] + 6.75 * mk[6] - 67.5 * mk[10] - 40.5 * mk[11] - 40.5 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] + 13.5 * mk[22] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]) + Gs[1] * (-24.75 * mk[0] + 155.25 * mk[1] + 6.75 * mk[2] + 6.75 * mk[3] - 162.0 * mk[4] - 135.0 * mk[5] - 135.0 * mk[6] + 27.0 * mk[7] + 54.0 * mk[8] + 27.0 * mk[9] + 22.5 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 13.5 * mk[13] + 27.0 * mk[14] + 13.5 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[5] = v_;
      out[100] = v_;
    }
    {
      const double M_ = 9.0 * m[2] - 27.0 * m[5] - 27.0 * m[7] - 27.0 * m[8] + 20.25 * m[11] + 40.5 * m[13] + 40.5 * m[14] + 20.25 * m[16] + 40.5 * m[17] + 20.25 * m[18] - 4.5 * m[21] - 13.5 * m[23] - 13.5 * m[24] - 13.5 * m[26] - 27.0 * m[27] - 13.5 * m[28] - 4.5 * m[30] - 13.5 * m[31] - 13.5 * m[32] - 4.5 * m[33];
      const double K_ = Gs[0] * (123.75 * mk[2] - 182.25 * mk[5] - 182.25 * mk[7] - 182.25 * mk[8] + 54.0 * mk[11] + 108.0 * mk[13] + 108.0 * mk[14] + 54.0 * mk[16] + 108.0 * mk[17] + 54.0 * mk[18] - 4.5 * mk[21] - 13.5 * mk[23] - 13.5 * mk[24] - 13.5 * mk[26] - 27.0 * mk[27] - 13.5 * mk[28] - 4.5 * mk[30] - 13.5 * mk[31] - 13.5 * mk[32] - 4.5 * mk[33]) + Gs[2] * (49.5 * mk[0] - 87.75 * mk[1] - 87.75 * mk[2] - 87.75 * mk[3] + 40.5 * mk[4] + 81.0 * mk[5] + 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[8] + 40.5 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] - 13.5 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[6] = v_;
      out[120] = v_;
    }
    {
      const double M_ = -4.5 * m[2] + 6.75 * m[5] + 20.25 * m[7] + 6.75 * m[8] + 6.75 * m[11] - 20.25 * m[13] + 13.5 * m[14] - 27.0 * m[16] - 20.25 * m[17] + 6.75 * m[18] - 4.5 * m[21] - 13.5 * m[24] + 13.5 * m[26] - 13.5 * m[28] + 9.0 * m[30] + 13.5 * m[31] - 4.5 * m[33];
      const double K_ = Gs[0] * (-24.75 * mk[2] + 6.75 * mk[5] + 81.0 * mk[7] + 6.75 * mk[8] + 27.0 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] - 67.5 * mk[16] - 40.5 * mk[17] + 27.0 * mk[18] - 4.5 * mk[21] - 13.5 * mk[24] + 13.5 * mk[26] - 13.5 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]) + Gs[2] * (-24.75 * mk[0] + 6.75 * mk[1] + 155.25 * mk[2] + 6.75 * mk[3] + 27.0 * mk[4] - 135.0 * mk[5] + 54.0 * mk[6] - 162.0 * mk[7] - 135.0 * mk[8] + 27.0 * mk[9] - 4.5 * mk[10] + 13.5 * mk[11] - 13.5 * mk[12] + 40.5 * mk[13] + 27.0 * mk[14] - 13.5 * mk[15] + 22.5 * mk[16] + 40.5 * mk[17] + 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[7] = v_;
      out[140] = v_;
    }
    {
      const double M_ = 9.0 * m[3] - 27.0 * m[6] - 27.0 * m[8] - 27.0 * m[9] + 20.25 * m[12] + 40.5 * m[14] + 40.5 * m[15] + 20.25 * m[17] + 40.5 * m[18] + 20.25 * m[19] - 4.5 * m[22] - 13.5 * m[24] - 13.5 * m[25] - 13.5 * m[27] - 27.0 * m[28] - 13.5 * m[29] - 4.5 * m[31] - 13.5 * m[32] - 13.5 * m[33] - 4.5 * m[34];
      const double K_ = Gs[0] * (123.75 * mk[3] - 182.25 * mk[6] - 182.25 * mk[8] - 182.25 * mk[9] + 54.0 * mk[12] + 108.0 * mk[14] + 108.0 * mk[15] + 54.0 * mk[17] + 108.0 * mk[18] + 54.0 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] - 13.5 * mk[25] - 13.5 * mk[27] - 27.0 * mk[28] - 13.5 * mk[29] - 4.5 * mk[31] - 13.5 * mk[32] - 13.5 * mk[33] - 4.5 * mk[34]) + Gs[3] * (49.5 * mk[0] - 87.75 * mk[1] - 87.75 * mk[2] - 87.75 * mk[3] + 40.5 * mk[4] + 81.0 * mk[5] + 81.0 * mk[6] + 40.5 * mk[7] + 81.0 * mk[8] + 40.5 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] - 13.5 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[8] = v_;
      out[160] = v_;
    }
    {
      const double M_ = -4.5 * m[3] + 6.75 * m[6] + 6.75 * m[8] + 20.25 * m[9] + 6.75 * m[12] + 13.5 * m[14] - 20.25 * m[15] + 6.75 * m[17] - 20.25 * m[18] - 27.0 * m[19] - 4.5 * m[22] - 13.5 * m[24] - 13.5 * m[27] + 13.5 * m[29] - 4.5 * m[31] + 13.5 * m[33] + 9.0 * m[34];
      const double K_ = Gs[0] * (-24.75 * mk[3] + 6.75 * mk[6] + 6.75 * mk[8] + 81.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] + 27.0 * mk[17] - 40.5 * mk[18] - 67.5 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] - 13.5 * mk[27] + 13.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[3] * (-24.75 * mk[0] + 6.75 * mk[1] + 6.75 * mk[2] + 155.25 * mk[3] + 27.0 * mk[4] + 54.0 * mk[5] - 135.0 * mk[6] + 27.0 * mk[7] - 135.0 * mk[8] - 162.0 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] + 13.5 * mk[12] - 13.5 * mk[13] + 27.0 * mk[14] + 40.5 * mk[15] - 4.5 * mk[16] + 13.5 * mk[17] + 40.5 * mk[18] + 22.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[9] = v_;
      out[180] = v_;
    }
    {
      const double M_ = -4.5 * m[5] + 20.25 * m[11] + 6.75 * m[13] + 6.75 * m[14] - 27.0 * m[21] - 20.25 * m[23] - 20.25 * m[24] + 6.75 * m[26] + 13.5 * m[27] + 6.75 * m[28] + 9.0 * m[36] + 13.5 * m[38] + 13.5 * m[39] - 4.5 * m[45] - 13.5 * m[46] - 13.5 * m[47] - 4.5 * m[48];
      const double K_ = Gs[1] * (-24.75 * mk[2] + 155.25 * mk[5] + 6.75 * mk[7] + 6.75 * mk[8] - 162.0 * mk[11] - 135.0 * mk[13] - 135.0 * mk[14] + 27.0 * mk[16] + 54.0 * mk[17] + 27.0 * mk[18] + 22.5 * mk[21] + 40.5 * mk[23] + 40.5 * mk[24] + 13.5 * mk[26] + 27.0 * mk[27] + 13.5 * mk[28] - 4.5 * mk[30] - 13.5 * mk[31] - 13.5 * mk[32] - 4.5 * mk[33]) + Gs[2] * (-24.75 * mk[1] + 81.0 * mk[4] + 6.75 * mk[5] + 6.75 * mk[6] - 67.5 * mk[10] - 40.5 * mk[11] - 40.5 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] + 13.5 * mk[22] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[10] = v_;
      out[200] = v_;
    }
    {
      const double M_ = -4.5 * m[5] + 6.75 * m[11] + 20.25 * m[13] + 6.75 * m[14] + 6.75 * m[21] - 20.25 * m[23] + 13.5 * m[24] - 27.0 * m[26] - 20.25 * m[27] + 6.75 * m[28] - 4.5 * m[36] - 13.5 * m[39] + 13.5 * m[41] - 13.5 * m[43] + 9.0 * m[45] + 13.5 * m[46] - 4.5 * m[48];
      const double K_ = Gs[1] * (-24.75 * mk[2] + 6.75 * mk[5] + 81.0 * mk[7] + 6.75 * mk[8] + 27.0 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] - 67.5 * mk[16] - 40.5 * mk[17] + 27.0 * mk[18] - 4.5 * mk[21] - 13.5 * mk[24] + 13.5 * mk[26] - 13.5 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]) + Gs[2] * (-24.75 * mk[1] + 6.75 * mk[4] + 155.25 * mk[5] + 6.75 * mk[6] + 27.0 * mk[10] - 135.0 * mk[11] + 54.0 * mk[12] - 162.0 * mk[13] - 135.0 * mk[14] + 27.0 * mk[15] - 4.5 * mk[20] + 13.5 * mk[21] - 13.5 * mk[22] + 40.5 * mk[23] + 27.0 * mk[24] - 13.5 * mk[25] + 22.5 * mk[26] + 40.5 * mk[27] + 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[11] = v_;
      out[220] = v_;
    }
    {
      const double M_ = -4.5 * m[6] + 20.25 * m[12] + 6.75 * m[14] + 6.75 * m[15] - 27.0 * m[22] - 20.25 * m[24] - 20.25 * m[25] + 6.75 * m[27] + 13.5 * m[28] + 6.75 * m[29] + 9.0 * m[37] + 13.5 * m[39] + 13.5 * m[40] - 4.5 * m[46] - 13.5 * m[47] - 13.5 * m[48] - 4.5 * m[49];
      const double K_ = Gs[1] * (-24.75 * mk[3] + 155.25 * mk[6] + 6.75 * mk[8] + 6.75 * mk[9] - 162.0 * mk[12] - 135.0 * mk[14] - 135.0 * mk[15] + 27.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[19] + 22.5 * mk[22] + 40.5 * mk[24] + 40.5 * mk[25] + 13.5 * mk[27] + 27.0 * mk[28] + 13.5 * mk[29] - 4.5 * mk[31] - 13.5 * mk[32] - 13.5 * mk[33] - 4.5 * mk[34]) + Gs[3] * (-24.75 * mk[1] + 81.0 * mk[4] + 6.75 * mk[5] + 6.75 * mk[6] - 67.5 * mk[10] - 40.5 * mk[11] - 40.5 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] + 13.5 * mk[22] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[12] = v_;
      out[240] = v_;
    }
    {
      const double M_ = -4.5 * m[6] + 6.75 * m[12] + 6.75 * m[14] + 20.25 * m[15] + 6.75 * m[22] + 13.5 * m[24] - 20.25 * m[25] + 6.75 * m[27] - 20.25 * m[28] - 27.0 * m[29] - 4.5 * m[37] - 13.5 * m[39] - 13.5 * m[42] + 13.5 * m[44] - 4.5 * m[46] + 13.5 * m[48] + 9.0 * m[49];
      const double K_ = Gs[1] * (-24.75 * mk[3] + 6.75 * mk[6] + 6.75 * mk[8] + 81.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] + 27.0 * mk[17] - 40.5 * mk[18] - 67.5 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] - 13.5 * mk[27] + 13.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[3] * (-24.75 * mk[1] + 6.75 * mk[4] + 6.75 * mk[5] + 155.25 * mk[6] + 27.0 * mk[10] + 54.0 * mk[11] - 135.0 * mk[12] + 27.0 * mk[13] - 135.0 * mk[14] - 162.0 * mk[15] - 4.5 * mk[20] - 13.5 * mk[21] + 13.5 * mk[22] - 13.5 * mk[23] + 27.0 * mk[24] + 40.5 * mk[25] - 4.5 * mk[26] + 13.5 * mk[27] + 40.5 * mk[28] + 22.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[13] = v_;
      out[260] = v_;
    }
    {
      const double M_ = -4.5 * m[8] + 6.75 * m[14] + 20.25 * m[17] + 6.75 * m[18] + 6.75 * m[24] - 20.25 * m[27] + 13.5 * m[28] - 27.0 * m[31] - 20.25 * m[32] + 6.75 * m[33] - 4.5 * m[39] - 13.5 * m[43] + 13.5 * m[46] - 13.5 * m[48] + 9.0 * m[51] + 13.5 * m[52] - 4.5 * m[54];
      const double K_ = Gs[2] * (-24.75 * mk[3] + 6.75 * mk[6] + 155.25 * mk[8] + 6.75 * mk[9] + 27.0 * mk[12] - 135.0 * mk[14] + 54.0 * mk[15] - 162.0 * mk[17] - 135.0 * mk[18] + 27.0 * mk[19] - 4.5 * mk[22] + 13.5 * mk[24] - 13.5 * mk[25] + 40.5 * mk[27] + 27.0 * mk[28] - 13.5 * mk[29] + 22.5 * mk[31] + 40.5 * mk[32] + 13.5 * mk[33] - 4.5 * mk[34]) + Gs[3] * (-24.75 * mk[2] + 6.75 * mk[5] + 81.0 * mk[7] + 6.75 * mk[8] + 27.0 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] - 67.5 * mk[16] - 40.5 * mk[17] + 27.0 * mk[18] - 4.5 * mk[21] - 13.5 * mk[24] + 13.5 * mk[26] - 13.5 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[14] = v_;
      out[280] = v_;
    }
    {
      const double M_ = -4.5 * m[8] + 6.75 * m[14] + 6.75 * m[17] + 20.25 * m[18] + 6.75 * m[24] + 13.5 * m[27] - 20.25 * m[28] + 6.75 * m[31] - 20.25 * m[32] - 27.0 * m[33] - 4.5 * m[39] - 13.5 * m[42] - 13.5 * m[46] + 13.5 * m[48] - 4.5 * m[51] + 13.5 * m[53] + 9.0 * m[54];
      const double K_ = Gs[2] * (-24.75 * mk[3] + 6.75 * mk[6] + 6.75 * mk[8] + 81.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] + 27.0 * mk[17] - 40.5 * mk[18] - 67.5 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] - 13.5 * mk[27] + 13.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[3] * (-24.75 * mk[2] + 6.75 * mk[5] + 6.75 * mk[7] + 155.25 * mk[8] + 27.0 * mk[11] + 54.0 * mk[13] - 135.0 * mk[14] + 27.0 * mk[16] - 135.0 * mk[17] - 162.0 * mk[18] - 4.5 * mk[21] - 13.5 * mk[23] + 13.5 * mk[24] - 13.5 * mk[26] + 27.0 * mk[27] + 40.5 * mk[28] - 4.5 * mk[30] + 13.5 * mk[31] + 40.5 * mk[32] + 22.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[15] = v_;
      out[300] = v_;
    }
    {
      const double M_ = 27.0 * m[5] - 67.5 * m[11] - 67.5 * m[13] - 67.5 * m[14] + 27.0 * m[21] + 54.0 * m[23] + 54.0 * m[24] + 27.0 * m[26] + 54.0 * m[27] + 27.0 * m[28];
      const double K_ = Gs[0] * (148.5 * mk[5] - 189.0 * mk[11] - 189.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[21] + 54.0 * mk[23] + 54.0 * mk[24] + 27.0 * mk[26] + 54.0 * mk[27] + 27.0 * mk[28]) + Gs[1] * (148.5 * mk[2] - 189.0 * mk[5] - 189.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] + 54.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[16] + 54.0 * mk[17] + 27.0 * mk[18]) + Gs[2] * (148.5 * mk[1] - 189.0 * mk[4] - 189.0 * mk[5] - 189.0 * mk[6] + 27.0 * mk[10] + 54.0 * mk[11] + 54.0 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[16] = v_;
      out[320] = v_;
    }
    {
      const double M_ = 27.0 * m[6] - 67.5 * m[12] - 67.5 * m[14] - 67.5 * m[15] + 27.0 * m[22] + 54.0 * m[24] + 54.0 * m[25] + 27.0 * m[27] + 54.0 * m[28] + 27.0 * m[29];
      const double K_ = Gs[0] * (148.5 * mk[6] - 189.0 * mk[12] - 189.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[22] + 54.0 * mk[24] + 54.0 * mk[25] + 27.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[29]) + Gs[1] * (148.5 * mk[3] - 189.0 * mk[6] - 189.0 * mk[8] - 189.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] + 54.0 * mk[15] + 27.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[19]) + Gs[3] * (148.5 * mk[1] - 189.0 * mk[4] - 189.0 * mk[5] - 189.0 * mk[6] + 27.0 * mk[10] + 54.0 * mk[11] + 54.0 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[17] = v_;
      out[340] = v_;
    }
    {
      const double M_ = 27.0 * m[8] - 67.5 * m[14] - 67.5 * m[17] - 67.5 * m[18] + 27.0 * m[24] + 54.0 * m[27] + 54.0 * m[28] + 27.0 * m[31] + 54.0 * m[32] + 27.0 * m[33];
      const double K_ = Gs[0] * (148.5 * mk[8] - 189.0 * mk[14] - 189.0 * mk[17] - 189.0 * mk[18] + 27.0 * mk[24] + 54.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[31] + 54.0 * mk[32] + 27.0 * mk[33]) + Gs[2] * (148.5 * mk[3] - 189.0 * mk[6] - 189.0 * mk[8] - 189.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] + 54.0 * mk[15] + 27.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[19]) + Gs[3] * (148.5 * mk[2] - 189.0 * mk[5] - 189.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] + 54.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[16] + 54.0 * mk[17] + 27.0 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[18] = v_;
      out[360] = v_;
    }
    {
      const double M_ = 27.0 * m[14] - 67.5 * m[24] - 67.5 * m[27] - 67.5 * m[28] + 27.0 * m[39] + 54.0 * m[42] + 54.0 * m[43] + 27.0 * m[46] + 54.0 * m[47] + 27.0 * m[48];
      const double K_ = Gs[1] * (148.5 * mk[8] - 189.0 * mk[14] - 189.0 * mk[17] - 189.0 * mk[18] + 27.0 * mk[24] + 54.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[31] + 54.0 * mk[32] + 27.0 * mk[33]) + Gs[2] * (148.5 * mk[6] - 189.0 * mk[12] - 189.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[22] + 54.0 * mk[24] + 54.0 * mk[25] + 27.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[29]) + Gs[3] * (148.5 * mk[5] - 189.0 * mk[11] - 189.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[21] + 54.0 * mk[23] + 54.0 * mk[24] + 27.0 * mk[26] + 54.0 * mk[27] + 27.0 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[19] = v_;
      out[380] = v_;
    }
    {
      const double M_ = m[4] - 5.0 * m[10] + 4.0 * m[11] + 4.0 * m[12] + 8.25 * m[20] - 15.0 * m[21] - 15.0 * m[22] + 6.0 * m[23] + 12.0 * m[24] + 6.0 * m[25] - 5.0 * m[35] + 16.5 * m[36] + 16.5 * m[37] - 15.0 * m[38] - 30.0 * m[39] - 15.0 * m[40] + 4.0 * m[41] + 12.0 * m[42] + 12.0 * m[43] + 4.0 * m[44] + m[56] - 5.0 * m[57] - 5.0 * m[58] + 8.25 * m[59] + 16.5 * m[60] + 8.25 * m[61] - 5.0 * m[62] - 15.0 * m[63] - 15.0 * m[64] - 5.0 * m[65] + m[66] + 4.0 * m[67] + 6.0 * m[68] + 4.0 * m[69] + m[70];
      const double K_ = Gs[4] * (mk[0] - 14.0 * mk[1] + 4.0 * mk[2] + 4.0 * mk[3] + 60.0 * mk[4] - 42.0 * mk[5] - 42.0 * mk[6] + 6.0 * mk[7] + 12.0 * mk[8] + 6.0 * mk[9] - 77.0 * mk[10] + 120.0 * mk[11] + 120.0 * mk[12] - 42.0 * mk[13] - 84.0 * mk[14] - 42.0 * mk[15] + 4.0 * mk[16] + 12.0 * mk[17] + 12.0 * mk[18] + 4.0 * mk[19] + 30.25 * mk[20] - 77.0 * mk[21] - 77.0 * mk[22] + 60.0 * mk[23] + 120.0 * mk[24] + 60.0 * mk[25] - 14.0 * mk[26] - 42.0 * mk[27] - 42.0 * mk[28] - 14.0 * mk[29] + mk[30] + 4.0 * mk[31] + 6.0 * mk[32] + 4.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[21] = v_;
    }
    {
      const double M_ = m[5] - 0.5 * m[11] - 0.5 * m[13] + 4.0 * m[14] - 3.0 * m[21] + 5.25 * m[23] - 1.5 * m[24] - 3.0 * m[26] - 1.5 * m[27] + 6.0 * m[28] - 0.5 * m[36] + 0.75 * m[38] - 6.0 * m[39] + 0.75 * m[41] + 10.5 * m[42] - 1.5 * m[43] - 0.5 * m[45] - 6.0 * m[46] - 1.5 * m[47] + 4.0 * m[48] + m[57] - 5.0 * m[59] - 0.5 * m[60] + 8.25 * m[62] + 0.75 * m[63] - 3.0 * m[64] - 5.0 * m[66] + 0.75 * m[67] + 5.25 * m[68] - 0.5 * m[69] + m[71] - 0.5 * m[72] - 3.0 * m[73] - 0.5 * m[74] + m[75];
      const double K_ = Gs[5] * (mk[0] - 5.0 * mk[1] - 5.0 * mk[2] + 4.0 * mk[3] - 7.5 * mk[4] + 39.0 * mk[5] - 15.0 * mk[6] - 7.5 * mk[7] - 15.0 * mk[8] + 6.0 * mk[9] + 4.0 * mk[10] - 1.5 * mk[11] - 15.0 * mk[12] - 1.5 * mk[13] + 78.0 * mk[14] - 15.0 * mk[15] + 4.0 * mk[16] - 15.0 * mk[17] - 15.0 * mk[18] + 4.0 * mk[19] + 5.5 * mk[20] - 45.5 * mk[21] + 4.0 * mk[22] + 80.25 * mk[23] - 1.5 * mk[24] - 7.5 * mk[25] - 45.5 * mk[26] - 1.5 * mk[27] + 39.0 * mk[28] - 5.0 * mk[29] + 5.5 * mk[30] + 4.0 * mk[31] - 7.5 * mk[32] - 5.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[22] = v_;
      out[41] = v_;
    }
    {
      const double M_ = m[6] - 0.5 * m[12] + 4.0 * m[14] - 0.5 * m[15] - 3.0 * m[22] - 1.5 * m[24] + 5.25 * m[25] + 6.0 * m[27] - 1.5 * m[28] - 3.0 * m[29] - 0.5 * m[37] - 6.0 * m[39] + 0.75 * m[40] - 1.5 * m[42] + 10.5 * m[43] + 0.75 * m[44] + 4.0 * m[46] - 1.5 * m[47] - 6.0 * m[48] - 0.5 * m[49] + m[58] - 0.5 * m[60] - 5.0 * m[61] - 3.0 * m[63] + 0.75 * m[64] + 8.25 * m[65] - 0.5 * m[67] + 5.25 * m[68] + 0.75 * m[69] - 5.0 * m[70] + m[72] - 0.5 * m[73] - 3.0 * m[74] - 0.5 * m[75] + m[76];
      const double K_ = Gs[6] * (mk[0] - 5.0 * mk[1] + 4.0 * mk[2] - 5.0 * mk[3] - 7.5 * mk[4] - 15.0 * mk[5] + 39.0 * mk[6] + 6.0 * mk[7] - 15.0 * mk[8] - 7.5 * mk[9] + 4.0 * mk[10] - 15.0 * mk[11] - 1.5 * mk[12] - 15.0 * mk[13] + 78.0 * mk[14] - 1.5 * mk[15] + 4.0 * mk[16] - 15.0 * mk[17] - 15.0 * mk[18] + 4.0 * mk[19] + 5.5 * mk[20] + 4.0 * mk[21] - 45.5 * mk[22] - 7.5 * mk[23] - 1.5 * mk[24] + 80.25 * mk[25] - 5.0 * mk[26] + 39.0 * mk[27] - 1.5 * mk[28] - 45.5 * mk[29] + mk[30] - 5.0 * mk[31] - 7.5 * mk[32] + 4.0 * mk[33] + 5.5 * mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[23] = v_;
      out[61] = v_;
    }
    {
      const double M_ = 9.0 * m[4] - 27.0 * m[10] + 13.5 * m[11] + 13.5 * m[12] + 20.25 * m[20] - 20.25 * m[21] - 20.25 * m[22] - 4.5 * m[35] + 6.75 * m[36] + 6.75 * m[37] + 6.75 * m[38] + 13.5 * m[39] + 6.75 * m[40] - 4.5 * m[41] - 13.5 * m[42] - 13.5 * m[43] - 4.5 * m[44];
      const double K_ = Gs[1] * (22.5 * mk[1] - 162.0 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 155.25 * mk[10] - 135.0 * mk[11] - 135.0 * mk[12] + 13.5 * mk[13] + 27.0 * mk[14] + 13.5 * mk[15] - 24.75 * mk[20] + 6.75 * mk[21] + 6.75 * mk[22] + 27.0 * mk[23] + 54.0 * mk[24] + 27.0 * mk[25] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]) + Gs[4] * (9.0 * mk[0] - 67.5 * mk[1] + 13.5 * mk[2] + 13.5 * mk[3] + 81.0 * mk[4] - 40.5 * mk[5] - 40.5 * mk[6] - 24.75 * mk[10] + 6.75 * mk[11] + 6.75 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[24] = v_;
      out[81] = v_;
    }
    {
      const double M_ = -4.5 * m[4] + 20.25 * m[10] - 13.5 * m[11] - 13.5 * m[12] - 27.0 * m[20] + 40.5 * m[21] + 40.5 * m[22] - 13.5 * m[23] - 27.0 * m[24] - 13.5 * m[25] + 9.0 * m[35] - 27.0 * m[36] - 27.0 * m[37] + 20.25 * m[38] + 40.5 * m[39] + 20.25 * m[40] - 4.5 * m[41] - 13.5 * m[42] - 13.5 * m[43] - 4.5 * m[44];
      const double K_ = Gs[1] * (-4.5 * mk[1] + 40.5 * mk[4] - 13.5 * mk[5] - 13.5 * mk[6] - 87.75 * mk[10] + 81.0 * mk[11] + 81.0 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] + 49.5 * mk[20] - 87.75 * mk[21] - 87.75 * mk[22] + 40.5 * mk[23] + 81.0 * mk[24] + 40.5 * mk[25] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]) + Gs[4] * (-4.5 * mk[0] + 54.0 * mk[1] - 13.5 * mk[2] - 13.5 * mk[3] - 182.25 * mk[4] + 108.0 * mk[5] + 108.0 * mk[6] - 13.5 * mk[7] - 27.0 * mk[8] - 13.5 * mk[9] + 123.75 * mk[10] - 182.25 * mk[11] - 182.25 * mk[12] + 54.0 * mk[13] + 108.0 * mk[14] + 54.0 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[25] = v_;
      out[101] = v_;
    }
    {
      const double M_ = 9.0 * m[5] - 27.0 * m[11] + 13.5 * m[13] + 13.5 * m[14] + 20.25 * m[21] - 20.25 * m[23] - 20.25 * m[24] - 4.5 * m[36] + 6.75 * m[38] + 6.75 * m[39] + 6.75 * m[41] + 13.5 * m[42] + 6.75 * m[43] - 4.5 * m[45] - 13.5 * m[46] - 13.5 * m[47] - 4.5 * m[48];
      const double K_ = Gs[1] * (22.5 * mk[2] - 162.0 * mk[5] + 40.5 * mk[7] + 40.5 * mk[8] + 155.25 * mk[11] - 135.0 * mk[13] - 135.0 * mk[14] + 13.5 * mk[16] + 27.0 * mk[17] + 13.5 * mk[18] - 24.75 * mk[21] + 6.75 * mk[23] + 6.75 * mk[24] + 27.0 * mk[26] + 54.0 * mk[27] + 27.0 * mk[28] - 4.5 * mk[30] - 13.5 * mk[31] - 13.5 * mk[32] - 4.5 * mk[33]) + Gs[5] * (9.0 * mk[0] - 67.5 * mk[1] + 13.5 * mk[2] + 13.5 * mk[3] + 81.0 * mk[4] - 40.5 * mk[5] - 40.5 * mk[6] - 24.75 * mk[10] + 6.75 * mk[11] + 6.75 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[26] = v_;
      out[121] = v_;
    }
    {
      const double M_ = -4.5 * m[5] + 6.75 * m[11] - 13.5 * m[14] + 6.75 * m[21] - 20.25 * m[23] + 13.5 * m[24] + 13.5 * m[26] - 13.5 * m[28] - 4.5 * m[36] + 20.25 * m[38] + 6.75 * m[39] - 27.0 * m[41] - 20.25 * m[42] + 6.75 * m[43] + 9.0 * m[45] + 13.5 * m[46] - 4.5 * m[48];
      const double K_ = Gs[1] * (-4.5 * mk[2] + 27.0 * mk[5] - 13.5 * mk[8] + 6.75 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] + 13.5 * mk[16] - 13.5 * mk[18] - 24.75 * mk[21] + 81.0 * mk[23] + 6.75 * mk[24] - 67.5 * mk[26] - 40.5 * mk[27] + 27.0 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]) + Gs[5] * (-4.5 * mk[0] + 27.0 * mk[1] + 13.5 * mk[2] - 13.5 * mk[3] + 6.75 * mk[4] - 135.0 * mk[5] + 54.0 * mk[6] + 40.5 * mk[7] + 27.0 * mk[8] - 13.5 * mk[9] - 24.75 * mk[10] + 155.25 * mk[11] + 6.75 * mk[12] - 162.0 * mk[13] - 135.0 * mk[14] + 27.0 * mk[15] + 22.5 * mk[16] + 40.5 * mk[17] + 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[27] = v_;
      out[141] = v_;
    }
    {
      const double M_ = 9.0 * m[6] - 27.0 * m[12] + 13.5 * m[14] + 13.5 * m[15] + 20.25 * m[22] - 20.25 * m[24] - 20.25 * m[25] - 4.5 * m[37] + 6.75 * m[39] + 6.75 * m[40] + 6.75 * m[42] + 13.5 * m[43] + 6.75 * m[44] - 4.5 * m[46] - 13.5 * m[47] - 13.5 * m[48] - 4.5 * m[49];
      const double K_ = Gs[1] * (22.5 * mk[3] - 162.0 * mk[6] + 40.5 * mk[8] + 40.5 * mk[9] + 155.25 * mk[12] - 135.0 * mk[14] - 135.0 * mk[15] + 13.5 * mk[17] + 27.0 * mk[18] + 13.5 * mk[19] - 24.75 * mk[22] + 6.75 * mk[24] + 6.75 * mk[25] + 27.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[29] - 4.5 * mk[31] - 13.5 * mk[32] - 13.5 * mk[33] - 4.5 * mk[34]) + Gs[6] * (9.0 * mk[0] - 67.5 * mk[1] + 13.5 * mk[2] + 13.5 * mk[3] + 81.0 * mk[4] - 40.5 * mk[5] - 40.5 * mk[6] - 24.75 * mk[10] + 6.75 * mk[11] + 6.75 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15] - 4.5 * mk[16] - 13.5 * mk[17] - 13.5 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[28] = v_;
      out[161] = v_;
    }
    {
      const double M_ = -4.5 * m[6] + 6.75 * m[12] - 13.5 * m[14] + 6.75 * m[22] + 13.5 * m[24] - 20.25 * m[25] - 13.5 * m[27] + 13.5 * m[29] - 4.5 * m[37] + 6.75 * m[39] + 20.25 * m[40] + 6.75 * m[42] - 20.25 * m[43] - 27.0 * m[44] - 4.5 * m[46] + 13.5 * m[48] + 9.0 * m[49];
      const double K_ = Gs[1] * (-4.5 * mk[3] + 27.0 * mk[6] - 13.5 * mk[8] + 6.75 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] - 13.5 * mk[17] + 13.5 * mk[19] - 24.75 * mk[22] + 6.75 * mk[24] + 81.0 * mk[25] + 27.0 * mk[27] - 40.5 * mk[28] - 67.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[6] * (-4.5 * mk[0] + 27.0 * mk[1] - 13.5 * mk[2] + 13.5 * mk[3] + 6.75 * mk[4] + 54.0 * mk[5] - 135.0 * mk[6] - 13.5 * mk[7] + 27.0 * mk[8] + 40.5 * mk[9] - 24.75 * mk[10] + 6.75 * mk[11] + 155.25 * mk[12] + 27.0 * mk[13] - 135.0 * mk[14] - 162.0 * mk[15] - 4.5 * mk[16] + 13.5 * mk[17] + 40.5 * mk[18] + 22.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[29] = v_;
      out[181] = v_;
    }
    {
      const double M_ = -4.5 * m[11] + 20.25 * m[21] - 13.5 * m[23] - 13.5 * m[24] - 27.0 * m[36] + 40.5 * m[38] + 40.5 * m[39] - 13.5 * m[41] - 27.0 * m[42] - 13.5 * m[43] + 9.0 * m[57] - 27.0 * m[59] - 27.0 * m[60] + 20.25 * m[62] + 40.5 * m[63] + 20.25 * m[64] - 4.5 * m[66] - 13.5 * m[67] - 13.5 * m[68] - 4.5 * m[69];
      const double K_ = Gs[4] * (-4.5 * mk[2] + 54.0 * mk[5] - 13.5 * mk[7] - 13.5 * mk[8] - 182.25 * mk[11] + 108.0 * mk[13] + 108.0 * mk[14] - 13.5 * mk[16] - 27.0 * mk[17] - 13.5 * mk[18] + 123.75 * mk[21] - 182.25 * mk[23] - 182.25 * mk[24] + 54.0 * mk[26] + 108.0 * mk[27] + 54.0 * mk[28] - 4.5 * mk[30] - 13.5 * mk[31] - 13.5 * mk[32] - 4.5 * mk[33]) + Gs[5] * (-4.5 * mk[1] + 40.5 * mk[4] - 13.5 * mk[5] - 13.5 * mk[6] - 87.75 * mk[10] + 81.0 * mk[11] + 81.0 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] + 49.5 * mk[20] - 87.75 * mk[21] - 87.75 * mk[22] + 40.5 * mk[23] + 81.0 * mk[24] + 40.5 * mk[25] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[30] = v_;
      out[201] = v_;
    }
    {
      const double M_ = -4.5 * m[11] + 6.75 * m[21] - 13.5 * m[24] + 6.75 * m[36] - 20.25 * m[38] + 13.5 * m[39] + 13.5 * m[41] - 13.5 * m[43] - 4.5 * m[57] + 20.25 * m[59] + 6.75 * m[60] - 27.0 * m[62] - 20.25 * m[63] + 6.75 * m[64] + 9.0 * m[66] + 13.5 * m[67] - 4.5 * m[69];
      const double K_ = Gs[4] * (-4.5 * mk[2] + 27.0 * mk[5] - 13.5 * mk[8] + 6.75 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] + 13.5 * mk[16] - 13.5 * mk[18] - 24.75 * mk[21] + 81.0 * mk[23] + 6.75 * mk[24] - 67.5 * mk[26] - 40.5 * mk[27] + 27.0 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]) + Gs[5] * (-4.5 * mk[1] + 27.0 * mk[4] + 13.5 * mk[5] - 13.5 * mk[6] + 6.75 * mk[10] - 135.0 * mk[11] + 54.0 * mk[12] + 40.5 * mk[13] + 27.0 * mk[14] - 13.5 * mk[15] - 24.75 * mk[20] + 155.25 * mk[21] + 6.75 * mk[22] - 162.0 * mk[23] - 135.0 * mk[24] + 27.0 * mk[25] + 22.5 * mk[26] + 40.5 * mk[27] + 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[31] = v_;
      out[221] = v_;
    }
    {
      const double M_ = -4.5 * m[12] + 20.25 * m[22] - 13.5 * m[24] - 13.5 * m[25] - 27.0 * m[37] + 40.5 * m[39] + 40.5 * m[40] - 13.5 * m[42] - 27.0 * m[43] - 13.5 * m[44] + 9.0 * m[58] - 27.0 * m[60] - 27.0 * m[61] + 20.25 * m[63] + 40.5 * m[64] + 20.25 * m[65] - 4.5 * m[67] - 13.5 * m[68] - 13.5 * m[69] - 4.5 * m[70];
      const double K_ = Gs[4] * (-4.5 * mk[3] + 54.0 * mk[6] - 13.5 * mk[8] - 13.5 * mk[9] - 182.25 * mk[12] + 108.0 * mk[14] + 108.0 * mk[15] - 13.5 * mk[17] - 27.0 * mk[18] - 13.5 * mk[19] + 123.75 * mk[22] - 182.25 * mk[24] - 182.25 * mk[25] + 54.0 * mk[27] + 108.0 * mk[28] + 54.0 * mk[29] - 4.5 * mk[31] - 13.5 * mk[32] - 13.5 * mk[33] - 4.5 * mk[34]) + Gs[6] * (-4.5 * mk[1] + 40.5 * mk[4] - 13.5 * mk[5] - 13.5 * mk[6] - 87.75 * mk[10] + 81.0 * mk[11] + 81.0 * mk[12] - 13.5 * mk[13] - 27.0 * mk[14] - 13.5 * mk[15] + 49.5 * mk[20] - 87.75 * mk[21] - 87.75 * mk[22] + 40.5 * mk[23] + 81.0 * mk[24] + 40.5 * mk[25] - 4.5 * mk[26] - 13.5 * mk[27] - 13.5 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[32] = v_;
      out[241] = v_;
    }
    {
      const double M_ = -4.5 * m[12] + 6.75 * m[22] - 13.5 * m[24] + 6.75 * m[37] + 13.5 * m[39] - 20.25 * m[40] - 13.5 * m[42] + 13.5 * m[44] - 4.5 * m[58] + 6.75 * m[60] + 20.25 * m[61] + 6.75 * m[63] - 20.25 * m[64] - 27.0 * m[65] - 4.5 * m[67] + 13.5 * m[69] + 9.0 * m[70];
      const double K_ = Gs[4] * (-4.5 * mk[3] + 27.0 * mk[6] - 13.5 * mk[8] + 6.75 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] - 13.5 * mk[17] + 13.5 * mk[19] - 24.75 * mk[22] + 6.75 * mk[24] + 81.0 * mk[25] + 27.0 * mk[27] - 40.5 * mk[28] - 67.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[6] * (-4.5 * mk[1] + 27.0 * mk[4] - 13.5 * mk[5] + 13.5 * mk[6] + 6.75 * mk[10] + 54.0 * mk[11] - 135.0 * mk[12] - 13.5 * mk[13] + 27.0 * mk[14] + 40.5 * mk[15] - 24.75 * mk[20] + 6.75 * mk[21] + 155.25 * mk[22] + 27.0 * mk[23] - 135.0 * mk[24] - 162.0 * mk[25] - 4.5 * mk[26] + 13.5 * mk[27] + 40.5 * mk[28] + 22.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[33] = v_;
      out[261] = v_;
    }
    {
      const double M_ = -4.5 * m[14] + 6.75 * m[24] - 13.5 * m[28] + 6.75 * m[39] - 20.25 * m[42] + 13.5 * m[43] + 13.5 * m[46] - 13.5 * m[48] - 4.5 * m[60] + 20.25 * m[63] + 6.75 * m[64] - 27.0 * m[67] - 20.25 * m[68] + 6.75 * m[69] + 9.0 * m[72] + 13.5 * m[73] - 4.5 * m[75];
      const double K_ = Gs[5] * (-4.5 * mk[3] + 27.0 * mk[6] + 13.5 * mk[8] - 13.5 * mk[9] + 6.75 * mk[12] - 135.0 * mk[14] + 54.0 * mk[15] + 40.5 * mk[17] + 27.0 * mk[18] - 13.5 * mk[19] - 24.75 * mk[22] + 155.25 * mk[24] + 6.75 * mk[25] - 162.0 * mk[27] - 135.0 * mk[28] + 27.0 * mk[29] + 22.5 * mk[31] + 40.5 * mk[32] + 13.5 * mk[33] - 4.5 * mk[34]) + Gs[6] * (-4.5 * mk[2] + 27.0 * mk[5] - 13.5 * mk[8] + 6.75 * mk[11] - 40.5 * mk[13] + 54.0 * mk[14] + 13.5 * mk[16] - 13.5 * mk[18] - 24.75 * mk[21] + 81.0 * mk[23] + 6.75 * mk[24] - 67.5 * mk[26] - 40.5 * mk[27] + 27.0 * mk[28] + 9.0 * mk[30] + 13.5 * mk[31] - 4.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[34] = v_;
      out[281] = v_;
    }
    {
      const double M_ = -4.5 * m[14] + 6.75 * m[24] - 13.5 * m[27] + 6.75 * m[39] + 13.5 * m[42] - 20.25 * m[43] - 13.5 * m[46] + 13.5 * m[48] - 4.5 * m[60] + 6.75 * m[63] + 20.25 * m[64] + 6.75 * m[67] - 20.25 * m[68] - 27.0 * m[69] - 4.5 * m[72] + 13.5 * m[74] + 9.0 * m[75];
      const double K_ = Gs[5] * (-4.5 * mk[3] + 27.0 * mk[6] - 13.5 * mk[8] + 6.75 * mk[12] + 54.0 * mk[14] - 40.5 * mk[15] - 13.5 * mk[17] + 13.5 * mk[19] - 24.75 * mk[22] + 6.75 * mk[24] + 81.0 * mk[25] + 27.0 * mk[27] - 40.5 * mk[28] - 67.5 * mk[29] - 4.5 * mk[31] + 13.5 * mk[33] + 9.0 * mk[34]) + Gs[6] * (-4.5 * mk[2] + 27.0 * mk[5] - 13.5 * mk[7] + 13.5 * mk[8] + 6.75 * mk[11] + 54.0 * mk[13] - 135.0 * mk[14] - 13.5 * mk[16] + 27.0 * mk[17] + 40.5 * mk[18] - 24.75 * mk[21] + 6.75 * mk[23] + 155.25 * mk[24] + 27.0 * mk[26] - 135.0 * mk[27] - 162.0 * mk[28] - 4.5 * mk[30] + 13.5 * mk[31] + 40.5 * mk[32] + 22.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[35] = v_;
      out[301] = v_;
    }
    {
      const double M_ = 27.0 * m[11] - 67.5 * m[21] + 54.0 * m[23] + 54.0 * m[24] + 27.0 * m[36] - 67.5 * m[38] - 67.5 * m[39] + 27.0 * m[41] + 54.0 * m[42] + 27.0 * m[43];
      const double K_ = Gs[1] * (27.0 * mk[5] - 189.0 * mk[11] + 54.0 * mk[13] + 54.0 * mk[14] + 148.5 * mk[21] - 189.0 * mk[23] - 189.0 * mk[24] + 27.0 * mk[26] + 54.0 * mk[27] + 27.0 * mk[28]) + Gs[4] * (27.0 * mk[2] - 189.0 * mk[5] + 54.0 * mk[7] + 54.0 * mk[8] + 148.5 * mk[11] - 189.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[16] + 54.0 * mk[17] + 27.0 * mk[18]) + Gs[5] * (27.0 * mk[1] - 189.0 * mk[4] + 54.0 * mk[5] + 54.0 * mk[6] + 148.5 * mk[10] - 189.0 * mk[11] - 189.0 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[36] = v_;
      out[321] = v_;
    }
    {
      const double M_ = 27.0 * m[12] - 67.5 * m[22] + 54.0 * m[24] + 54.0 * m[25] + 27.0 * m[37] - 67.5 * m[39] - 67.5 * m[40] + 27.0 * m[42] + 54.0 * m[43] + 27.0 * m[44];
      const double K_ = Gs[1] * (27.0 * mk[6] - 189.0 * mk[12] + 54.0 * mk[14] + 54.0 * mk[15] + 148.5 * mk[22] - 189.0 * mk[24] - 189.0 * mk[25] + 27.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[29]) + Gs[4] * (27.0 * mk[3] - 189.0 * mk[6] + 54.0 * mk[8] + 54.0 * mk[9] + 148.5 * mk[12] - 189.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[19]) + Gs[6] * (27.0 * mk[1] - 189.0 * mk[4] + 54.0 * mk[5] + 54.0 * mk[6] + 148.5 * mk[10] - 189.0 * mk[11] - 189.0 * mk[12] + 27.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[37] = v_;
      out[341] = v_;
    }
    {
      const double M_ = 27.0 * m[14] - 67.5 * m[24] + 54.0 * m[27] + 54.0 * m[28] + 27.0 * m[39] - 67.5 * m[42] - 67.5 * m[43] + 27.0 * m[46] + 54.0 * m[47] + 27.0 * m[48];
      const double K_ = Gs[1] * (27.0 * mk[8] - 189.0 * mk[14] + 54.0 * mk[17] + 54.0 * mk[18] + 148.5 * mk[24] - 189.0 * mk[27] - 189.0 * mk[28] + 27.0 * mk[31] + 54.0 * mk[32] + 27.0 * mk[33]) + Gs[5] * (27.0 * mk[3] - 189.0 * mk[6] + 54.0 * mk[8] + 54.0 * mk[9] + 148.5 * mk[12] - 189.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[19]) + Gs[6] * (27.0 * mk[2] - 189.0 * mk[5] + 54.0 * mk[7] + 54.0 * mk[8] + 148.5 * mk[11] - 189.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[16] + 54.0 * mk[17] + 27.0 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[38] = v_;
      out[361] = v_;
    }
    {
      const double M_ = 27.0 * m[24] - 67.5 * m[39] + 54.0 * m[42] + 54.0 * m[43] + 27.0 * m[60] - 67.5 * m[63] - 67.5 * m[64] + 27.0 * m[67] + 54.0 * m[68] + 27.0 * m[69];
      const double K_ = Gs[4] * (27.0 * mk[8] - 189.0 * mk[14] + 54.0 * mk[17] + 54.0 * mk[18] + 148.5 * mk[24] - 189.0 * mk[27] - 189.0 * mk[28] + 27.0 * mk[31] + 54.0 * mk[32] + 27.0 * mk[33]) + Gs[5] * (27.0 * mk[6] - 189.0 * mk[12] + 54.0 * mk[14] + 54.0 * mk[15] + 148.5 * mk[22] - 189.0 * mk[24] - 189.0 * mk[25] + 27.0 * mk[27] + 54.0 * mk[28] + 27.0 * mk[29]) + Gs[6] * (27.0 * mk[5] - 189.0 * mk[11] + 54.0 * mk[13] + 54.0 * mk[14] + 148.5 * mk[21] - 189.0 * mk[23] - 189.0 * mk[24] + 27.0 * mk[26] + 54.0 * mk[27] + 27.0 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[39] = v_;
      out[381] = v_;
    }
    {
      const double M_ = m[7] + 4.0 * m[13] - 5.0 * m[16] + 4.0 * m[17] + 6.0 * m[23] - 15.0 * m[26] + 12.0 * m[27] + 8.25 * m[30] - 15.0 * m[31] + 6.0 * m[32] + 4.0 * m[38] - 15.0 * m[41] + 12.0 * m[42] + 16.5 * m[45] - 30.0 * m[46] + 12.0 * m[47] - 5.0 * m[50] + 16.5 * m[51] - 15.0 * m[52] + 4.0 * m[53] + m[59] - 5.0 * m[62] + 4.0 * m[63] + 8.25 * m[66] - 15.0 * m[67] + 6.0 * m[68] - 5.0 * m[71] + 16.5 * m[72] - 15.0 * m[73] + 4.0 * m[74] + m[77] - 5.0 * m[78] + 8.25 * m[79] - 5.0 * m[80] + m[81];
      const double K_ = Gs[7] * (mk[0] + 4.0 * mk[1] - 14.0 * mk[2] + 4.0 * mk[3] + 6.0 * mk[4] - 42.0 * mk[5] + 12.0 * mk[6] + 60.0 * mk[7] - 42.0 * mk[8] + 6.0 * mk[9] + 4.0 * mk[10] - 42.0 * mk[11] + 12.0 * mk[12] + 120.0 * mk[13] - 84.0 * mk[14] + 12.0 * mk[15] - 77.0 * mk[16] + 120.0 * mk[17] - 42.0 * mk[18] + 4.0 * mk[19] + mk[20] - 14.0 * mk[21] + 4.0 * mk[22] + 60.0 * mk[23] - 42.0 * mk[24] + 6.0 * mk[25] - 77.0 * mk[26] + 120.0 * mk[27] - 42.0 * mk[28] + 4.0 * mk[29] + 30.25 * mk[30] - 77.0 * mk[31] + 60.0 * mk[32] - 14.0 * mk[33] + mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[42] = v_;
    }
    {
      const double M_ = m[8] + 4.0 * m[14] - 0.5 * m[17] - 0.5 * m[18] + 6.0 * m[24] - 1.5 * m[27] - 1.5 * m[28] - 3.0 * m[31] + 5.25 * m[32] - 3.0 * m[33] + 4.0 * m[39] - 1.5 * m[42] - 1.5 * m[43] - 6.0 * m[46] + 10.5 * m[47] - 6.0 * m[48] - 0.5 * m[51] + 0.75 * m[52] + 0.75 * m[53] - 0.5 * m[54] + m[60] - 0.5 * m[63] - 0.5 * m[64] - 3.0 * m[67] + 5.25 * m[68] - 3.0 * m[69] - 0.5 * m[72] + 0.75 * m[73] + 0.75 * m[74] - 0.5 * m[75] + m[78] - 5.0 * m[79] + 8.25 * m[80] - 5.0 * m[81] + m[82];
      const double K_ = Gs[8] * (mk[0] + 4.0 * mk[1] - 5.0 * mk[2] - 5.0 * mk[3] + 6.0 * mk[4] - 15.0 * mk[5] - 15.0 * mk[6] - 7.5 * mk[7] + 39.0 * mk[8] - 7.5 * mk[9] + 4.0 * mk[10] - 15.0 * mk[11] - 15.0 * mk[12] - 15.0 * mk[13] + 78.0 * mk[14] - 15.0 * mk[15] + 4.0 * mk[16] - 1.5 * mk[17] - 1.5 * mk[18] + 4.0 * mk[19] + mk[20] - 5.0 * mk[21] - 5.0 * mk[22] - 7.5 * mk[23] + 39.0 * mk[24] - 7.5 * mk[25] + 4.0 * mk[26] - 1.5 * mk[27] - 1.5 * mk[28] + 4.0 * mk[29] + 5.5 * mk[30] - 45.5 * mk[31] + 80.25 * mk[32] - 45.5 * mk[33] + 5.5 * mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[43] = v_;
      out[62] = v_;
    }
    {
      const double M_ = 9.0 * m[5] + 13.5 * m[11] - 27.0 * m[13] + 13.5 * m[14] - 20.25 * m[23] + 20.25 * m[26] - 20.25 * m[27] - 4.5 * m[36] + 6.75 * m[38] - 13.5 * m[39] + 6.75 * m[41] + 13.5 * m[42] - 13.5 * m[43] - 4.5 * m[45] + 6.75 * m[46] + 6.75 * m[47] - 4.5 * m[48];
      const double K_ = Gs[2] * (22.5 * mk[1] + 40.5 * mk[4] - 162.0 * mk[5] + 40.5 * mk[6] + 13.5 * mk[10] - 135.0 * mk[11] + 27.0 * mk[12] + 155.25 * mk[13] - 135.0 * mk[14] + 13.5 * mk[15] - 4.5 * mk[20] + 27.0 * mk[21] - 13.5 * mk[22] + 6.75 * mk[23] + 54.0 * mk[24] - 13.5 * mk[25] - 24.75 * mk[26] + 6.75 * mk[27] + 27.0 * mk[28] - 4.5 * mk[29]) + Gs[5] * (9.0 * mk[0] + 13.5 * mk[1] - 67.5 * mk[2] + 13.5 * mk[3] - 40.5 * mk[5] + 81.0 * mk[7] - 40.5 * mk[8] - 4.5 * mk[10] + 27.0 * mk[11] - 13.5 * mk[12] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] - 24.75 * mk[16] + 6.75 * mk[17] + 27.0 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[44] = v_;
      out[82] = v_;
    }
    {
      const double M_ = -4.5 * m[5] + 6.75 * m[13] - 13.5 * m[14] + 13.5 * m[21] - 20.25 * m[23] + 6.75 * m[26] + 13.5 * m[27] - 13.5 * m[28] + 9.0 * m[36] - 27.0 * m[38] + 13.5 * m[39] + 20.25 * m[41] - 20.25 * m[42] - 4.5 * m[45] + 6.75 * m[46] + 6.75 * m[47] - 4.5 * m[48];
      const double K_ = Gs[2] * (-4.5 * mk[1] + 27.0 * mk[5] - 13.5 * mk[6] + 13.5 * mk[10] - 40.5 * mk[11] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] + 9.0 * mk[20] - 67.5 * mk[21] + 13.5 * mk[22] + 81.0 * mk[23] - 40.5 * mk[24] - 24.75 * mk[26] + 6.75 * mk[27] + 27.0 * mk[28] - 4.5 * mk[29]) + Gs[5] * (-4.5 * mk[0] + 13.5 * mk[1] + 27.0 * mk[2] - 13.5 * mk[3] + 40.5 * mk[4] - 135.0 * mk[5] + 27.0 * mk[6] + 6.75 * mk[7] + 54.0 * mk[8] - 13.5 * mk[9] + 22.5 * mk[10] - 162.0 * mk[11] + 40.5 * mk[12] + 155.25 * mk[13] - 135.0 * mk[14] + 13.5 * mk[15] - 24.75 * mk[16] + 6.75 * mk[17] + 27.0 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[45] = v_;
      out[102] = v_;
    }
    {
      const double M_ = 9.0 * m[7] + 13.5 * m[13] - 27.0 * m[16] + 13.5 * m[17] - 20.25 * m[26] + 20.25 * m[30] - 20.25 * m[31] - 4.5 * m[38] + 6.75 * m[41] - 13.5 * m[42] + 6.75 * m[45] + 13.5 * m[46] - 13.5 * m[47] - 4.5 * m[50] + 6.75 * m[51] + 6.75 * m[52] - 4.5 * m[53];
      const double K_ = Gs[2] * (22.5 * mk[2] + 40.5 * mk[5] - 162.0 * mk[7] + 40.5 * mk[8] + 13.5 * mk[11] - 135.0 * mk[13] + 27.0 * mk[14] + 155.25 * mk[16] - 135.0 * mk[17] + 13.5 * mk[18] - 4.5 * mk[21] + 27.0 * mk[23] - 13.5 * mk[24] + 6.75 * mk[26] + 54.0 * mk[27] - 13.5 * mk[28] - 24.75 * mk[30] + 6.75 * mk[31] + 27.0 * mk[32] - 4.5 * mk[33]) + Gs[7] * (9.0 * mk[0] + 13.5 * mk[1] - 67.5 * mk[2] + 13.5 * mk[3] - 40.5 * mk[5] + 81.0 * mk[7] - 40.5 * mk[8] - 4.5 * mk[10] + 27.0 * mk[11] - 13.5 * mk[12] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] - 24.75 * mk[16] + 6.75 * mk[17] + 27.0 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[46] = v_;
      out[122] = v_;
    }
    {
      const double M_ = -4.5 * m[7] - 13.5 * m[13] + 20.25 * m[16] - 13.5 * m[17] - 13.5 * m[23] + 40.5 * m[26] - 27.0 * m[27] - 27.0 * m[30] + 40.5 * m[31] - 13.5 * m[32] - 4.5 * m[38] + 20.25 * m[41] - 13.5 * m[42] - 27.0 * m[45] + 40.5 * m[46] - 13.5 * m[47] + 9.0 * m[50] - 27.0 * m[51] + 20.25 * m[52] - 4.5 * m[53];
      const double K_ = Gs[2] * (-4.5 * mk[2] - 13.5 * mk[5] + 40.5 * mk[7] - 13.5 * mk[8] - 13.5 * mk[11] + 81.0 * mk[13] - 27.0 * mk[14] - 87.75 * mk[16] + 81.0 * mk[17] - 13.5 * mk[18] - 4.5 * mk[21] + 40.5 * mk[23] - 13.5 * mk[24] - 87.75 * mk[26] + 81.0 * mk[27] - 13.5 * mk[28] + 49.5 * mk[30] - 87.75 * mk[31] + 40.5 * mk[32] - 4.5 * mk[33]) + Gs[7] * (-4.5 * mk[0] - 13.5 * mk[1] + 54.0 * mk[2] - 13.5 * mk[3] - 13.5 * mk[4] + 108.0 * mk[5] - 27.0 * mk[6] - 182.25 * mk[7] + 108.0 * mk[8] - 13.5 * mk[9] - 4.5 * mk[10] + 54.0 * mk[11] - 13.5 * mk[12] - 182.25 * mk[13] + 108.0 * mk[14] - 13.5 * mk[15] + 123.75 * mk[16] - 182.25 * mk[17] + 54.0 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[47] = v_;
      out[142] = v_;
    }
    {
      const double M_ = 9.0 * m[8] + 13.5 * m[14] - 27.0 * m[17] + 13.5 * m[18] - 20.25 * m[27] + 20.25 * m[31] - 20.25 * m[32] - 4.5 * m[39] + 6.75 * m[42] - 13.5 * m[43] + 6.75 * m[46] + 13.5 * m[47] - 13.5 * m[48] - 4.5 * m[51] + 6.75 * m[52] + 6.75 * m[53] - 4.5 * m[54];
      const double K_ = Gs[2] * (22.5 * mk[3] + 40.5 * mk[6] - 162.0 * mk[8] + 40.5 * mk[9] + 13.5 * mk[12] - 135.0 * mk[14] + 27.0 * mk[15] + 155.25 * mk[17] - 135.0 * mk[18] + 13.5 * mk[19] - 4.5 * mk[22] + 27.0 * mk[24] - 13.5 * mk[25] + 6.75 * mk[27] + 54.0 * mk[28] - 13.5 * mk[29] - 24.75 * mk[31] + 6.75 * mk[32] + 27.0 * mk[33] - 4.5 * mk[34]) + Gs[8] * (9.0 * mk[0] + 13.5 * mk[1] - 67.5 * mk[2] + 13.5 * mk[3] - 40.5 * mk[5] + 81.0 * mk[7] - 40.5 * mk[8] - 4.5 * mk[10] + 27.0 * mk[11] - 13.5 * mk[12] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] - 24.75 * mk[16] + 6.75 * mk[17] + 27.0 * mk[18] - 4.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[48] = v_;
      out[162] = v_;
    }
    {
      const double M_ = -4.5 * m[8] - 13.5 * m[14] + 6.75 * m[17] - 13.5 * m[24] + 13.5 * m[27] + 6.75 * m[31] - 20.25 * m[32] + 13.5 * m[33] - 4.5 * m[39] + 6.75 * m[42] + 6.75 * m[46] - 20.25 * m[47] + 13.5 * m[48] - 4.5 * m[51] + 20.25 * m[52] - 27.0 * m[53] + 9.0 * m[54];
      const double K_ = Gs[2] * (-4.5 * mk[3] - 13.5 * mk[6] + 27.0 * mk[8] - 13.5 * mk[12] + 54.0 * mk[14] + 6.75 * mk[17] - 40.5 * mk[18] + 13.5 * mk[19] - 4.5 * mk[22] + 27.0 * mk[24] + 6.75 * mk[27] - 40.5 * mk[28] + 13.5 * mk[29] - 24.75 * mk[31] + 81.0 * mk[32] - 67.5 * mk[33] + 9.0 * mk[34]) + Gs[8] * (-4.5 * mk[0] - 13.5 * mk[1] + 27.0 * mk[2] + 13.5 * mk[3] - 13.5 * mk[4] + 54.0 * mk[5] + 27.0 * mk[6] + 6.75 * mk[7] - 135.0 * mk[8] + 40.5 * mk[9] - 4.5 * mk[10] + 27.0 * mk[11] + 13.5 * mk[12] + 6.75 * mk[13] - 135.0 * mk[14] + 40.5 * mk[15] - 24.75 * mk[16] + 155.25 * mk[17] - 162.0 * mk[18] + 22.5 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[49] = v_;
      out[182] = v_;
    }
    {
      const double M_ = -4.5 * m[13] + 6.75 * m[26] - 13.5 * m[27] + 13.5 * m[38] - 20.25 * m[41] + 6.75 * m[45] + 13.5 * m[46] - 13.5 * m[47] + 9.0 * m[59] - 27.0 * m[62] + 13.5 * m[63] + 20.25 * m[66] - 20.25 * m[67] - 4.5 * m[71] + 6.75 * m[72] + 6.75 * m[73] - 4.5 * m[74];
      const double K_ = Gs[5] * (-4.5 * mk[2] + 13.5 * mk[5] + 27.0 * mk[7] - 13.5 * mk[8] + 40.5 * mk[11] - 135.0 * mk[13] + 27.0 * mk[14] + 6.75 * mk[16] + 54.0 * mk[17] - 13.5 * mk[18] + 22.5 * mk[21] - 162.0 * mk[23] + 40.5 * mk[24] + 155.25 * mk[26] - 135.0 * mk[27] + 13.5 * mk[28] - 24.75 * mk[30] + 6.75 * mk[31] + 27.0 * mk[32] - 4.5 * mk[33]) + Gs[7] * (-4.5 * mk[1] + 27.0 * mk[5] - 13.5 * mk[6] + 13.5 * mk[10] - 40.5 * mk[11] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] + 9.0 * mk[20] - 67.5 * mk[21] + 13.5 * mk[22] + 81.0 * mk[23] - 40.5 * mk[24] - 24.75 * mk[26] + 6.75 * mk[27] + 27.0 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[50] = v_;
      out[202] = v_;
    }
    {
      const double M_ = -4.5 * m[13] - 13.5 * m[23] + 20.25 * m[26] - 13.5 * m[27] - 13.5 * m[38] + 40.5 * m[41] - 27.0 * m[42] - 27.0 * m[45] + 40.5 * m[46] - 13.5 * m[47] - 4.5 * m[59] + 20.25 * m[62] - 13.5 * m[63] - 27.0 * m[66] + 40.5 * m[67] - 13.5 * m[68] + 9.0 * m[71] - 27.0 * m[72] + 20.25 * m[73] - 4.5 * m[74];
      const double K_ = Gs[5] * (-4.5 * mk[2] - 13.5 * mk[5] + 40.5 * mk[7] - 13.5 * mk[8] - 13.5 * mk[11] + 81.0 * mk[13] - 27.0 * mk[14] - 87.75 * mk[16] + 81.0 * mk[17] - 13.5 * mk[18] - 4.5 * mk[21] + 40.5 * mk[23] - 13.5 * mk[24] - 87.75 * mk[26] + 81.0 * mk[27] - 13.5 * mk[28] + 49.5 * mk[30] - 87.75 * mk[31] + 40.5 * mk[32] - 4.5 * mk[33]) + Gs[7] * (-4.5 * mk[1] - 13.5 * mk[4] + 54.0 * mk[5] - 13.5 * mk[6] - 13.5 * mk[10] + 108.0 * mk[11] - 27.0 * mk[12] - 182.25 * mk[13] + 108.0 * mk[14] - 13.5 * mk[15] - 4.5 * mk[20] + 54.0 * mk[21] - 13.5 * mk[22] - 182.25 * mk[23] + 108.0 * mk[24] - 13.5 * mk[25] + 123.75 * mk[26] - 182.25 * mk[27] + 54.0 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[51] = v_;
      out[222] = v_;
    }
    {
      const double M_ = -4.5 * m[14] + 6.75 * m[27] - 13.5 * m[28] + 13.5 * m[39] - 20.25 * m[42] + 6.75 * m[46] + 13.5 * m[47] - 13.5 * m[48] + 9.0 * m[60] - 27.0 * m[63] + 13.5 * m[64] + 20.25 * m[67] - 20.25 * m[68] - 4.5 * m[72] + 6.75 * m[73] + 6.75 * m[74] - 4.5 * m[75];
      const double K_ = Gs[5] * (-4.5 * mk[3] + 13.5 * mk[6] + 27.0 * mk[8] - 13.5 * mk[9] + 40.5 * mk[12] - 135.0 * mk[14] + 27.0 * mk[15] + 6.75 * mk[17] + 54.0 * mk[18] - 13.5 * mk[19] + 22.5 * mk[22] - 162.0 * mk[24] + 40.5 * mk[25] + 155.25 * mk[27] - 135.0 * mk[28] + 13.5 * mk[29] - 24.75 * mk[31] + 6.75 * mk[32] + 27.0 * mk[33] - 4.5 * mk[34]) + Gs[8] * (-4.5 * mk[1] + 27.0 * mk[5] - 13.5 * mk[6] + 13.5 * mk[10] - 40.5 * mk[11] + 6.75 * mk[13] + 54.0 * mk[14] - 13.5 * mk[15] + 9.0 * mk[20] - 67.5 * mk[21] + 13.5 * mk[22] + 81.0 * mk[23] - 40.5 * mk[24] - 24.75 * mk[26] + 6.75 * mk[27] + 27.0 * mk[28] - 4.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[52] = v_;
      out[242] = v_;
    }
    {
      const double M_ = -4.5 * m[14] - 13.5 * m[24] + 6.75 * m[27] - 13.5 * m[39] + 13.5 * m[42] + 6.75 * m[46] - 20.25 * m[47] + 13.5 * m[48] - 4.5 * m[60] + 6.75 * m[63] + 6.75 * m[67] - 20.25 * m[68] + 13.5 * m[69] - 4.5 * m[72] + 20.25 * m[73] - 27.0 * m[74] + 9.0 * m[75];
      const double K_ = Gs[5] * (-4.5 * mk[3] - 13.5 * mk[6] + 27.0 * mk[8] - 13.5 * mk[12] + 54.0 * mk[14] + 6.75 * mk[17] - 40.5 * mk[18] + 13.5 * mk[19] - 4.5 * mk[22] + 27.0 * mk[24] + 6.75 * mk[27] - 40.5 * mk[28] + 13.5 * mk[29] - 24.75 * mk[31] + 81.0 * mk[32] - 67.5 * mk[33] + 9.0 * mk[34]) + Gs[8] * (-4.5 * mk[1] - 13.5 * mk[4] + 27.0 * mk[5] + 13.5 * mk[6] - 13.5 * mk[10] + 54.0 * mk[11] + 27.0 * mk[12] + 6.75 * mk[13] - 135.0 * mk[14] + 40.5 * mk[15] - 4.5 * mk[20] + 27.0 * mk[21] + 13.5 * mk[22] + 6.75 * mk[23] - 135.0 * mk[24] + 40.5 * mk[25] - 24.75 * mk[26] + 155.25 * mk[27] - 162.0 * mk[28] + 22.5 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[53] = v_;
      out[262] = v_;
    }
    {
      const double M_ = -4.5 * m[17] - 13.5 * m[27] + 20.25 * m[31] - 13.5 * m[32] - 13.5 * m[42] + 40.5 * m[46] - 27.0 * m[47] - 27.0 * m[51] + 40.5 * m[52] - 13.5 * m[53] - 4.5 * m[63] + 20.25 * m[67] - 13.5 * m[68] - 27.0 * m[72] + 40.5 * m[73] - 13.5 * m[74] + 9.0 * m[78] - 27.0 * m[79] + 20.25 * m[80] - 4.5 * m[81];
      const double K_ = Gs[7] * (-4.5 * mk[3] - 13.5 * mk[6] + 54.0 * mk[8] - 13.5 * mk[9] - 13.5 * mk[12] + 108.0 * mk[14] - 27.0 * mk[15] - 182.25 * mk[17] + 108.0 * mk[18] - 13.5 * mk[19] - 4.5 * mk[22] + 54.0 * mk[24] - 13.5 * mk[25] - 182.25 * mk[27] + 108.0 * mk[28] - 13.5 * mk[29] + 123.75 * mk[31] - 182.25 * mk[32] + 54.0 * mk[33] - 4.5 * mk[34]) + Gs[8] * (-4.5 * mk[2] - 13.5 * mk[5] + 40.5 * mk[7] - 13.5 * mk[8] - 13.5 * mk[11] + 81.0 * mk[13] - 27.0 * mk[14] - 87.75 * mk[16] + 81.0 * mk[17] - 13.5 * mk[18] - 4.5 * mk[21] + 40.5 * mk[23] - 13.5 * mk[24] - 87.75 * mk[26] + 81.0 * mk[27] - 13.5 * mk[28] + 49.5 * mk[30] - 87.75 * mk[31] + 40.5 * mk[32] - 4.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[54] = v_;
      out[282] = v_;
    }
    {
      const double M_ = -4.5 * m[17] - 13.5 * m[27] + 6.75 * m[31] - 13.5 * m[42] + 13.5 * m[46] + 6.75 * m[51] - 20.25 * m[52] + 13.5 * m[53] - 4.5 * m[63] + 6.75 * m[67] + 6.75 * m[72] - 20.25 * m[73] + 13.5 * m[74] - 4.5 * m[78] + 20.25 * m[79] - 27.0 * m[80] + 9.0 * m[81];
      const double K_ = Gs[7] * (-4.5 * mk[3] - 13.5 * mk[6] + 27.0 * mk[8] - 13.5 * mk[12] + 54.0 * mk[14] + 6.75 * mk[17] - 40.5 * mk[18] + 13.5 * mk[19] - 4.5 * mk[22] + 27.0 * mk[24] + 6.75 * mk[27] - 40.5 * mk[28] + 13.5 * mk[29] - 24.75 * mk[31] + 81.0 * mk[32] - 67.5 * mk[33] + 9.0 * mk[34]) + Gs[8] * (-4.5 * mk[2] - 13.5 * mk[5] + 27.0 * mk[7] + 13.5 * mk[8] - 13.5 * mk[11] + 54.0 * mk[13] + 27.0 * mk[14] + 6.75 * mk[16] - 135.0 * mk[17] + 40.5 * mk[18] - 4.5 * mk[21] + 27.0 * mk[23] + 13.5 * mk[24] + 6.75 * mk[26] - 135.0 * mk[27] + 40.5 * mk[28] - 24.75 * mk[30] + 155.25 * mk[31] - 162.0 * mk[32] + 22.5 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[55] = v_;
      out[302] = v_;
    }
    {
      const double M_ = 27.0 * m[13] + 54.0 * m[23] - 67.5 * m[26] + 54.0 * m[27] + 27.0 * m[38] - 67.5 * m[41] + 54.0 * m[42] + 27.0 * m[45] - 67.5 * m[46] + 27.0 * m[47];
      const double K_ = Gs[2] * (27.0 * mk[5] + 54.0 * mk[11] - 189.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[21] - 189.0 * mk[23] + 54.0 * mk[24] + 148.5 * mk[26] - 189.0 * mk[27] + 27.0 * mk[28]) + Gs[5] * (27.0 * mk[2] + 54.0 * mk[5] - 189.0 * mk[7] + 54.0 * mk[8] + 27.0 * mk[11] - 189.0 * mk[13] + 54.0 * mk[14] + 148.5 * mk[16] - 189.0 * mk[17] + 27.0 * mk[18]) + Gs[7] * (27.0 * mk[1] + 54.0 * mk[4] - 189.0 * mk[5] + 54.0 * mk[6] + 27.0 * mk[10] - 189.0 * mk[11] + 54.0 * mk[12] + 148.5 * mk[13] - 189.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[56] = v_;
      out[322] = v_;
    }
    {
      const double M_ = 27.0 * m[14] + 54.0 * m[24] - 67.5 * m[27] + 54.0 * m[28] + 27.0 * m[39] - 67.5 * m[42] + 54.0 * m[43] + 27.0 * m[46] - 67.5 * m[47] + 27.0 * m[48];
      const double K_ = Gs[2] * (27.0 * mk[6] + 54.0 * mk[12] - 189.0 * mk[14] + 54.0 * mk[15] + 27.0 * mk[22] - 189.0 * mk[24] + 54.0 * mk[25] + 148.5 * mk[27] - 189.0 * mk[28] + 27.0 * mk[29]) + Gs[5] * (27.0 * mk[3] + 54.0 * mk[6] - 189.0 * mk[8] + 54.0 * mk[9] + 27.0 * mk[12] - 189.0 * mk[14] + 54.0 * mk[15] + 148.5 * mk[17] - 189.0 * mk[18] + 27.0 * mk[19]) + Gs[8] * (27.0 * mk[1] + 54.0 * mk[4] - 189.0 * mk[5] + 54.0 * mk[6] + 27.0 * mk[10] - 189.0 * mk[11] + 54.0 * mk[12] + 148.5 * mk[13] - 189.0 * mk[14] + 27.0 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[57] = v_;
      out[342] = v_;
    }
    {
      const double M_ = 27.0 * m[17] + 54.0 * m[27] - 67.5 * m[31] + 54.0 * m[32] + 27.0 * m[42] - 67.5 * m[46] + 54.0 * m[47] + 27.0 * m[51] - 67.5 * m[52] + 27.0 * m[53];
      const double K_ = Gs[2] * (27.0 * mk[8] + 54.0 * mk[14] - 189.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[24] - 189.0 * mk[27] + 54.0 * mk[28] + 148.5 * mk[31] - 189.0 * mk[32] + 27.0 * mk[33]) + Gs[7] * (27.0 * mk[3] + 54.0 * mk[6] - 189.0 * mk[8] + 54.0 * mk[9] + 27.0 * mk[12] - 189.0 * mk[14] + 54.0 * mk[15] + 148.5 * mk[17] - 189.0 * mk[18] + 27.0 * mk[19]) + Gs[8] * (27.0 * mk[2] + 54.0 * mk[5] - 189.0 * mk[7] + 54.0 * mk[8] + 27.0 * mk[11] - 189.0 * mk[13] + 54.0 * mk[14] + 148.5 * mk[16] - 189.0 * mk[17] + 27.0 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[58] = v_;
      out[362] = v_;
    }
    {
      const double M_ = 27.0 * m[27] + 54.0 * m[42] - 67.5 * m[46] + 54.0 * m[47] + 27.0 * m[63] - 67.5 * m[67] + 54.0 * m[68] + 27.0 * m[72] - 67.5 * m[73] + 27.0 * m[74];
      const double K_ = Gs[5] * (27.0 * mk[8] + 54.0 * mk[14] - 189.0 * mk[17] + 54.0 * mk[18] + 27.0 * mk[24] - 189.0 * mk[27] + 54.0 * mk[28] + 148.5 * mk[31] - 189.0 * mk[32] + 27.0 * mk[33]) + Gs[7] * (27.0 * mk[6] + 54.0 * mk[12] - 189.0 * mk[14] + 54.0 * mk[15] + 27.0 * mk[22] - 189.0 * mk[24] + 54.0 * mk[25] + 148.5 * mk[27] - 189.0 * mk[28] + 27.0 * mk[29]) + Gs[8] * (27.0 * mk[5] + 54.0 * mk[11] - 189.0 * mk[13] + 54.0 * mk[14] + 27.0 * mk[21] - 189.0 * mk[23] + 54.0 * mk[24] + 148.5 * mk[26] - 189.0 * mk[27] + 27.0 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[59] = v_;
      out[382] = v_;
    }
    {
      const double M_ = m[9] + 4.0 * m[15] + 4.0 * m[18] - 5.0 * m[19] + 6.0 * m[25] + 12.0 * m[28] - 15.0 * m[29] + 6.0 * m[32] - 15.0 * m[33] + 8.25 * m[34] + 4.0 * m[40] + 12.0 * m[43] - 15.0 * m[44] + 12.0 * m[47] - 30.0 * m[48] + 16.5 * m[49] + 4.0 * m[52] - 15.0 * m[53] + 16.5 * m[54] - 5.0 * m[55] + m[61] + 4.0 * m[64] - 5.0 * m[65] + 6.0 * m[68] - 15.0 * m[69] + 8.25 * m[70] + 4.0 * m[73] - 15.0 * m[74] + 16.5 * m[75] - 5.0 * m[76] + m[79] - 5.0 * m[80] + 8.25 * m[81] - 5.0 * m[82] + m[83];
      const double K_ = Gs[9] * (mk[0] + 4.0 * mk[1] + 4.0 * mk[2] - 14.0 * mk[3] + 6.0 * mk[4] + 12.0 * mk[5] - 42.0 * mk[6] + 6.0 * mk[7] - 42.0 * mk[8] + 60.0 * mk[9] + 4.0 * mk[10] + 12.0 * mk[11] - 42.0 * mk[12] + 12.0 * mk[13] - 84.0 * mk[14] + 120.0 * mk[15] + 4.0 * mk[16] - 42.0 * mk[17] + 120.0 * mk[18] - 77.0 * mk[19] + mk[20] + 4.0 * mk[21] - 14.0 * mk[22] + 6.0 * mk[23] - 42.0 * mk[24] + 60.0 * mk[25] + 4.0 * mk[26] - 42.0 * mk[27] + 120.0 * mk[28] - 77.0 * mk[29] + mk[30] - 14.0 * mk[31] + 60.0 * mk[32] - 77.0 * mk[33] + 30.25 * mk[34]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[63] = v_;
    }
    {
      const double M_ = 9.0 * m[6] + 13.5 * m[12] + 13.5 * m[14] - 27.0 * m[15] - 20.25 * m[25] - 20.25 * m[28] + 20.25 * m[29] - 4.5 * m[37] - 13.5 * m[39] + 6.75 * m[40] - 13.5 * m[42] + 13.5 * m[43] + 6.75 * m[44] - 4.5 * m[46] + 6.75 * m[47] + 6.75 * m[48] - 4.5 * m[49];
      const double K_ = Gs[3] * (22.5 * mk[1] + 40.5 * mk[4] + 40.5 * mk[5] - 162.0 * mk[6] + 13.5 * mk[10] + 27.0 * mk[11] - 135.0 * mk[12] + 13.5 * mk[13] - 135.0 * mk[14] + 155.25 * mk[15] - 4.5 * mk[20] - 13.5 * mk[21] + 27.0 * mk[22] - 13.5 * mk[23] + 54.0 * mk[24] + 6.75 * mk[25] - 4.5 * mk[26] + 27.0 * mk[27] + 6.75 * mk[28] - 24.75 * mk[29]) + Gs[6] * (9.0 * mk[0] + 13.5 * mk[1] + 13.5 * mk[2] - 67.5 * mk[3] - 40.5 * mk[6] - 40.5 * mk[8] + 81.0 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] + 27.0 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] - 4.5 * mk[16] + 27.0 * mk[17] + 6.75 * mk[18] - 24.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[64] = v_;
      out[83] = v_;
    }
    {
      const double M_ = -4.5 * m[6] - 13.5 * m[14] + 6.75 * m[15] + 13.5 * m[22] - 20.25 * m[25] - 13.5 * m[27] + 13.5 * m[28] + 6.75 * m[29] + 9.0 * m[37] + 13.5 * m[39] - 27.0 * m[40] - 20.25 * m[43] + 20.25 * m[44] - 4.5 * m[46] + 6.75 * m[47] + 6.75 * m[48] - 4.5 * m[49];
      const double K_ = Gs[3] * (-4.5 * mk[1] - 13.5 * mk[5] + 27.0 * mk[6] + 13.5 * mk[10] - 40.5 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] - 67.5 * mk[22] - 40.5 * mk[24] + 81.0 * mk[25] - 4.5 * mk[26] + 27.0 * mk[27] + 6.75 * mk[28] - 24.75 * mk[29]) + Gs[6] * (-4.5 * mk[0] + 13.5 * mk[1] - 13.5 * mk[2] + 27.0 * mk[3] + 40.5 * mk[4] + 27.0 * mk[5] - 135.0 * mk[6] - 13.5 * mk[7] + 54.0 * mk[8] + 6.75 * mk[9] + 22.5 * mk[10] + 40.5 * mk[11] - 162.0 * mk[12] + 13.5 * mk[13] - 135.0 * mk[14] + 155.25 * mk[15] - 4.5 * mk[16] + 27.0 * mk[17] + 6.75 * mk[18] - 24.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[65] = v_;
      out[103] = v_;
    }
    {
      const double M_ = 9.0 * m[8] + 13.5 * m[14] + 13.5 * m[17] - 27.0 * m[18] - 20.25 * m[28] - 20.25 * m[32] + 20.25 * m[33] - 4.5 * m[39] - 13.5 * m[42] + 6.75 * m[43] - 13.5 * m[46] + 13.5 * m[47] + 6.75 * m[48] - 4.5 * m[51] + 6.75 * m[52] + 6.75 * m[53] - 4.5 * m[54];
      const double K_ = Gs[3] * (22.5 * mk[2] + 40.5 * mk[5] + 40.5 * mk[7] - 162.0 * mk[8] + 13.5 * mk[11] + 27.0 * mk[13] - 135.0 * mk[14] + 13.5 * mk[16] - 135.0 * mk[17] + 155.25 * mk[18] - 4.5 * mk[21] - 13.5 * mk[23] + 27.0 * mk[24] - 13.5 * mk[26] + 54.0 * mk[27] + 6.75 * mk[28] - 4.5 * mk[30] + 27.0 * mk[31] + 6.75 * mk[32] - 24.75 * mk[33]) + Gs[8] * (9.0 * mk[0] + 13.5 * mk[1] + 13.5 * mk[2] - 67.5 * mk[3] - 40.5 * mk[6] - 40.5 * mk[8] + 81.0 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] + 27.0 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] - 4.5 * mk[16] + 27.0 * mk[17] + 6.75 * mk[18] - 24.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[66] = v_;
      out[123] = v_;
    }
    {
      const double M_ = -4.5 * m[8] - 13.5 * m[14] + 6.75 * m[18] - 13.5 * m[24] + 13.5 * m[28] + 13.5 * m[31] - 20.25 * m[32] + 6.75 * m[33] - 4.5 * m[39] + 6.75 * m[43] + 13.5 * m[46] - 20.25 * m[47] + 6.75 * m[48] + 9.0 * m[51] - 27.0 * m[52] + 20.25 * m[53] - 4.5 * m[54];
      const double K_ = Gs[3] * (-4.5 * mk[2] - 13.5 * mk[5] + 27.0 * mk[8] - 13.5 * mk[11] + 54.0 * mk[14] + 13.5 * mk[16] - 40.5 * mk[17] + 6.75 * mk[18] - 4.5 * mk[21] + 27.0 * mk[24] + 13.5 * mk[26] - 40.5 * mk[27] + 6.75 * mk[28] + 9.0 * mk[30] - 67.5 * mk[31] + 81.0 * mk[32] - 24.75 * mk[33]) + Gs[8] * (-4.5 * mk[0] - 13.5 * mk[1] + 13.5 * mk[2] + 27.0 * mk[3] - 13.5 * mk[4] + 27.0 * mk[5] + 54.0 * mk[6] + 40.5 * mk[7] - 135.0 * mk[8] + 6.75 * mk[9] - 4.5 * mk[10] + 13.5 * mk[11] + 27.0 * mk[12] + 40.5 * mk[13] - 135.0 * mk[14] + 6.75 * mk[15] + 22.5 * mk[16] - 162.0 * mk[17] + 155.25 * mk[18] - 24.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[67] = v_;
      out[143] = v_;
    }
    {
      const double M_ = 9.0 * m[9] + 13.5 * m[15] + 13.5 * m[18] - 27.0 * m[19] - 20.25 * m[29] - 20.25 * m[33] + 20.25 * m[34] - 4.5 * m[40] - 13.5 * m[43] + 6.75 * m[44] - 13.5 * m[47] + 13.5 * m[48] + 6.75 * m[49] - 4.5 * m[52] + 6.75 * m[53] + 6.75 * m[54] - 4.5 * m[55];
      const double K_ = Gs[3] * (22.5 * mk[3] + 40.5 * mk[6] + 40.5 * mk[8] - 162.0 * mk[9] + 13.5 * mk[12] + 27.0 * mk[14] - 135.0 * mk[15] + 13.5 * mk[17] - 135.0 * mk[18] + 155.25 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] + 27.0 * mk[25] - 13.5 * mk[27] + 54.0 * mk[28] + 6.75 * mk[29] - 4.5 * mk[31] + 27.0 * mk[32] + 6.75 * mk[33] - 24.75 * mk[34]) + Gs[9] * (9.0 * mk[0] + 13.5 * mk[1] + 13.5 * mk[2] - 67.5 * mk[3] - 40.5 * mk[6] - 40.5 * mk[8] + 81.0 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] + 27.0 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] - 4.5 * mk[16] + 27.0 * mk[17] + 6.75 * mk[18] - 24.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[68] = v_;
      out[163] = v_;
    }
    {
      const double M_ = -4.5 * m[9] - 13.5 * m[15] - 13.5 * m[18] + 20.25 * m[19] - 13.5 * m[25] - 27.0 * m[28] + 40.5 * m[29] - 13.5 * m[32] + 40.5 * m[33] - 27.0 * m[34] - 4.5 * m[40] - 13.5 * m[43] + 20.25 * m[44] - 13.5 * m[47] + 40.5 * m[48] - 27.0 * m[49] - 4.5 * m[52] + 20.25 * m[53] - 27.0 * m[54] + 9.0 * m[55];
      const double K_ = Gs[3] * (-4.5 * mk[3] - 13.5 * mk[6] - 13.5 * mk[8] + 40.5 * mk[9] - 13.5 * mk[12] - 27.0 * mk[14] + 81.0 * mk[15] - 13.5 * mk[17] + 81.0 * mk[18] - 87.75 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] + 40.5 * mk[25] - 13.5 * mk[27] + 81.0 * mk[28] - 87.75 * mk[29] - 4.5 * mk[31] + 40.5 * mk[32] - 87.75 * mk[33] + 49.5 * mk[34]) + Gs[9] * (-4.5 * mk[0] - 13.5 * mk[1] - 13.5 * mk[2] + 54.0 * mk[3] - 13.5 * mk[4] - 27.0 * mk[5] + 108.0 * mk[6] - 13.5 * mk[7] + 108.0 * mk[8] - 182.25 * mk[9] - 4.5 * mk[10] - 13.5 * mk[11] + 54.0 * mk[12] - 13.5 * mk[13] + 108.0 * mk[14] - 182.25 * mk[15] - 4.5 * mk[16] + 54.0 * mk[17] - 182.25 * mk[18] + 123.75 * mk[19]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[69] = v_;
      out[183] = v_;
    }
    {
      const double M_ = -4.5 * m[14] - 13.5 * m[27] + 6.75 * m[28] + 13.5 * m[39] - 20.25 * m[43] - 13.5 * m[46] + 13.5 * m[47] + 6.75 * m[48] + 9.0 * m[60] + 13.5 * m[63] - 27.0 * m[64] - 20.25 * m[68] + 20.25 * m[69] - 4.5 * m[72] + 6.75 * m[73] + 6.75 * m[74] - 4.5 * m[75];
      const double K_ = Gs[6] * (-4.5 * mk[2] + 13.5 * mk[5] - 13.5 * mk[7] + 27.0 * mk[8] + 40.5 * mk[11] + 27.0 * mk[13] - 135.0 * mk[14] - 13.5 * mk[16] + 54.0 * mk[17] + 6.75 * mk[18] + 22.5 * mk[21] + 40.5 * mk[23] - 162.0 * mk[24] + 13.5 * mk[26] - 135.0 * mk[27] + 155.25 * mk[28] - 4.5 * mk[30] + 27.0 * mk[31] + 6.75 * mk[32] - 24.75 * mk[33]) + Gs[8] * (-4.5 * mk[1] - 13.5 * mk[5] + 27.0 * mk[6] + 13.5 * mk[10] - 40.5 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] - 67.5 * mk[22] - 40.5 * mk[24] + 81.0 * mk[25] - 4.5 * mk[26] + 27.0 * mk[27] + 6.75 * mk[28] - 24.75 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[70] = v_;
      out[203] = v_;
    }
    {
      const double M_ = -4.5 * m[14] - 13.5 * m[24] + 6.75 * m[28] - 13.5 * m[39] + 13.5 * m[43] + 13.5 * m[46] - 20.25 * m[47] + 6.75 * m[48] - 4.5 * m[60] + 6.75 * m[64] + 13.5 * m[67] - 20.25 * m[68] + 6.75 * m[69] + 9.0 * m[72] - 27.0 * m[73] + 20.25 * m[74] - 4.5 * m[75];
      const double K_ = Gs[6] * (-4.5 * mk[2] - 13.5 * mk[5] + 27.0 * mk[8] - 13.5 * mk[11] + 54.0 * mk[14] + 13.5 * mk[16] - 40.5 * mk[17] + 6.75 * mk[18] - 4.5 * mk[21] + 27.0 * mk[24] + 13.5 * mk[26] - 40.5 * mk[27] + 6.75 * mk[28] + 9.0 * mk[30] - 67.5 * mk[31] + 81.0 * mk[32] - 24.75 * mk[33]) + Gs[8] * (-4.5 * mk[1] - 13.5 * mk[4] + 13.5 * mk[5] + 27.0 * mk[6] - 13.5 * mk[10] + 27.0 * mk[11] + 54.0 * mk[12] + 40.5 * mk[13] - 135.0 * mk[14] + 6.75 * mk[15] - 4.5 * mk[20] + 13.5 * mk[21] + 27.0 * mk[22] + 40.5 * mk[23] - 135.0 * mk[24] + 6.75 * mk[25] + 22.5 * mk[26] - 162.0 * mk[27] + 155.25 * mk[28] - 24.75 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[71] = v_;
      out[223] = v_;
    }
    {
      const double M_ = -4.5 * m[15] - 13.5 * m[28] + 6.75 * m[29] + 13.5 * m[40] - 20.25 * m[44] - 13.5 * m[47] + 13.5 * m[48] + 6.75 * m[49] + 9.0 * m[61] + 13.5 * m[64] - 27.0 * m[65] - 20.25 * m[69] + 20.25 * m[70] - 4.5 * m[73] + 6.75 * m[74] + 6.75 * m[75] - 4.5 * m[76];
      const double K_ = Gs[6] * (-4.5 * mk[3] + 13.5 * mk[6] - 13.5 * mk[8] + 27.0 * mk[9] + 40.5 * mk[12] + 27.0 * mk[14] - 135.0 * mk[15] - 13.5 * mk[17] + 54.0 * mk[18] + 6.75 * mk[19] + 22.5 * mk[22] + 40.5 * mk[24] - 162.0 * mk[25] + 13.5 * mk[27] - 135.0 * mk[28] + 155.25 * mk[29] - 4.5 * mk[31] + 27.0 * mk[32] + 6.75 * mk[33] - 24.75 * mk[34]) + Gs[9] * (-4.5 * mk[1] - 13.5 * mk[5] + 27.0 * mk[6] + 13.5 * mk[10] - 40.5 * mk[12] - 13.5 * mk[13] + 54.0 * mk[14] + 6.75 * mk[15] + 9.0 * mk[20] + 13.5 * mk[21] - 67.5 * mk[22] - 40.5 * mk[24] + 81.0 * mk[25] - 4.5 * mk[26] + 27.0 * mk[27] + 6.75 * mk[28] - 24.75 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[72] = v_;
      out[243] = v_;
    }
    {
      const double M_ = -4.5 * m[15] - 13.5 * m[25] - 13.5 * m[28] + 20.25 * m[29] - 13.5 * m[40] - 27.0 * m[43] + 40.5 * m[44] - 13.5 * m[47] + 40.5 * m[48] - 27.0 * m[49] - 4.5 * m[61] - 13.5 * m[64] + 20.25 * m[65] - 13.5 * m[68] + 40.5 * m[69] - 27.0 * m[70] - 4.5 * m[73] + 20.25 * m[74] - 27.0 * m[75] + 9.0 * m[76];
      const double K_ = Gs[6] * (-4.5 * mk[3] - 13.5 * mk[6] - 13.5 * mk[8] + 40.5 * mk[9] - 13.5 * mk[12] - 27.0 * mk[14] + 81.0 * mk[15] - 13.5 * mk[17] + 81.0 * mk[18] - 87.75 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] + 40.5 * mk[25] - 13.5 * mk[27] + 81.0 * mk[28] - 87.75 * mk[29] - 4.5 * mk[31] + 40.5 * mk[32] - 87.75 * mk[33] + 49.5 * mk[34]) + Gs[9] * (-4.5 * mk[1] - 13.5 * mk[4] - 13.5 * mk[5] + 54.0 * mk[6] - 13.5 * mk[10] - 27.0 * mk[11] + 108.0 * mk[12] - 13.5 * mk[13] + 108.0 * mk[14] - 182.25 * mk[15] - 4.5 * mk[20] - 13.5 * mk[21] + 54.0 * mk[22] - 13.5 * mk[23] + 108.0 * mk[24] - 182.25 * mk[25] - 4.5 * mk[26] + 54.0 * mk[27] - 182.25 * mk[28] + 123.75 * mk[29]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[73] = v_;
      out[263] = v_;
    }
    {
      const double M_ = -4.5 * m[18] - 13.5 * m[28] + 6.75 * m[33] - 13.5 * m[43] + 13.5 * m[48] + 13.5 * m[52] - 20.25 * m[53] + 6.75 * m[54] - 4.5 * m[64] + 6.75 * m[69] + 13.5 * m[73] - 20.25 * m[74] + 6.75 * m[75] + 9.0 * m[79] - 27.0 * m[80] + 20.25 * m[81] - 4.5 * m[82];
      const double K_ = Gs[8] * (-4.5 * mk[3] - 13.5 * mk[6] + 13.5 * mk[8] + 27.0 * mk[9] - 13.5 * mk[12] + 27.0 * mk[14] + 54.0 * mk[15] + 40.5 * mk[17] - 135.0 * mk[18] + 6.75 * mk[19] - 4.5 * mk[22] + 13.5 * mk[24] + 27.0 * mk[25] + 40.5 * mk[27] - 135.0 * mk[28] + 6.75 * mk[29] + 22.5 * mk[31] - 162.0 * mk[32] + 155.25 * mk[33] - 24.75 * mk[34]) + Gs[9] * (-4.5 * mk[2] - 13.5 * mk[5] + 27.0 * mk[8] - 13.5 * mk[11] + 54.0 * mk[14] + 13.5 * mk[16] - 40.5 * mk[17] + 6.75 * mk[18] - 4.5 * mk[21] + 27.0 * mk[24] + 13.5 * mk[26] - 40.5 * mk[27] + 6.75 * mk[28] + 9.0 * mk[30] - 67.5 * mk[31] + 81.0 * mk[32] - 24.75 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[74] = v_;
      out[283] = v_;
    }
    {
      const double M_ = -4.5 * m[18] - 13.5 * m[28] - 13.5 * m[32] + 20.25 * m[33] - 13.5 * m[43] - 27.0 * m[47] + 40.5 * m[48] - 13.5 * m[52] + 40.5 * m[53] - 27.0 * m[54] - 4.5 * m[64] - 13.5 * m[68] + 20.25 * m[69] - 13.5 * m[73] + 40.5 * m[74] - 27.0 * m[75] - 4.5 * m[79] + 20.25 * m[80] - 27.0 * m[81] + 9.0 * m[82];
      const double K_ = Gs[8] * (-4.5 * mk[3] - 13.5 * mk[6] - 13.5 * mk[8] + 40.5 * mk[9] - 13.5 * mk[12] - 27.0 * mk[14] + 81.0 * mk[15] - 13.5 * mk[17] + 81.0 * mk[18] - 87.75 * mk[19] - 4.5 * mk[22] - 13.5 * mk[24] + 40.5 * mk[25] - 13.5 * mk[27] + 81.0 * mk[28] - 87.75 * mk[29] - 4.5 * mk[31] + 40.5 * mk[32] - 87.75 * mk[33] + 49.5 * mk[34]) + Gs[9] * (-4.5 * mk[2] - 13.5 * mk[5] - 13.5 * mk[7] + 54.0 * mk[8] - 13.5 * mk[11] - 27.0 * mk[13] + 108.0 * mk[14] - 13.5 * mk[16] + 108.0 * mk[17] - 182.25 * mk[18] - 4.5 * mk[21] - 13.5 * mk[23] + 54.0 * mk[24] - 13.5 * mk[26] + 108.0 * mk[27] - 182.25 * mk[28] - 4.5 * mk[30] + 54.0 * mk[31] - 182.25 * mk[32] + 123.75 * mk[33]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[75] = v_;
      out[303] = v_;
    }
    {
      const double M_ = 27.0 * m[14] + 54.0 * m[24] + 54.0 * m[27] - 67.5 * m[28] + 27.0 * m[39] + 54.0 * m[42] - 67.5 * m[43] + 27.0 * m[46] - 67.5 * m[47] + 27.0 * m[48];
      const double K_ = Gs[3] * (27.0 * mk[5] + 54.0 * mk[11] + 54.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[21] + 54.0 * mk[23] - 189.0 * mk[24] + 27.0 * mk[26] - 189.0 * mk[27] + 148.5 * mk[28]) + Gs[6] * (27.0 * mk[2] + 54.0 * mk[5] + 54.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] + 54.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[16] - 189.0 * mk[17] + 148.5 * mk[18]) + Gs[8] * (27.0 * mk[1] + 54.0 * mk[4] + 54.0 * mk[5] - 189.0 * mk[6] + 27.0 * mk[10] + 54.0 * mk[11] - 189.0 * mk[12] + 27.0 * mk[13] - 189.0 * mk[14] + 148.5 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[76] = v_;
      out[323] = v_;
    }
    {
      const double M_ = 27.0 * m[15] + 54.0 * m[25] + 54.0 * m[28] - 67.5 * m[29] + 27.0 * m[40] + 54.0 * m[43] - 67.5 * m[44] + 27.0 * m[47] - 67.5 * m[48] + 27.0 * m[49];
      const double K_ = Gs[3] * (27.0 * mk[6] + 54.0 * mk[12] + 54.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[22] + 54.0 * mk[24] - 189.0 * mk[25] + 27.0 * mk[27] - 189.0 * mk[28] + 148.5 * mk[29]) + Gs[6] * (27.0 * mk[3] + 54.0 * mk[6] + 54.0 * mk[8] - 189.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[17] - 189.0 * mk[18] + 148.5 * mk[19]) + Gs[9] * (27.0 * mk[1] + 54.0 * mk[4] + 54.0 * mk[5] - 189.0 * mk[6] + 27.0 * mk[10] + 54.0 * mk[11] - 189.0 * mk[12] + 27.0 * mk[13] - 189.0 * mk[14] + 148.5 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[77] = v_;
      out[343] = v_;
    }
    {
      const double M_ = 27.0 * m[18] + 54.0 * m[28] + 54.0 * m[32] - 67.5 * m[33] + 27.0 * m[43] + 54.0 * m[47] - 67.5 * m[48] + 27.0 * m[52] - 67.5 * m[53] + 27.0 * m[54];
      const double K_ = Gs[3] * (27.0 * mk[8] + 54.0 * mk[14] + 54.0 * mk[17] - 189.0 * mk[18] + 27.0 * mk[24] + 54.0 * mk[27] - 189.0 * mk[28] + 27.0 * mk[31] - 189.0 * mk[32] + 148.5 * mk[33]) + Gs[8] * (27.0 * mk[3] + 54.0 * mk[6] + 54.0 * mk[8] - 189.0 * mk[9] + 27.0 * mk[12] + 54.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[17] - 189.0 * mk[18] + 148.5 * mk[19]) + Gs[9] * (27.0 * mk[2] + 54.0 * mk[5] + 54.0 * mk[7] - 189.0 * mk[8] + 27.0 * mk[11] + 54.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[16] - 189.0 * mk[17] + 148.5 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[78] = v_;
      out[363] = v_;
    }
    {
      const double M_ = 27.0 * m[28] + 54.0 * m[43] + 54.0 * m[47] - 67.5 * m[48] + 27.0 * m[64] + 54.0 * m[68] - 67.5 * m[69] + 27.0 * m[73] - 67.5 * m[74] + 27.0 * m[75];
      const double K_ = Gs[6] * (27.0 * mk[8] + 54.0 * mk[14] + 54.0 * mk[17] - 189.0 * mk[18] + 27.0 * mk[24] + 54.0 * mk[27] - 189.0 * mk[28] + 27.0 * mk[31] - 189.0 * mk[32] + 148.5 * mk[33]) + Gs[8] * (27.0 * mk[6] + 54.0 * mk[12] + 54.0 * mk[14] - 189.0 * mk[15] + 27.0 * mk[22] + 54.0 * mk[24] - 189.0 * mk[25] + 27.0 * mk[27] - 189.0 * mk[28] + 148.5 * mk[29]) + Gs[9] * (27.0 * mk[5] + 54.0 * mk[11] + 54.0 * mk[13] - 189.0 * mk[14] + 27.0 * mk[21] + 54.0 * mk[23] - 189.0 * mk[24] + 27.0 * mk[26] - 189.0 * mk[27] + 148.5 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[79] = v_;
      out[383] = v_;
    }
    {
      const double M_ = 81.0 * m[4] - 81.0 * m[10] - 81.0 * m[11] - 81.0 * m[12] + 20.25 * m[20] + 40.5 * m[21] + 40.5 * m[22] + 20.25 * m[23] + 40.5 * m[24] + 20.25 * m[25];
      const double K_ = Gs[0] * (506.25 * mk[4] - 202.5 * mk[10] - 202.5 * mk[11] - 202.5 * mk[12] + 20.25 * mk[20] + 40.5 * mk[21] + 40.5 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[1] * (405.0 * mk[1] - 283.5 * mk[4] - 283.5 * mk[5] - 283.5 * mk[6] + 40.5 * mk[10] + 81.0 * mk[11] + 81.0 * mk[12] + 40.5 * mk[13] + 81.0 * mk[14] + 40.5 * mk[15]) + Gs[4] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[84] = v_;
    }
    {
      const double M_ = -40.5 * m[4] + 101.25 * m[10] - 20.25 * m[11] - 20.25 * m[12] - 40.5 * m[20] - 20.25 * m[21] - 20.25 * m[22] + 20.25 * m[23] + 40.5 * m[24] + 20.25 * m[25];
      const double K_ = Gs[0] * (-101.25 * mk[4] + 222.75 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] - 20.25 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[1] * (-141.75 * mk[1] + 627.75 * mk[4] - 101.25 * mk[5] - 101.25 * mk[6] - 141.75 * mk[10] - 101.25 * mk[11] - 101.25 * mk[12] + 40.5 * mk[13] + 81.0 * mk[14] + 40.5 * mk[15]) + Gs[4] * (-40.5 * mk[0] + 222.75 * mk[1] - 20.25 * mk[2] - 20.25 * mk[3] - 101.25 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[85] = v_;
      out[104] = v_;
    }
    {
      const double M_ = 81.0 * m[5] - 81.0 * m[11] - 81.0 * m[13] - 81.0 * m[14] + 20.25 * m[21] + 40.5 * m[23] + 40.5 * m[24] + 20.25 * m[26] + 40.5 * m[27] + 20.25 * m[28];
      const double K_ = Gs[0] * (506.25 * mk[5] - 202.5 * mk[11] - 202.5 * mk[13] - 202.5 * mk[14] + 20.25 * mk[21] + 40.5 * mk[23] + 40.5 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[1] * (202.5 * mk[2] - 141.75 * mk[5] - 141.75 * mk[7] - 141.75 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] + 40.5 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[2] * (202.5 * mk[1] - 141.75 * mk[4] - 141.75 * mk[5] - 141.75 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]) + Gs[5] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[86] = v_;
      out[124] = v_;
    }
    {
      const double M_ = -40.5 * m[5] - 20.25 * m[11] + 101.25 * m[13] - 20.25 * m[14] + 20.25 * m[21] - 20.25 * m[23] + 40.5 * m[24] - 40.5 * m[26] - 20.25 * m[27] + 20.25 * m[28];
      const double K_ = Gs[0] * (-101.25 * mk[5] - 81.0 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] + 40.5 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[1] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[2] * (-101.25 * mk[1] - 81.0 * mk[4] + 526.5 * mk[5] - 81.0 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]) + Gs[5] * (-40.5 * mk[0] - 20.25 * mk[1] + 222.75 * mk[2] - 20.25 * mk[3] + 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[87] = v_;
      out[144] = v_;
    }
    {
      const double M_ = 81.0 * m[6] - 81.0 * m[12] - 81.0 * m[14] - 81.0 * m[15] + 20.25 * m[22] + 40.5 * m[24] + 40.5 * m[25] + 20.25 * m[27] + 40.5 * m[28] + 20.25 * m[29];
      const double K_ = Gs[0] * (506.25 * mk[6] - 202.5 * mk[12] - 202.5 * mk[14] - 202.5 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] + 40.5 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[1] * (202.5 * mk[3] - 141.75 * mk[6] - 141.75 * mk[8] - 141.75 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] + 40.5 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[3] * (202.5 * mk[1] - 141.75 * mk[4] - 141.75 * mk[5] - 141.75 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]) + Gs[6] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[88] = v_;
      out[164] = v_;
    }
    {
      const double M_ = -40.5 * m[6] - 20.25 * m[12] - 20.25 * m[14] + 101.25 * m[15] + 20.25 * m[22] + 40.5 * m[24] - 20.25 * m[25] + 20.25 * m[27] - 20.25 * m[28] - 40.5 * m[29];
      const double K_ = Gs[0] * (-101.25 * mk[6] - 81.0 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[1] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[3] * (-101.25 * mk[1] - 81.0 * mk[4] - 81.0 * mk[5] + 526.5 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]) + Gs[6] * (-40.5 * mk[0] - 20.25 * mk[1] - 20.25 * mk[2] + 222.75 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] - 81.0 * mk[8] - 101.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[89] = v_;
      out[184] = v_;
    }
    {
      const double M_ = -40.5 * m[11] + 101.25 * m[21] - 20.25 * m[23] - 20.25 * m[24] - 40.5 * m[36] - 20.25 * m[38] - 20.25 * m[39] + 20.25 * m[41] + 40.5 * m[42] + 20.25 * m[43];
      const double K_ = Gs[1] * (-101.25 * mk[5] + 526.5 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] - 101.25 * mk[21] - 81.0 * mk[23] - 81.0 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[2] * (-101.25 * mk[4] + 222.75 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] - 20.25 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[4] * (-40.5 * mk[2] + 222.75 * mk[5] - 20.25 * mk[7] - 20.25 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[5] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[90] = v_;
      out[204] = v_;
    }
    {
      const double M_ = -40.5 * m[11] - 20.25 * m[21] + 101.25 * m[23] - 20.25 * m[24] + 20.25 * m[36] - 20.25 * m[38] + 40.5 * m[39] - 40.5 * m[41] - 20.25 * m[42] + 20.25 * m[43];
      const double K_ = Gs[1] * (-101.25 * mk[5] - 81.0 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] + 40.5 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[2] * (-101.25 * mk[4] - 81.0 * mk[10] + 526.5 * mk[11] - 81.0 * mk[12] + 20.25 * mk[20] - 81.0 * mk[21] + 40.5 * mk[22] - 101.25 * mk[23] - 81.0 * mk[24] + 20.25 * mk[25]) + Gs[4] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[5] * (-40.5 * mk[1] - 20.25 * mk[4] + 222.75 * mk[5] - 20.25 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[91] = v_;
      out[224] = v_;
    }
    {
      const double M_ = -40.5 * m[12] + 101.25 * m[22] - 20.25 * m[24] - 20.25 * m[25] - 40.5 * m[37] - 20.25 * m[39] - 20.25 * m[40] + 20.25 * m[42] + 40.5 * m[43] + 20.25 * m[44];
      const double K_ = Gs[1] * (-101.25 * mk[6] + 526.5 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] - 101.25 * mk[22] - 81.0 * mk[24] - 81.0 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[3] * (-101.25 * mk[4] + 222.75 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] - 20.25 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[4] * (-40.5 * mk[3] + 222.75 * mk[6] - 20.25 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[6] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[92] = v_;
      out[244] = v_;
    }
    {
      const double M_ = -40.5 * m[12] - 20.25 * m[22] - 20.25 * m[24] + 101.25 * m[25] + 20.25 * m[37] + 40.5 * m[39] - 20.25 * m[40] + 20.25 * m[42] - 20.25 * m[43] - 40.5 * m[44];
      const double K_ = Gs[1] * (-101.25 * mk[6] - 81.0 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[3] * (-101.25 * mk[4] - 81.0 * mk[10] - 81.0 * mk[11] + 526.5 * mk[12] + 20.25 * mk[20] + 40.5 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] - 81.0 * mk[24] - 101.25 * mk[25]) + Gs[4] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[6] * (-40.5 * mk[1] - 20.25 * mk[4] - 20.25 * mk[5] + 222.75 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[93] = v_;
      out[264] = v_;
    }
    {
      const double M_ = -40.5 * m[14] - 20.25 * m[24] + 101.25 * m[27] - 20.25 * m[28] + 20.25 * m[39] - 20.25 * m[42] + 40.5 * m[43] - 40.5 * m[46] - 20.25 * m[47] + 20.25 * m[48];
      const double K_ = Gs[2] * (-101.25 * mk[6] - 81.0 * mk[12] + 526.5 * mk[14] - 81.0 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] + 40.5 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[3] * (-101.25 * mk[5] - 81.0 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] + 40.5 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[5] * (-40.5 * mk[3] - 20.25 * mk[6] + 222.75 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[6] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[94] = v_;
      out[284] = v_;
    }
    {
      const double M_ = -40.5 * m[14] - 20.25 * m[24] - 20.25 * m[27] + 101.25 * m[28] + 20.25 * m[39] + 40.5 * m[42] - 20.25 * m[43] + 20.25 * m[46] - 20.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[2] * (-101.25 * mk[6] - 81.0 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[3] * (-101.25 * mk[5] - 81.0 * mk[11] - 81.0 * mk[13] + 526.5 * mk[14] + 20.25 * mk[21] + 40.5 * mk[23] - 81.0 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]) + Gs[5] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[6] * (-40.5 * mk[2] - 20.25 * mk[5] - 20.25 * mk[7] + 222.75 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[95] = v_;
      out[304] = v_;
    }
    {
      const double M_ = 243.0 * m[11] - 121.5 * m[21] - 121.5 * m[23] - 121.5 * m[24];
      const double K_ = Gs[0] * (607.5 * mk[11] - 121.5 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[1] * (850.5 * mk[5] - 243.0 * mk[11] - 243.0 * mk[13] - 243.0 * mk[14]) + Gs[2] * (607.5 * mk[4] - 121.5 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]) + Gs[4] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]) + Gs[5] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[96] = v_;
      out[324] = v_;
    }
    {
      const double M_ = 243.0 * m[12] - 121.5 * m[22] - 121.5 * m[24] - 121.5 * m[25];
      const double K_ = Gs[0] * (607.5 * mk[12] - 121.5 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[1] * (850.5 * mk[6] - 243.0 * mk[12] - 243.0 * mk[14] - 243.0 * mk[15]) + Gs[3] * (607.5 * mk[4] - 121.5 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]) + Gs[4] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[6] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[97] = v_;
      out[344] = v_;
    }
    {
      const double M_ = 243.0 * m[14] - 121.5 * m[24] - 121.5 * m[27] - 121.5 * m[28];
      const double K_ = Gs[0] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[1] * (243.0 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[2] * (607.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[3] * (607.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[5] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[6] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[98] = v_;
      out[364] = v_;
    }
    {
      const double M_ = 243.0 * m[24] - 121.5 * m[39] - 121.5 * m[42] - 121.5 * m[43];
      const double K_ = Gs[1] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[2] * (607.5 * mk[12] - 121.5 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[3] * (607.5 * mk[11] - 121.5 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[4] * (243.0 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[5] * (243.0 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[6] * (243.0 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[99] = v_;
      out[384] = v_;
    }
    {
      const double M_ = 20.25 * m[4] - 81.0 * m[10] + 40.5 * m[11] + 40.5 * m[12] + 81.0 * m[20] - 81.0 * m[21] - 81.0 * m[22] + 20.25 * m[23] + 40.5 * m[24] + 20.25 * m[25];
      const double K_ = Gs[0] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[1] * (40.5 * mk[1] - 283.5 * mk[4] + 81.0 * mk[5] + 81.0 * mk[6] + 405.0 * mk[10] - 283.5 * mk[11] - 283.5 * mk[12] + 40.5 * mk[13] + 81.0 * mk[14] + 40.5 * mk[15]) + Gs[4] * (20.25 * mk[0] - 202.5 * mk[1] + 40.5 * mk[2] + 40.5 * mk[3] + 506.25 * mk[4] - 202.5 * mk[5] - 202.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[105] = v_;
    }
    {
      const double M_ = -40.5 * m[5] + 101.25 * m[11] - 20.25 * m[13] - 20.25 * m[14] - 40.5 * m[21] - 20.25 * m[23] - 20.25 * m[24] + 20.25 * m[26] + 40.5 * m[27] + 20.25 * m[28];
      const double K_ = Gs[0] * (-101.25 * mk[5] + 222.75 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] - 20.25 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[1] * (-101.25 * mk[2] + 526.5 * mk[5] - 81.0 * mk[7] - 81.0 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[2] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]) + Gs[5] * (-40.5 * mk[0] + 222.75 * mk[1] - 20.25 * mk[2] - 20.25 * mk[3] - 101.25 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[106] = v_;
      out[125] = v_;
    }
    {
      const double M_ = 20.25 * m[5] - 20.25 * m[11] - 20.25 * m[13] + 40.5 * m[14] - 40.5 * m[21] + 101.25 * m[23] - 20.25 * m[24] - 40.5 * m[26] - 20.25 * m[27] + 20.25 * m[28];
      const double K_ = Gs[0] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[1] * (20.25 * mk[2] - 81.0 * mk[5] - 20.25 * mk[7] + 40.5 * mk[8] - 101.25 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[2] * (20.25 * mk[1] - 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 40.5 * mk[10] + 222.75 * mk[11] - 20.25 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]) + Gs[5] * (20.25 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] + 40.5 * mk[3] - 101.25 * mk[4] + 526.5 * mk[5] - 81.0 * mk[6] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[107] = v_;
      out[145] = v_;
    }
    {
      const double M_ = -40.5 * m[6] + 101.25 * m[12] - 20.25 * m[14] - 20.25 * m[15] - 40.5 * m[22] - 20.25 * m[24] - 20.25 * m[25] + 20.25 * m[27] + 40.5 * m[28] + 20.25 * m[29];
      const double K_ = Gs[0] * (-101.25 * mk[6] + 222.75 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[1] * (-101.25 * mk[3] + 526.5 * mk[6] - 81.0 * mk[8] - 81.0 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[3] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]) + Gs[6] * (-40.5 * mk[0] + 222.75 * mk[1] - 20.25 * mk[2] - 20.25 * mk[3] - 101.25 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[108] = v_;
      out[165] = v_;
    }
    {
      const double M_ = 20.25 * m[6] - 20.25 * m[12] + 40.5 * m[14] - 20.25 * m[15] - 40.5 * m[22] - 20.25 * m[24] + 101.25 * m[25] + 20.25 * m[27] - 20.25 * m[28] - 40.5 * m[29];
      const double K_ = Gs[0] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[1] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[3] * (20.25 * mk[1] - 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] + 222.75 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]) + Gs[6] * (20.25 * mk[0] - 81.0 * mk[1] + 40.5 * mk[2] - 81.0 * mk[3] - 101.25 * mk[4] - 81.0 * mk[5] + 526.5 * mk[6] + 20.25 * mk[7] - 81.0 * mk[8] - 101.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[109] = v_;
      out[185] = v_;
    }
    {
      const double M_ = 20.25 * m[11] - 81.0 * m[21] + 40.5 * m[23] + 40.5 * m[24] + 81.0 * m[36] - 81.0 * m[38] - 81.0 * m[39] + 20.25 * m[41] + 40.5 * m[42] + 20.25 * m[43];
      const double K_ = Gs[1] * (20.25 * mk[5] - 141.75 * mk[11] + 40.5 * mk[13] + 40.5 * mk[14] + 202.5 * mk[21] - 141.75 * mk[23] - 141.75 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[2] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[4] * (20.25 * mk[2] - 202.5 * mk[5] + 40.5 * mk[7] + 40.5 * mk[8] + 506.25 * mk[11] - 202.5 * mk[13] - 202.5 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[5] * (20.25 * mk[1] - 141.75 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 202.5 * mk[10] - 141.75 * mk[11] - 141.75 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[110] = v_;
      out[205] = v_;
    }
    {
      const double M_ = 20.25 * m[11] - 20.25 * m[21] - 20.25 * m[23] + 40.5 * m[24] - 40.5 * m[36] + 101.25 * m[38] - 20.25 * m[39] - 40.5 * m[41] - 20.25 * m[42] + 20.25 * m[43];
      const double K_ = Gs[1] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[2] * (20.25 * mk[4] - 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 40.5 * mk[20] + 222.75 * mk[21] - 20.25 * mk[22] - 101.25 * mk[23] - 81.0 * mk[24] + 20.25 * mk[25]) + Gs[4] * (20.25 * mk[2] - 81.0 * mk[5] - 20.25 * mk[7] + 40.5 * mk[8] - 101.25 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[5] * (20.25 * mk[1] - 81.0 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 101.25 * mk[10] + 526.5 * mk[11] - 81.0 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[111] = v_;
      out[225] = v_;
    }
    {
      const double M_ = 20.25 * m[12] - 81.0 * m[22] + 40.5 * m[24] + 40.5 * m[25] + 81.0 * m[37] - 81.0 * m[39] - 81.0 * m[40] + 20.25 * m[42] + 40.5 * m[43] + 20.25 * m[44];
      const double K_ = Gs[1] * (20.25 * mk[6] - 141.75 * mk[12] + 40.5 * mk[14] + 40.5 * mk[15] + 202.5 * mk[22] - 141.75 * mk[24] - 141.75 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[3] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]) + Gs[4] * (20.25 * mk[3] - 202.5 * mk[6] + 40.5 * mk[8] + 40.5 * mk[9] + 506.25 * mk[12] - 202.5 * mk[14] - 202.5 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[6] * (20.25 * mk[1] - 141.75 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 202.5 * mk[10] - 141.75 * mk[11] - 141.75 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[112] = v_;
      out[245] = v_;
    }
    {
      const double M_ = 20.25 * m[12] - 20.25 * m[22] + 40.5 * m[24] - 20.25 * m[25] - 40.5 * m[37] - 20.25 * m[39] + 101.25 * m[40] + 20.25 * m[42] - 20.25 * m[43] - 40.5 * m[44];
      const double K_ = Gs[1] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[3] * (20.25 * mk[4] - 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] + 222.75 * mk[22] + 20.25 * mk[23] - 81.0 * mk[24] - 101.25 * mk[25]) + Gs[4] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[6] * (20.25 * mk[1] - 81.0 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] - 101.25 * mk[10] - 81.0 * mk[11] + 526.5 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[113] = v_;
      out[265] = v_;
    }
    {
      const double M_ = 20.25 * m[14] - 20.25 * m[24] - 20.25 * m[27] + 40.5 * m[28] - 40.5 * m[39] + 101.25 * m[42] - 20.25 * m[43] - 40.5 * m[46] - 20.25 * m[47] + 20.25 * m[48];
      const double K_ = Gs[2] * (20.25 * mk[6] - 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 40.5 * mk[22] + 222.75 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[3] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[5] * (20.25 * mk[3] - 81.0 * mk[6] - 81.0 * mk[8] + 40.5 * mk[9] - 101.25 * mk[12] + 526.5 * mk[14] - 81.0 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[6] * (20.25 * mk[2] - 81.0 * mk[5] - 20.25 * mk[7] + 40.5 * mk[8] - 101.25 * mk[11] + 222.75 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[114] = v_;
      out[285] = v_;
    }
    {
      const double M_ = 20.25 * m[14] - 20.25 * m[24] + 40.5 * m[27] - 20.25 * m[28] - 40.5 * m[39] - 20.25 * m[42] + 101.25 * m[43] + 20.25 * m[46] - 20.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[2] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[3] * (20.25 * mk[5] - 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] + 222.75 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]) + Gs[5] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] + 222.75 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[6] * (20.25 * mk[2] - 81.0 * mk[5] + 40.5 * mk[7] - 81.0 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] + 526.5 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[115] = v_;
      out[305] = v_;
    }
    {
      const double M_ = -121.5 * m[11] + 243.0 * m[21] - 121.5 * m[23] - 121.5 * m[24];
      const double K_ = Gs[0] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[1] * (-243.0 * mk[5] + 850.5 * mk[11] - 243.0 * mk[13] - 243.0 * mk[14]) + Gs[2] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]) + Gs[4] * (-121.5 * mk[2] + 607.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]) + Gs[5] * (-121.5 * mk[1] + 607.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[116] = v_;
      out[325] = v_;
    }
    {
      const double M_ = -121.5 * m[12] + 243.0 * m[22] - 121.5 * m[24] - 121.5 * m[25];
      const double K_ = Gs[0] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[1] * (-243.0 * mk[6] + 850.5 * mk[12] - 243.0 * mk[14] - 243.0 * mk[15]) + Gs[3] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]) + Gs[4] * (-121.5 * mk[3] + 607.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[6] * (-121.5 * mk[1] + 607.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[117] = v_;
      out[345] = v_;
    }
    {
      const double M_ = -121.5 * m[14] + 243.0 * m[24] - 121.5 * m[27] - 121.5 * m[28];
      const double K_ = Gs[0] * (-121.5 * mk[14] + 243.0 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[1] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[2] * (-121.5 * mk[6] + 243.0 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[3] * (-121.5 * mk[5] + 243.0 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[5] * (-121.5 * mk[3] + 607.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[6] * (-121.5 * mk[2] + 607.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[118] = v_;
      out[365] = v_;
    }
    {
      const double M_ = -121.5 * m[24] + 243.0 * m[39] - 121.5 * m[42] - 121.5 * m[43];
      const double K_ = Gs[1] * (-121.5 * mk[14] + 243.0 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[2] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[3] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[4] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[5] * (-121.5 * mk[6] + 607.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[6] * (-121.5 * mk[5] + 607.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[119] = v_;
      out[385] = v_;
    }
    {
      const double M_ = 81.0 * m[7] - 81.0 * m[13] - 81.0 * m[16] - 81.0 * m[17] + 20.25 * m[23] + 40.5 * m[26] + 40.5 * m[27] + 20.25 * m[30] + 40.5 * m[31] + 20.25 * m[32];
      const double K_ = Gs[0] * (506.25 * mk[7] - 202.5 * mk[13] - 202.5 * mk[16] - 202.5 * mk[17] + 20.25 * mk[23] + 40.5 * mk[26] + 40.5 * mk[27] + 20.25 * mk[30] + 40.5 * mk[31] + 20.25 * mk[32]) + Gs[2] * (405.0 * mk[2] - 283.5 * mk[5] - 283.5 * mk[7] - 283.5 * mk[8] + 40.5 * mk[11] + 81.0 * mk[13] + 81.0 * mk[14] + 40.5 * mk[16] + 81.0 * mk[17] + 40.5 * mk[18]) + Gs[7] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[126] = v_;
    }
    {
      const double M_ = -40.5 * m[7] - 20.25 * m[13] + 101.25 * m[16] - 20.25 * m[17] + 20.25 * m[23] - 20.25 * m[26] + 40.5 * m[27] - 40.5 * m[30] - 20.25 * m[31] + 20.25 * m[32];
      const double K_ = Gs[0] * (-101.25 * mk[7] - 81.0 * mk[13] + 222.75 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] + 40.5 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[2] * (-141.75 * mk[2] - 101.25 * mk[5] + 627.75 * mk[7] - 101.25 * mk[8] + 40.5 * mk[11] - 101.25 * mk[13] + 81.0 * mk[14] - 141.75 * mk[16] - 101.25 * mk[17] + 40.5 * mk[18]) + Gs[7] * (-40.5 * mk[0] - 20.25 * mk[1] + 222.75 * mk[2] - 20.25 * mk[3] + 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[127] = v_;
      out[146] = v_;
    }
    {
      const double M_ = 81.0 * m[8] - 81.0 * m[14] - 81.0 * m[17] - 81.0 * m[18] + 20.25 * m[24] + 40.5 * m[27] + 40.5 * m[28] + 20.25 * m[31] + 40.5 * m[32] + 20.25 * m[33];
      const double K_ = Gs[0] * (506.25 * mk[8] - 202.5 * mk[14] - 202.5 * mk[17] - 202.5 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] + 40.5 * mk[28] + 20.25 * mk[31] + 40.5 * mk[32] + 20.25 * mk[33]) + Gs[2] * (202.5 * mk[3] - 141.75 * mk[6] - 141.75 * mk[8] - 141.75 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] + 40.5 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[3] * (202.5 * mk[2] - 141.75 * mk[5] - 141.75 * mk[7] - 141.75 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] + 40.5 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[8] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[128] = v_;
      out[166] = v_;
    }
    {
      const double M_ = -40.5 * m[8] - 20.25 * m[14] - 20.25 * m[17] + 101.25 * m[18] + 20.25 * m[24] + 40.5 * m[27] - 20.25 * m[28] + 20.25 * m[31] - 20.25 * m[32] - 40.5 * m[33];
      const double K_ = Gs[0] * (-101.25 * mk[8] - 81.0 * mk[14] - 81.0 * mk[17] + 222.75 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 20.25 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[2] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[3] * (-101.25 * mk[2] - 81.0 * mk[5] - 81.0 * mk[7] + 526.5 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]) + Gs[8] * (-40.5 * mk[0] - 20.25 * mk[1] - 20.25 * mk[2] + 222.75 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] - 81.0 * mk[8] - 101.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[129] = v_;
      out[186] = v_;
    }
    {
      const double M_ = -40.5 * m[13] + 101.25 * m[23] - 20.25 * m[26] - 20.25 * m[27] - 40.5 * m[38] - 20.25 * m[41] - 20.25 * m[42] + 20.25 * m[45] + 40.5 * m[46] + 20.25 * m[47];
      const double K_ = Gs[1] * (-101.25 * mk[7] + 526.5 * mk[13] - 81.0 * mk[16] - 81.0 * mk[17] - 101.25 * mk[23] - 81.0 * mk[26] - 81.0 * mk[27] + 20.25 * mk[30] + 40.5 * mk[31] + 20.25 * mk[32]) + Gs[2] * (-101.25 * mk[5] + 222.75 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] - 20.25 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[5] * (-40.5 * mk[2] + 222.75 * mk[5] - 20.25 * mk[7] - 20.25 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[7] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[130] = v_;
      out[206] = v_;
    }
    {
      const double M_ = -40.5 * m[13] - 20.25 * m[23] + 101.25 * m[26] - 20.25 * m[27] + 20.25 * m[38] - 20.25 * m[41] + 40.5 * m[42] - 40.5 * m[45] - 20.25 * m[46] + 20.25 * m[47];
      const double K_ = Gs[1] * (-101.25 * mk[7] - 81.0 * mk[13] + 222.75 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] + 40.5 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[2] * (-101.25 * mk[5] - 81.0 * mk[11] + 526.5 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 81.0 * mk[23] + 40.5 * mk[24] - 101.25 * mk[26] - 81.0 * mk[27] + 20.25 * mk[28]) + Gs[5] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[7] * (-40.5 * mk[1] - 20.25 * mk[4] + 222.75 * mk[5] - 20.25 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[131] = v_;
      out[226] = v_;
    }
    {
      const double M_ = -40.5 * m[14] + 101.25 * m[24] - 20.25 * m[27] - 20.25 * m[28] - 40.5 * m[39] - 20.25 * m[42] - 20.25 * m[43] + 20.25 * m[46] + 40.5 * m[47] + 20.25 * m[48];
      const double K_ = Gs[1] * (-101.25 * mk[8] + 526.5 * mk[14] - 81.0 * mk[17] - 81.0 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] - 81.0 * mk[28] + 20.25 * mk[31] + 40.5 * mk[32] + 20.25 * mk[33]) + Gs[3] * (-101.25 * mk[5] + 222.75 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] - 20.25 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[5] * (-40.5 * mk[3] + 222.75 * mk[6] - 20.25 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[8] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[132] = v_;
      out[246] = v_;
    }
    {
      const double M_ = -40.5 * m[14] - 20.25 * m[24] - 20.25 * m[27] + 101.25 * m[28] + 20.25 * m[39] + 40.5 * m[42] - 20.25 * m[43] + 20.25 * m[46] - 20.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[1] * (-101.25 * mk[8] - 81.0 * mk[14] - 81.0 * mk[17] + 222.75 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 20.25 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[3] * (-101.25 * mk[5] - 81.0 * mk[11] - 81.0 * mk[13] + 526.5 * mk[14] + 20.25 * mk[21] + 40.5 * mk[23] - 81.0 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]) + Gs[5] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[8] * (-40.5 * mk[1] - 20.25 * mk[4] - 20.25 * mk[5] + 222.75 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[133] = v_;
      out[266] = v_;
    }
    {
      const double M_ = -40.5 * m[17] - 20.25 * m[27] + 101.25 * m[31] - 20.25 * m[32] + 20.25 * m[42] - 20.25 * m[46] + 40.5 * m[47] - 40.5 * m[51] - 20.25 * m[52] + 20.25 * m[53];
      const double K_ = Gs[2] * (-101.25 * mk[8] - 81.0 * mk[14] + 526.5 * mk[17] - 81.0 * mk[18] + 20.25 * mk[24] - 81.0 * mk[27] + 40.5 * mk[28] - 101.25 * mk[31] - 81.0 * mk[32] + 20.25 * mk[33]) + Gs[3] * (-101.25 * mk[7] - 81.0 * mk[13] + 222.75 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] + 40.5 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[7] * (-40.5 * mk[3] - 20.25 * mk[6] + 222.75 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[8] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[134] = v_;
      out[286] = v_;
    }
    {
      const double M_ = -40.5 * m[17] - 20.25 * m[27] - 20.25 * m[31] + 101.25 * m[32] + 20.25 * m[42] + 40.5 * m[46] - 20.25 * m[47] + 20.25 * m[51] - 20.25 * m[52] - 40.5 * m[53];
      const double K_ = Gs[2] * (-101.25 * mk[8] - 81.0 * mk[14] - 81.0 * mk[17] + 222.75 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 20.25 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[3] * (-101.25 * mk[7] - 81.0 * mk[13] - 81.0 * mk[16] + 526.5 * mk[17] + 20.25 * mk[23] + 40.5 * mk[26] - 81.0 * mk[27] + 20.25 * mk[30] - 81.0 * mk[31] - 101.25 * mk[32]) + Gs[7] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[8] * (-40.5 * mk[2] - 20.25 * mk[5] - 20.25 * mk[7] + 222.75 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[135] = v_;
      out[306] = v_;
    }
    {
      const double M_ = 243.0 * m[13] - 121.5 * m[23] - 121.5 * m[26] - 121.5 * m[27];
      const double K_ = Gs[0] * (607.5 * mk[13] - 121.5 * mk[23] - 121.5 * mk[26] - 121.5 * mk[27]) + Gs[1] * (607.5 * mk[7] - 121.5 * mk[13] - 121.5 * mk[16] - 121.5 * mk[17]) + Gs[2] * (850.5 * mk[5] - 243.0 * mk[11] - 243.0 * mk[13] - 243.0 * mk[14]) + Gs[5] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]) + Gs[7] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[136] = v_;
      out[326] = v_;
    }
    {
      const double M_ = 243.0 * m[14] - 121.5 * m[24] - 121.5 * m[27] - 121.5 * m[28];
      const double K_ = Gs[0] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[1] * (607.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[2] * (243.0 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[3] * (607.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[5] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[8] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[137] = v_;
      out[346] = v_;
    }
    {
      const double M_ = 243.0 * m[17] - 121.5 * m[27] - 121.5 * m[31] - 121.5 * m[32];
      const double K_ = Gs[0] * (607.5 * mk[17] - 121.5 * mk[27] - 121.5 * mk[31] - 121.5 * mk[32]) + Gs[2] * (850.5 * mk[8] - 243.0 * mk[14] - 243.0 * mk[17] - 243.0 * mk[18]) + Gs[3] * (607.5 * mk[7] - 121.5 * mk[13] - 121.5 * mk[16] - 121.5 * mk[17]) + Gs[7] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[8] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[138] = v_;
      out[366] = v_;
    }
    {
      const double M_ = 243.0 * m[27] - 121.5 * m[42] - 121.5 * m[46] - 121.5 * m[47];
      const double K_ = Gs[1] * (607.5 * mk[17] - 121.5 * mk[27] - 121.5 * mk[31] - 121.5 * mk[32]) + Gs[2] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[3] * (607.5 * mk[13] - 121.5 * mk[23] - 121.5 * mk[26] - 121.5 * mk[27]) + Gs[5] * (243.0 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[7] * (243.0 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[8] * (243.0 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[139] = v_;
      out[386] = v_;
    }
    {
      const double M_ = 20.25 * m[7] + 40.5 * m[13] - 81.0 * m[16] + 40.5 * m[17] + 20.25 * m[23] - 81.0 * m[26] + 40.5 * m[27] + 81.0 * m[30] - 81.0 * m[31] + 20.25 * m[32];
      const double K_ = Gs[0] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]) + Gs[2] * (40.5 * mk[2] + 81.0 * mk[5] - 283.5 * mk[7] + 81.0 * mk[8] + 40.5 * mk[11] - 283.5 * mk[13] + 81.0 * mk[14] + 405.0 * mk[16] - 283.5 * mk[17] + 40.5 * mk[18]) + Gs[7] * (20.25 * mk[0] + 40.5 * mk[1] - 202.5 * mk[2] + 40.5 * mk[3] + 20.25 * mk[4] - 202.5 * mk[5] + 40.5 * mk[6] + 506.25 * mk[7] - 202.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[147] = v_;
    }
    {
      const double M_ = -40.5 * m[8] - 20.25 * m[14] + 101.25 * m[17] - 20.25 * m[18] + 20.25 * m[24] - 20.25 * m[27] + 40.5 * m[28] - 40.5 * m[31] - 20.25 * m[32] + 20.25 * m[33];
      const double K_ = Gs[0] * (-101.25 * mk[8] - 81.0 * mk[14] + 222.75 * mk[17] - 81.0 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] + 40.5 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[2] * (-101.25 * mk[3] - 81.0 * mk[6] + 526.5 * mk[8] - 81.0 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[3] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[8] * (-40.5 * mk[0] - 20.25 * mk[1] + 222.75 * mk[2] - 20.25 * mk[3] + 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 101.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[148] = v_;
      out[167] = v_;
    }
    {
      const double M_ = 20.25 * m[8] + 40.5 * m[14] - 20.25 * m[17] - 20.25 * m[18] + 20.25 * m[24] - 20.25 * m[27] - 20.25 * m[28] - 40.5 * m[31] + 101.25 * m[32] - 40.5 * m[33];
      const double K_ = Gs[0] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[2] * (20.25 * mk[3] + 40.5 * mk[6] - 81.0 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] - 101.25 * mk[17] + 222.75 * mk[18] - 40.5 * mk[19]) + Gs[3] * (20.25 * mk[2] + 40.5 * mk[5] - 20.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] + 222.75 * mk[17] - 101.25 * mk[18]) + Gs[8] * (20.25 * mk[0] + 40.5 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] - 101.25 * mk[7] + 526.5 * mk[8] - 101.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[149] = v_;
      out[187] = v_;
    }
    {
      const double M_ = 20.25 * m[13] - 20.25 * m[23] - 20.25 * m[26] + 40.5 * m[27] - 40.5 * m[38] + 101.25 * m[41] - 20.25 * m[42] - 40.5 * m[45] - 20.25 * m[46] + 20.25 * m[47];
      const double K_ = Gs[1] * (20.25 * mk[7] - 81.0 * mk[13] - 20.25 * mk[16] + 40.5 * mk[17] - 101.25 * mk[23] + 222.75 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[2] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[5] * (20.25 * mk[2] - 81.0 * mk[5] - 81.0 * mk[7] + 40.5 * mk[8] - 101.25 * mk[11] + 526.5 * mk[13] - 81.0 * mk[14] - 101.25 * mk[16] - 81.0 * mk[17] + 20.25 * mk[18]) + Gs[7] * (20.25 * mk[1] - 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 40.5 * mk[10] + 222.75 * mk[11] - 20.25 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[150] = v_;
      out[207] = v_;
    }
    {
      const double M_ = 20.25 * m[13] + 40.5 * m[23] - 81.0 * m[26] + 40.5 * m[27] + 20.25 * m[38] - 81.0 * m[41] + 40.5 * m[42] + 81.0 * m[45] - 81.0 * m[46] + 20.25 * m[47];
      const double K_ = Gs[1] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]) + Gs[2] * (20.25 * mk[5] + 40.5 * mk[11] - 141.75 * mk[13] + 40.5 * mk[14] + 20.25 * mk[21] - 141.75 * mk[23] + 40.5 * mk[24] + 202.5 * mk[26] - 141.75 * mk[27] + 20.25 * mk[28]) + Gs[5] * (20.25 * mk[2] + 40.5 * mk[5] - 141.75 * mk[7] + 40.5 * mk[8] + 20.25 * mk[11] - 141.75 * mk[13] + 40.5 * mk[14] + 202.5 * mk[16] - 141.75 * mk[17] + 20.25 * mk[18]) + Gs[7] * (20.25 * mk[1] + 40.5 * mk[4] - 202.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[10] - 202.5 * mk[11] + 40.5 * mk[12] + 506.25 * mk[13] - 202.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[151] = v_;
      out[227] = v_;
    }
    {
      const double M_ = 20.25 * m[14] - 20.25 * m[24] - 20.25 * m[27] + 40.5 * m[28] - 40.5 * m[39] + 101.25 * m[42] - 20.25 * m[43] - 40.5 * m[46] - 20.25 * m[47] + 20.25 * m[48];
      const double K_ = Gs[1] * (20.25 * mk[8] - 81.0 * mk[14] - 20.25 * mk[17] + 40.5 * mk[18] - 101.25 * mk[24] + 222.75 * mk[27] - 81.0 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[3] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[5] * (20.25 * mk[3] - 81.0 * mk[6] - 81.0 * mk[8] + 40.5 * mk[9] - 101.25 * mk[12] + 526.5 * mk[14] - 81.0 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[8] * (20.25 * mk[1] - 20.25 * mk[4] - 81.0 * mk[5] + 40.5 * mk[6] - 40.5 * mk[10] + 222.75 * mk[11] - 20.25 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[152] = v_;
      out[247] = v_;
    }
    {
      const double M_ = 20.25 * m[14] + 40.5 * m[24] - 20.25 * m[27] - 20.25 * m[28] + 20.25 * m[39] - 20.25 * m[42] - 20.25 * m[43] - 40.5 * m[46] + 101.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[1] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[3] * (20.25 * mk[5] + 40.5 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] - 81.0 * mk[24] - 40.5 * mk[26] + 222.75 * mk[27] - 101.25 * mk[28]) + Gs[5] * (20.25 * mk[3] + 40.5 * mk[6] - 81.0 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] - 101.25 * mk[17] + 222.75 * mk[18] - 40.5 * mk[19]) + Gs[8] * (20.25 * mk[1] + 40.5 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] - 101.25 * mk[13] + 526.5 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[153] = v_;
      out[267] = v_;
    }
    {
      const double M_ = 20.25 * m[17] + 40.5 * m[27] - 81.0 * m[31] + 40.5 * m[32] + 20.25 * m[42] - 81.0 * m[46] + 40.5 * m[47] + 81.0 * m[51] - 81.0 * m[52] + 20.25 * m[53];
      const double K_ = Gs[2] * (20.25 * mk[8] + 40.5 * mk[14] - 141.75 * mk[17] + 40.5 * mk[18] + 20.25 * mk[24] - 141.75 * mk[27] + 40.5 * mk[28] + 202.5 * mk[31] - 141.75 * mk[32] + 20.25 * mk[33]) + Gs[3] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]) + Gs[7] * (20.25 * mk[3] + 40.5 * mk[6] - 202.5 * mk[8] + 40.5 * mk[9] + 20.25 * mk[12] - 202.5 * mk[14] + 40.5 * mk[15] + 506.25 * mk[17] - 202.5 * mk[18] + 20.25 * mk[19]) + Gs[8] * (20.25 * mk[2] + 40.5 * mk[5] - 141.75 * mk[7] + 40.5 * mk[8] + 20.25 * mk[11] - 141.75 * mk[13] + 40.5 * mk[14] + 202.5 * mk[16] - 141.75 * mk[17] + 20.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[154] = v_;
      out[287] = v_;
    }
    {
      const double M_ = 20.25 * m[17] + 40.5 * m[27] - 20.25 * m[31] - 20.25 * m[32] + 20.25 * m[42] - 20.25 * m[46] - 20.25 * m[47] - 40.5 * m[51] + 101.25 * m[52] - 40.5 * m[53];
      const double K_ = Gs[2] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[3] * (20.25 * mk[7] + 40.5 * mk[13] - 20.25 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] + 222.75 * mk[31] - 101.25 * mk[32]) + Gs[7] * (20.25 * mk[3] + 40.5 * mk[6] - 81.0 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] - 101.25 * mk[17] + 222.75 * mk[18] - 40.5 * mk[19]) + Gs[8] * (20.25 * mk[2] + 40.5 * mk[5] - 81.0 * mk[7] - 81.0 * mk[8] + 20.25 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] - 101.25 * mk[16] + 526.5 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[155] = v_;
      out[307] = v_;
    }
    {
      const double M_ = -121.5 * m[13] - 121.5 * m[23] + 243.0 * m[26] - 121.5 * m[27];
      const double K_ = Gs[0] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]) + Gs[1] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]) + Gs[2] * (-243.0 * mk[5] - 243.0 * mk[11] + 850.5 * mk[13] - 243.0 * mk[14]) + Gs[5] * (-121.5 * mk[2] - 121.5 * mk[5] + 607.5 * mk[7] - 121.5 * mk[8]) + Gs[7] * (-121.5 * mk[1] - 121.5 * mk[4] + 607.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[156] = v_;
      out[327] = v_;
    }
    {
      const double M_ = -121.5 * m[14] - 121.5 * m[24] + 243.0 * m[27] - 121.5 * m[28];
      const double K_ = Gs[0] * (-121.5 * mk[14] - 121.5 * mk[24] + 243.0 * mk[27] - 121.5 * mk[28]) + Gs[1] * (-121.5 * mk[8] - 121.5 * mk[14] + 243.0 * mk[17] - 121.5 * mk[18]) + Gs[2] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[3] * (-121.5 * mk[5] - 121.5 * mk[11] + 243.0 * mk[13] - 121.5 * mk[14]) + Gs[5] * (-121.5 * mk[3] - 121.5 * mk[6] + 607.5 * mk[8] - 121.5 * mk[9]) + Gs[8] * (-121.5 * mk[1] - 121.5 * mk[4] + 607.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[157] = v_;
      out[347] = v_;
    }
    {
      const double M_ = -121.5 * m[17] - 121.5 * m[27] + 243.0 * m[31] - 121.5 * m[32];
      const double K_ = Gs[0] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[2] * (-243.0 * mk[8] - 243.0 * mk[14] + 850.5 * mk[17] - 243.0 * mk[18]) + Gs[3] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]) + Gs[7] * (-121.5 * mk[3] - 121.5 * mk[6] + 607.5 * mk[8] - 121.5 * mk[9]) + Gs[8] * (-121.5 * mk[2] - 121.5 * mk[5] + 607.5 * mk[7] - 121.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[158] = v_;
      out[367] = v_;
    }
    {
      const double M_ = -121.5 * m[27] - 121.5 * m[42] + 243.0 * m[46] - 121.5 * m[47];
      const double K_ = Gs[1] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[2] * (-121.5 * mk[14] - 121.5 * mk[24] + 243.0 * mk[27] - 121.5 * mk[28]) + Gs[3] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]) + Gs[5] * (-121.5 * mk[8] - 121.5 * mk[14] + 607.5 * mk[17] - 121.5 * mk[18]) + Gs[7] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[8] * (-121.5 * mk[5] - 121.5 * mk[11] + 607.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[159] = v_;
      out[387] = v_;
    }
    {
      const double M_ = 81.0 * m[9] - 81.0 * m[15] - 81.0 * m[18] - 81.0 * m[19] + 20.25 * m[25] + 40.5 * m[28] + 40.5 * m[29] + 20.25 * m[32] + 40.5 * m[33] + 20.25 * m[34];
      const double K_ = Gs[0] * (506.25 * mk[9] - 202.5 * mk[15] - 202.5 * mk[18] - 202.5 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] + 40.5 * mk[29] + 20.25 * mk[32] + 40.5 * mk[33] + 20.25 * mk[34]) + Gs[3] * (405.0 * mk[3] - 283.5 * mk[6] - 283.5 * mk[8] - 283.5 * mk[9] + 40.5 * mk[12] + 81.0 * mk[14] + 81.0 * mk[15] + 40.5 * mk[17] + 81.0 * mk[18] + 40.5 * mk[19]) + Gs[9] * (81.0 * mk[0] - 81.0 * mk[1] - 81.0 * mk[2] - 81.0 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] + 40.5 * mk[6] + 20.25 * mk[7] + 40.5 * mk[8] + 20.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[168] = v_;
    }
    {
      const double M_ = -40.5 * m[9] - 20.25 * m[15] - 20.25 * m[18] + 101.25 * m[19] + 20.25 * m[25] + 40.5 * m[28] - 20.25 * m[29] + 20.25 * m[32] - 20.25 * m[33] - 40.5 * m[34];
      const double K_ = Gs[0] * (-101.25 * mk[9] - 81.0 * mk[15] - 81.0 * mk[18] + 222.75 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 20.25 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[3] * (-141.75 * mk[3] - 101.25 * mk[6] - 101.25 * mk[8] + 627.75 * mk[9] + 40.5 * mk[12] + 81.0 * mk[14] - 101.25 * mk[15] + 40.5 * mk[17] - 101.25 * mk[18] - 141.75 * mk[19]) + Gs[9] * (-40.5 * mk[0] - 20.25 * mk[1] - 20.25 * mk[2] + 222.75 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] + 20.25 * mk[7] - 81.0 * mk[8] - 101.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[169] = v_;
      out[188] = v_;
    }
    {
      const double M_ = -40.5 * m[14] + 101.25 * m[24] - 20.25 * m[27] - 20.25 * m[28] - 40.5 * m[39] - 20.25 * m[42] - 20.25 * m[43] + 20.25 * m[46] + 40.5 * m[47] + 20.25 * m[48];
      const double K_ = Gs[1] * (-101.25 * mk[8] + 526.5 * mk[14] - 81.0 * mk[17] - 81.0 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] - 81.0 * mk[28] + 20.25 * mk[31] + 40.5 * mk[32] + 20.25 * mk[33]) + Gs[2] * (-101.25 * mk[6] + 222.75 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[6] * (-40.5 * mk[2] + 222.75 * mk[5] - 20.25 * mk[7] - 20.25 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] + 40.5 * mk[17] + 20.25 * mk[18]) + Gs[8] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[170] = v_;
      out[208] = v_;
    }
    {
      const double M_ = -40.5 * m[14] - 20.25 * m[24] + 101.25 * m[27] - 20.25 * m[28] + 20.25 * m[39] - 20.25 * m[42] + 40.5 * m[43] - 40.5 * m[46] - 20.25 * m[47] + 20.25 * m[48];
      const double K_ = Gs[1] * (-101.25 * mk[8] - 81.0 * mk[14] + 222.75 * mk[17] - 81.0 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] + 40.5 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[2] * (-101.25 * mk[6] - 81.0 * mk[12] + 526.5 * mk[14] - 81.0 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] + 40.5 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[6] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]) + Gs[8] * (-40.5 * mk[1] - 20.25 * mk[4] + 222.75 * mk[5] - 20.25 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 101.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[171] = v_;
      out[228] = v_;
    }
    {
      const double M_ = -40.5 * m[15] + 101.25 * m[25] - 20.25 * m[28] - 20.25 * m[29] - 40.5 * m[40] - 20.25 * m[43] - 20.25 * m[44] + 20.25 * m[47] + 40.5 * m[48] + 20.25 * m[49];
      const double K_ = Gs[1] * (-101.25 * mk[9] + 526.5 * mk[15] - 81.0 * mk[18] - 81.0 * mk[19] - 101.25 * mk[25] - 81.0 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] + 40.5 * mk[33] + 20.25 * mk[34]) + Gs[3] * (-101.25 * mk[6] + 222.75 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] - 20.25 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[6] * (-40.5 * mk[3] + 222.75 * mk[6] - 20.25 * mk[8] - 20.25 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] + 20.25 * mk[17] + 40.5 * mk[18] + 20.25 * mk[19]) + Gs[9] * (-40.5 * mk[1] + 101.25 * mk[4] - 20.25 * mk[5] - 20.25 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] - 20.25 * mk[12] + 20.25 * mk[13] + 40.5 * mk[14] + 20.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[172] = v_;
      out[248] = v_;
    }
    {
      const double M_ = -40.5 * m[15] - 20.25 * m[25] - 20.25 * m[28] + 101.25 * m[29] + 20.25 * m[40] + 40.5 * m[43] - 20.25 * m[44] + 20.25 * m[47] - 20.25 * m[48] - 40.5 * m[49];
      const double K_ = Gs[1] * (-101.25 * mk[9] - 81.0 * mk[15] - 81.0 * mk[18] + 222.75 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 20.25 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[3] * (-101.25 * mk[6] - 81.0 * mk[12] - 81.0 * mk[14] + 526.5 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 81.0 * mk[25] + 20.25 * mk[27] - 81.0 * mk[28] - 101.25 * mk[29]) + Gs[6] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[9] * (-40.5 * mk[1] - 20.25 * mk[4] - 20.25 * mk[5] + 222.75 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[173] = v_;
      out[268] = v_;
    }
    {
      const double M_ = -40.5 * m[18] - 20.25 * m[28] + 101.25 * m[32] - 20.25 * m[33] + 20.25 * m[43] - 20.25 * m[47] + 40.5 * m[48] - 40.5 * m[52] - 20.25 * m[53] + 20.25 * m[54];
      const double K_ = Gs[2] * (-101.25 * mk[9] - 81.0 * mk[15] + 526.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] - 81.0 * mk[28] + 40.5 * mk[29] - 101.25 * mk[32] - 81.0 * mk[33] + 20.25 * mk[34]) + Gs[3] * (-101.25 * mk[8] - 81.0 * mk[14] + 222.75 * mk[17] - 81.0 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] + 40.5 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[8] * (-40.5 * mk[3] - 20.25 * mk[6] + 222.75 * mk[8] - 20.25 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 101.25 * mk[17] - 81.0 * mk[18] + 20.25 * mk[19]) + Gs[9] * (-40.5 * mk[2] - 20.25 * mk[5] + 101.25 * mk[7] - 20.25 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[16] - 20.25 * mk[17] + 20.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[174] = v_;
      out[288] = v_;
    }
    {
      const double M_ = -40.5 * m[18] - 20.25 * m[28] - 20.25 * m[32] + 101.25 * m[33] + 20.25 * m[43] + 40.5 * m[47] - 20.25 * m[48] + 20.25 * m[52] - 20.25 * m[53] - 40.5 * m[54];
      const double K_ = Gs[2] * (-101.25 * mk[9] - 81.0 * mk[15] - 81.0 * mk[18] + 222.75 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 20.25 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[3] * (-101.25 * mk[8] - 81.0 * mk[14] - 81.0 * mk[17] + 526.5 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 81.0 * mk[28] + 20.25 * mk[31] - 81.0 * mk[32] - 101.25 * mk[33]) + Gs[8] * (-40.5 * mk[3] - 20.25 * mk[6] - 20.25 * mk[8] + 101.25 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] + 20.25 * mk[17] - 20.25 * mk[18] - 40.5 * mk[19]) + Gs[9] * (-40.5 * mk[2] - 20.25 * mk[5] - 20.25 * mk[7] + 222.75 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[175] = v_;
      out[308] = v_;
    }
    {
      const double M_ = 243.0 * m[14] - 121.5 * m[24] - 121.5 * m[27] - 121.5 * m[28];
      const double K_ = Gs[0] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[1] * (607.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[2] * (607.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[3] * (243.0 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[6] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]) + Gs[8] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[176] = v_;
      out[328] = v_;
    }
    {
      const double M_ = 243.0 * m[15] - 121.5 * m[25] - 121.5 * m[28] - 121.5 * m[29];
      const double K_ = Gs[0] * (607.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] - 121.5 * mk[29]) + Gs[1] * (607.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] - 121.5 * mk[19]) + Gs[3] * (850.5 * mk[6] - 243.0 * mk[12] - 243.0 * mk[14] - 243.0 * mk[15]) + Gs[6] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[9] * (243.0 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] - 121.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[177] = v_;
      out[348] = v_;
    }
    {
      const double M_ = 243.0 * m[18] - 121.5 * m[28] - 121.5 * m[32] - 121.5 * m[33];
      const double K_ = Gs[0] * (607.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] - 121.5 * mk[33]) + Gs[2] * (607.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] - 121.5 * mk[19]) + Gs[3] * (850.5 * mk[8] - 243.0 * mk[14] - 243.0 * mk[17] - 243.0 * mk[18]) + Gs[8] * (243.0 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] - 121.5 * mk[9]) + Gs[9] * (243.0 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] - 121.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[178] = v_;
      out[368] = v_;
    }
    {
      const double M_ = 243.0 * m[28] - 121.5 * m[43] - 121.5 * m[47] - 121.5 * m[48];
      const double K_ = Gs[1] * (607.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] - 121.5 * mk[33]) + Gs[2] * (607.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] - 121.5 * mk[29]) + Gs[3] * (607.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[6] * (243.0 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[8] * (243.0 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[9] * (243.0 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[179] = v_;
      out[388] = v_;
    }
    {
      const double M_ = 20.25 * m[9] + 40.5 * m[15] + 40.5 * m[18] - 81.0 * m[19] + 20.25 * m[25] + 40.5 * m[28] - 81.0 * m[29] + 20.25 * m[32] - 81.0 * m[33] + 81.0 * m[34];
      const double K_ = Gs[0] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[3] * (40.5 * mk[3] + 81.0 * mk[6] + 81.0 * mk[8] - 283.5 * mk[9] + 40.5 * mk[12] + 81.0 * mk[14] - 283.5 * mk[15] + 40.5 * mk[17] - 283.5 * mk[18] + 405.0 * mk[19]) + Gs[9] * (20.25 * mk[0] + 40.5 * mk[1] + 40.5 * mk[2] - 202.5 * mk[3] + 20.25 * mk[4] + 40.5 * mk[5] - 202.5 * mk[6] + 20.25 * mk[7] - 202.5 * mk[8] + 506.25 * mk[9]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[189] = v_;
    }
    {
      const double M_ = 20.25 * m[14] - 20.25 * m[24] + 40.5 * m[27] - 20.25 * m[28] - 40.5 * m[39] - 20.25 * m[42] + 101.25 * m[43] + 20.25 * m[46] - 20.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[1] * (20.25 * mk[8] - 81.0 * mk[14] + 40.5 * mk[17] - 20.25 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] + 222.75 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[2] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[6] * (20.25 * mk[2] - 81.0 * mk[5] + 40.5 * mk[7] - 81.0 * mk[8] - 101.25 * mk[11] - 81.0 * mk[13] + 526.5 * mk[14] + 20.25 * mk[16] - 81.0 * mk[17] - 101.25 * mk[18]) + Gs[8] * (20.25 * mk[1] - 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] + 222.75 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[190] = v_;
      out[209] = v_;
    }
    {
      const double M_ = 20.25 * m[14] + 40.5 * m[24] - 20.25 * m[27] - 20.25 * m[28] + 20.25 * m[39] - 20.25 * m[42] - 20.25 * m[43] - 40.5 * m[46] + 101.25 * m[47] - 40.5 * m[48];
      const double K_ = Gs[1] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[2] * (20.25 * mk[6] + 40.5 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] + 222.75 * mk[28] - 40.5 * mk[29]) + Gs[6] * (20.25 * mk[2] + 40.5 * mk[5] - 20.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] + 222.75 * mk[17] - 101.25 * mk[18]) + Gs[8] * (20.25 * mk[1] + 40.5 * mk[4] - 81.0 * mk[5] - 81.0 * mk[6] + 20.25 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] - 101.25 * mk[13] + 526.5 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[191] = v_;
      out[229] = v_;
    }
    {
      const double M_ = 20.25 * m[15] - 20.25 * m[25] + 40.5 * m[28] - 20.25 * m[29] - 40.5 * m[40] - 20.25 * m[43] + 101.25 * m[44] + 20.25 * m[47] - 20.25 * m[48] - 40.5 * m[49];
      const double K_ = Gs[1] * (20.25 * mk[9] - 81.0 * mk[15] + 40.5 * mk[18] - 20.25 * mk[19] - 101.25 * mk[25] - 81.0 * mk[28] + 222.75 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[3] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[6] * (20.25 * mk[3] - 81.0 * mk[6] + 40.5 * mk[8] - 81.0 * mk[9] - 101.25 * mk[12] - 81.0 * mk[14] + 526.5 * mk[15] + 20.25 * mk[17] - 81.0 * mk[18] - 101.25 * mk[19]) + Gs[9] * (20.25 * mk[1] - 20.25 * mk[4] + 40.5 * mk[5] - 81.0 * mk[6] - 40.5 * mk[10] - 20.25 * mk[11] + 222.75 * mk[12] + 20.25 * mk[13] - 81.0 * mk[14] - 101.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[192] = v_;
      out[249] = v_;
    }
    {
      const double M_ = 20.25 * m[15] + 40.5 * m[25] + 40.5 * m[28] - 81.0 * m[29] + 20.25 * m[40] + 40.5 * m[43] - 81.0 * m[44] + 20.25 * m[47] - 81.0 * m[48] + 81.0 * m[49];
      const double K_ = Gs[1] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[3] * (20.25 * mk[6] + 40.5 * mk[12] + 40.5 * mk[14] - 141.75 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 141.75 * mk[25] + 20.25 * mk[27] - 141.75 * mk[28] + 202.5 * mk[29]) + Gs[6] * (20.25 * mk[3] + 40.5 * mk[6] + 40.5 * mk[8] - 141.75 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 141.75 * mk[15] + 20.25 * mk[17] - 141.75 * mk[18] + 202.5 * mk[19]) + Gs[9] * (20.25 * mk[1] + 40.5 * mk[4] + 40.5 * mk[5] - 202.5 * mk[6] + 20.25 * mk[10] + 40.5 * mk[11] - 202.5 * mk[12] + 20.25 * mk[13] - 202.5 * mk[14] + 506.25 * mk[15]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[193] = v_;
      out[269] = v_;
    }
    {
      const double M_ = 20.25 * m[18] + 40.5 * m[28] - 20.25 * m[32] - 20.25 * m[33] + 20.25 * m[43] - 20.25 * m[47] - 20.25 * m[48] - 40.5 * m[52] + 101.25 * m[53] - 40.5 * m[54];
      const double K_ = Gs[2] * (20.25 * mk[9] + 40.5 * mk[15] - 81.0 * mk[18] - 20.25 * mk[19] + 20.25 * mk[25] - 81.0 * mk[28] - 20.25 * mk[29] - 101.25 * mk[32] + 222.75 * mk[33] - 40.5 * mk[34]) + Gs[3] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[8] * (20.25 * mk[3] + 40.5 * mk[6] - 81.0 * mk[8] - 81.0 * mk[9] + 20.25 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] - 101.25 * mk[17] + 526.5 * mk[18] - 101.25 * mk[19]) + Gs[9] * (20.25 * mk[2] + 40.5 * mk[5] - 20.25 * mk[7] - 81.0 * mk[8] + 20.25 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] - 40.5 * mk[16] + 222.75 * mk[17] - 101.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[194] = v_;
      out[289] = v_;
    }
    {
      const double M_ = 20.25 * m[18] + 40.5 * m[28] + 40.5 * m[32] - 81.0 * m[33] + 20.25 * m[43] + 40.5 * m[47] - 81.0 * m[48] + 20.25 * m[52] - 81.0 * m[53] + 81.0 * m[54];
      const double K_ = Gs[2] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[3] * (20.25 * mk[8] + 40.5 * mk[14] + 40.5 * mk[17] - 141.75 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 141.75 * mk[28] + 20.25 * mk[31] - 141.75 * mk[32] + 202.5 * mk[33]) + Gs[8] * (20.25 * mk[3] + 40.5 * mk[6] + 40.5 * mk[8] - 141.75 * mk[9] + 20.25 * mk[12] + 40.5 * mk[14] - 141.75 * mk[15] + 20.25 * mk[17] - 141.75 * mk[18] + 202.5 * mk[19]) + Gs[9] * (20.25 * mk[2] + 40.5 * mk[5] + 40.5 * mk[7] - 202.5 * mk[8] + 20.25 * mk[11] + 40.5 * mk[13] - 202.5 * mk[14] + 20.25 * mk[16] - 202.5 * mk[17] + 506.25 * mk[18]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[195] = v_;
      out[309] = v_;
    }
    {
      const double M_ = -121.5 * m[14] - 121.5 * m[24] - 121.5 * m[27] + 243.0 * m[28];
      const double K_ = Gs[0] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 243.0 * mk[28]) + Gs[1] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 243.0 * mk[18]) + Gs[2] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 243.0 * mk[15]) + Gs[3] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]) + Gs[6] * (-121.5 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] + 607.5 * mk[8]) + Gs[8] * (-121.5 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] + 607.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[196] = v_;
      out[329] = v_;
    }
    {
      const double M_ = -121.5 * m[15] - 121.5 * m[25] - 121.5 * m[28] + 243.0 * m[29];
      const double K_ = Gs[0] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[1] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[3] * (-243.0 * mk[6] - 243.0 * mk[12] - 243.0 * mk[14] + 850.5 * mk[15]) + Gs[6] * (-121.5 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] + 607.5 * mk[9]) + Gs[9] * (-121.5 * mk[1] - 121.5 * mk[4] - 121.5 * mk[5] + 607.5 * mk[6]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[197] = v_;
      out[349] = v_;
    }
    {
      const double M_ = -121.5 * m[18] - 121.5 * m[28] - 121.5 * m[32] + 243.0 * m[33];
      const double K_ = Gs[0] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[2] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[3] * (-243.0 * mk[8] - 243.0 * mk[14] - 243.0 * mk[17] + 850.5 * mk[18]) + Gs[8] * (-121.5 * mk[3] - 121.5 * mk[6] - 121.5 * mk[8] + 607.5 * mk[9]) + Gs[9] * (-121.5 * mk[2] - 121.5 * mk[5] - 121.5 * mk[7] + 607.5 * mk[8]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[198] = v_;
      out[369] = v_;
    }
    {
      const double M_ = -121.5 * m[28] - 121.5 * m[43] - 121.5 * m[47] + 243.0 * m[48];
      const double K_ = Gs[1] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[2] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[3] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 243.0 * mk[28]) + Gs[6] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 607.5 * mk[18]) + Gs[8] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 607.5 * mk[15]) + Gs[9] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[199] = v_;
      out[389] = v_;
    }
    {
      const double M_ = 20.25 * m[23] - 81.0 * m[38] + 40.5 * m[41] + 40.5 * m[42] + 81.0 * m[59] - 81.0 * m[62] - 81.0 * m[63] + 20.25 * m[66] + 40.5 * m[67] + 20.25 * m[68];
      const double K_ = Gs[4] * (20.25 * mk[7] - 202.5 * mk[13] + 40.5 * mk[16] + 40.5 * mk[17] + 506.25 * mk[23] - 202.5 * mk[26] - 202.5 * mk[27] + 20.25 * mk[30] + 40.5 * mk[31] + 20.25 * mk[32]) + Gs[5] * (40.5 * mk[5] - 283.5 * mk[11] + 81.0 * mk[13] + 81.0 * mk[14] + 405.0 * mk[21] - 283.5 * mk[23] - 283.5 * mk[24] + 40.5 * mk[26] + 81.0 * mk[27] + 40.5 * mk[28]) + Gs[7] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[210] = v_;
    }
    {
      const double M_ = 20.25 * m[23] - 20.25 * m[38] - 20.25 * m[41] + 40.5 * m[42] - 40.5 * m[59] + 101.25 * m[62] - 20.25 * m[63] - 40.5 * m[66] - 20.25 * m[67] + 20.25 * m[68];
      const double K_ = Gs[4] * (20.25 * mk[7] - 81.0 * mk[13] - 20.25 * mk[16] + 40.5 * mk[17] - 101.25 * mk[23] + 222.75 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[5] * (40.5 * mk[5] - 101.25 * mk[11] - 101.25 * mk[13] + 81.0 * mk[14] - 141.75 * mk[21] + 627.75 * mk[23] - 101.25 * mk[24] - 141.75 * mk[26] - 101.25 * mk[27] + 40.5 * mk[28]) + Gs[7] * (20.25 * mk[4] - 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 40.5 * mk[20] + 222.75 * mk[21] - 20.25 * mk[22] - 101.25 * mk[23] - 81.0 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[211] = v_;
      out[230] = v_;
    }
    {
      const double M_ = 20.25 * m[24] - 81.0 * m[39] + 40.5 * m[42] + 40.5 * m[43] + 81.0 * m[60] - 81.0 * m[63] - 81.0 * m[64] + 20.25 * m[67] + 40.5 * m[68] + 20.25 * m[69];
      const double K_ = Gs[4] * (20.25 * mk[8] - 202.5 * mk[14] + 40.5 * mk[17] + 40.5 * mk[18] + 506.25 * mk[24] - 202.5 * mk[27] - 202.5 * mk[28] + 20.25 * mk[31] + 40.5 * mk[32] + 20.25 * mk[33]) + Gs[5] * (20.25 * mk[6] - 141.75 * mk[12] + 40.5 * mk[14] + 40.5 * mk[15] + 202.5 * mk[22] - 141.75 * mk[24] - 141.75 * mk[25] + 20.25 * mk[27] + 40.5 * mk[28] + 20.25 * mk[29]) + Gs[6] * (20.25 * mk[5] - 141.75 * mk[11] + 40.5 * mk[13] + 40.5 * mk[14] + 202.5 * mk[21] - 141.75 * mk[23] - 141.75 * mk[24] + 20.25 * mk[26] + 40.5 * mk[27] + 20.25 * mk[28]) + Gs[8] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[212] = v_;
      out[250] = v_;
    }
    {
      const double M_ = 20.25 * m[24] - 20.25 * m[39] + 40.5 * m[42] - 20.25 * m[43] - 40.5 * m[60] - 20.25 * m[63] + 101.25 * m[64] + 20.25 * m[67] - 20.25 * m[68] - 40.5 * m[69];
      const double K_ = Gs[4] * (20.25 * mk[8] - 81.0 * mk[14] + 40.5 * mk[17] - 20.25 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] + 222.75 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[5] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[6] * (20.25 * mk[5] - 81.0 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] - 101.25 * mk[21] - 81.0 * mk[23] + 526.5 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]) + Gs[8] * (20.25 * mk[4] - 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] + 222.75 * mk[22] + 20.25 * mk[23] - 81.0 * mk[24] - 101.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[213] = v_;
      out[270] = v_;
    }
    {
      const double M_ = 20.25 * m[27] - 20.25 * m[42] - 20.25 * m[46] + 40.5 * m[47] - 40.5 * m[63] + 101.25 * m[67] - 20.25 * m[68] - 40.5 * m[72] - 20.25 * m[73] + 20.25 * m[74];
      const double K_ = Gs[5] * (20.25 * mk[8] - 81.0 * mk[14] - 81.0 * mk[17] + 40.5 * mk[18] - 101.25 * mk[24] + 526.5 * mk[27] - 81.0 * mk[28] - 101.25 * mk[31] - 81.0 * mk[32] + 20.25 * mk[33]) + Gs[6] * (20.25 * mk[7] - 81.0 * mk[13] - 20.25 * mk[16] + 40.5 * mk[17] - 101.25 * mk[23] + 222.75 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] - 20.25 * mk[31] + 20.25 * mk[32]) + Gs[7] * (20.25 * mk[6] - 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 40.5 * mk[22] + 222.75 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[8] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[214] = v_;
      out[290] = v_;
    }
    {
      const double M_ = 20.25 * m[27] - 20.25 * m[42] + 40.5 * m[46] - 20.25 * m[47] - 40.5 * m[63] - 20.25 * m[67] + 101.25 * m[68] + 20.25 * m[72] - 20.25 * m[73] - 40.5 * m[74];
      const double K_ = Gs[5] * (20.25 * mk[8] - 81.0 * mk[14] + 40.5 * mk[17] - 20.25 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] + 222.75 * mk[28] + 20.25 * mk[31] - 20.25 * mk[32] - 40.5 * mk[33]) + Gs[6] * (20.25 * mk[7] - 81.0 * mk[13] + 40.5 * mk[16] - 81.0 * mk[17] - 101.25 * mk[23] - 81.0 * mk[26] + 526.5 * mk[27] + 20.25 * mk[30] - 81.0 * mk[31] - 101.25 * mk[32]) + Gs[7] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[8] * (20.25 * mk[5] - 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] + 222.75 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[215] = v_;
      out[310] = v_;
    }
    {
      const double M_ = -121.5 * m[23] + 243.0 * m[38] - 121.5 * m[41] - 121.5 * m[42];
      const double K_ = Gs[1] * (-121.5 * mk[13] + 607.5 * mk[23] - 121.5 * mk[26] - 121.5 * mk[27]) + Gs[2] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[4] * (-121.5 * mk[7] + 607.5 * mk[13] - 121.5 * mk[16] - 121.5 * mk[17]) + Gs[5] * (-243.0 * mk[5] + 850.5 * mk[11] - 243.0 * mk[13] - 243.0 * mk[14]) + Gs[7] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[216] = v_;
      out[330] = v_;
    }
    {
      const double M_ = -121.5 * m[24] + 243.0 * m[39] - 121.5 * m[42] - 121.5 * m[43];
      const double K_ = Gs[1] * (-121.5 * mk[14] + 607.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[2] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[4] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[5] * (-121.5 * mk[6] + 243.0 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[6] * (-121.5 * mk[5] + 607.5 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[8] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[217] = v_;
      out[350] = v_;
    }
    {
      const double M_ = -121.5 * m[27] + 243.0 * m[42] - 121.5 * m[46] - 121.5 * m[47];
      const double K_ = Gs[1] * (-121.5 * mk[17] + 607.5 * mk[27] - 121.5 * mk[31] - 121.5 * mk[32]) + Gs[2] * (-121.5 * mk[14] + 243.0 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[5] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[6] * (-121.5 * mk[7] + 607.5 * mk[13] - 121.5 * mk[16] - 121.5 * mk[17]) + Gs[7] * (-121.5 * mk[6] + 243.0 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[8] * (-121.5 * mk[5] + 243.0 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[218] = v_;
      out[370] = v_;
    }
    {
      const double M_ = -121.5 * m[42] + 243.0 * m[63] - 121.5 * m[67] - 121.5 * m[68];
      const double K_ = Gs[4] * (-121.5 * mk[17] + 607.5 * mk[27] - 121.5 * mk[31] - 121.5 * mk[32]) + Gs[5] * (-243.0 * mk[14] + 850.5 * mk[24] - 243.0 * mk[27] - 243.0 * mk[28]) + Gs[6] * (-121.5 * mk[13] + 607.5 * mk[23] - 121.5 * mk[26] - 121.5 * mk[27]) + Gs[7] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[8] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[219] = v_;
      out[390] = v_;
    }
    {
      const double M_ = 20.25 * m[23] + 40.5 * m[38] - 81.0 * m[41] + 40.5 * m[42] + 20.25 * m[59] - 81.0 * m[62] + 40.5 * m[63] + 81.0 * m[66] - 81.0 * m[67] + 20.25 * m[68];
      const double K_ = Gs[4] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]) + Gs[5] * (40.5 * mk[5] + 81.0 * mk[11] - 283.5 * mk[13] + 81.0 * mk[14] + 40.5 * mk[21] - 283.5 * mk[23] + 81.0 * mk[24] + 405.0 * mk[26] - 283.5 * mk[27] + 40.5 * mk[28]) + Gs[7] * (20.25 * mk[4] + 40.5 * mk[10] - 202.5 * mk[11] + 40.5 * mk[12] + 20.25 * mk[20] - 202.5 * mk[21] + 40.5 * mk[22] + 506.25 * mk[23] - 202.5 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[231] = v_;
    }
    {
      const double M_ = 20.25 * m[24] - 20.25 * m[39] - 20.25 * m[42] + 40.5 * m[43] - 40.5 * m[60] + 101.25 * m[63] - 20.25 * m[64] - 40.5 * m[67] - 20.25 * m[68] + 20.25 * m[69];
      const double K_ = Gs[4] * (20.25 * mk[8] - 81.0 * mk[14] - 20.25 * mk[17] + 40.5 * mk[18] - 101.25 * mk[24] + 222.75 * mk[27] - 81.0 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[5] * (20.25 * mk[6] - 81.0 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 101.25 * mk[22] + 526.5 * mk[24] - 81.0 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[6] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]) + Gs[8] * (20.25 * mk[4] - 20.25 * mk[10] - 81.0 * mk[11] + 40.5 * mk[12] - 40.5 * mk[20] + 222.75 * mk[21] - 20.25 * mk[22] - 101.25 * mk[23] - 81.0 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[232] = v_;
      out[251] = v_;
    }
    {
      const double M_ = 20.25 * m[24] + 40.5 * m[39] - 20.25 * m[42] - 20.25 * m[43] + 20.25 * m[60] - 20.25 * m[63] - 20.25 * m[64] - 40.5 * m[67] + 101.25 * m[68] - 40.5 * m[69];
      const double K_ = Gs[4] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[5] * (20.25 * mk[6] + 40.5 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] + 222.75 * mk[28] - 40.5 * mk[29]) + Gs[6] * (20.25 * mk[5] + 40.5 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] - 81.0 * mk[24] - 40.5 * mk[26] + 222.75 * mk[27] - 101.25 * mk[28]) + Gs[8] * (20.25 * mk[4] + 40.5 * mk[10] - 81.0 * mk[11] - 81.0 * mk[12] + 20.25 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] - 101.25 * mk[23] + 526.5 * mk[24] - 101.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[233] = v_;
      out[271] = v_;
    }
    {
      const double M_ = 20.25 * m[27] + 40.5 * m[42] - 81.0 * m[46] + 40.5 * m[47] + 20.25 * m[63] - 81.0 * m[67] + 40.5 * m[68] + 81.0 * m[72] - 81.0 * m[73] + 20.25 * m[74];
      const double K_ = Gs[5] * (20.25 * mk[8] + 40.5 * mk[14] - 141.75 * mk[17] + 40.5 * mk[18] + 20.25 * mk[24] - 141.75 * mk[27] + 40.5 * mk[28] + 202.5 * mk[31] - 141.75 * mk[32] + 20.25 * mk[33]) + Gs[6] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]) + Gs[7] * (20.25 * mk[6] + 40.5 * mk[12] - 202.5 * mk[14] + 40.5 * mk[15] + 20.25 * mk[22] - 202.5 * mk[24] + 40.5 * mk[25] + 506.25 * mk[27] - 202.5 * mk[28] + 20.25 * mk[29]) + Gs[8] * (20.25 * mk[5] + 40.5 * mk[11] - 141.75 * mk[13] + 40.5 * mk[14] + 20.25 * mk[21] - 141.75 * mk[23] + 40.5 * mk[24] + 202.5 * mk[26] - 141.75 * mk[27] + 20.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[234] = v_;
      out[291] = v_;
    }
    {
      const double M_ = 20.25 * m[27] + 40.5 * m[42] - 20.25 * m[46] - 20.25 * m[47] + 20.25 * m[63] - 20.25 * m[67] - 20.25 * m[68] - 40.5 * m[72] + 101.25 * m[73] - 40.5 * m[74];
      const double K_ = Gs[5] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[6] * (20.25 * mk[7] + 40.5 * mk[13] - 20.25 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] + 222.75 * mk[31] - 101.25 * mk[32]) + Gs[7] * (20.25 * mk[6] + 40.5 * mk[12] - 81.0 * mk[14] - 20.25 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] + 222.75 * mk[28] - 40.5 * mk[29]) + Gs[8] * (20.25 * mk[5] + 40.5 * mk[11] - 81.0 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 81.0 * mk[23] - 81.0 * mk[24] - 101.25 * mk[26] + 526.5 * mk[27] - 101.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[235] = v_;
      out[311] = v_;
    }
    {
      const double M_ = -121.5 * m[23] - 121.5 * m[38] + 243.0 * m[41] - 121.5 * m[42];
      const double K_ = Gs[1] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]) + Gs[2] * (-121.5 * mk[11] - 121.5 * mk[21] + 607.5 * mk[23] - 121.5 * mk[24]) + Gs[4] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]) + Gs[5] * (-243.0 * mk[5] - 243.0 * mk[11] + 850.5 * mk[13] - 243.0 * mk[14]) + Gs[7] * (-121.5 * mk[4] - 121.5 * mk[10] + 607.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[236] = v_;
      out[331] = v_;
    }
    {
      const double M_ = -121.5 * m[24] - 121.5 * m[39] + 243.0 * m[42] - 121.5 * m[43];
      const double K_ = Gs[1] * (-121.5 * mk[14] - 121.5 * mk[24] + 243.0 * mk[27] - 121.5 * mk[28]) + Gs[2] * (-121.5 * mk[12] - 121.5 * mk[22] + 607.5 * mk[24] - 121.5 * mk[25]) + Gs[4] * (-121.5 * mk[8] - 121.5 * mk[14] + 243.0 * mk[17] - 121.5 * mk[18]) + Gs[5] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[6] * (-121.5 * mk[5] - 121.5 * mk[11] + 243.0 * mk[13] - 121.5 * mk[14]) + Gs[8] * (-121.5 * mk[4] - 121.5 * mk[10] + 607.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[237] = v_;
      out[351] = v_;
    }
    {
      const double M_ = -121.5 * m[27] - 121.5 * m[42] + 243.0 * m[46] - 121.5 * m[47];
      const double K_ = Gs[1] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[2] * (-121.5 * mk[14] - 121.5 * mk[24] + 607.5 * mk[27] - 121.5 * mk[28]) + Gs[5] * (-121.5 * mk[8] - 121.5 * mk[14] + 243.0 * mk[17] - 121.5 * mk[18]) + Gs[6] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]) + Gs[7] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[8] * (-121.5 * mk[5] - 121.5 * mk[11] + 607.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[238] = v_;
      out[371] = v_;
    }
    {
      const double M_ = -121.5 * m[42] - 121.5 * m[63] + 243.0 * m[67] - 121.5 * m[68];
      const double K_ = Gs[4] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[5] * (-243.0 * mk[14] - 243.0 * mk[24] + 850.5 * mk[27] - 243.0 * mk[28]) + Gs[6] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]) + Gs[7] * (-121.5 * mk[12] - 121.5 * mk[22] + 607.5 * mk[24] - 121.5 * mk[25]) + Gs[8] * (-121.5 * mk[11] - 121.5 * mk[21] + 607.5 * mk[23] - 121.5 * mk[24]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[239] = v_;
      out[391] = v_;
    }
    {
      const double M_ = 20.25 * m[25] - 81.0 * m[40] + 40.5 * m[43] + 40.5 * m[44] + 81.0 * m[61] - 81.0 * m[64] - 81.0 * m[65] + 20.25 * m[68] + 40.5 * m[69] + 20.25 * m[70];
      const double K_ = Gs[4] * (20.25 * mk[9] - 202.5 * mk[15] + 40.5 * mk[18] + 40.5 * mk[19] + 506.25 * mk[25] - 202.5 * mk[28] - 202.5 * mk[29] + 20.25 * mk[32] + 40.5 * mk[33] + 20.25 * mk[34]) + Gs[6] * (40.5 * mk[6] - 283.5 * mk[12] + 81.0 * mk[14] + 81.0 * mk[15] + 405.0 * mk[22] - 283.5 * mk[24] - 283.5 * mk[25] + 40.5 * mk[27] + 81.0 * mk[28] + 40.5 * mk[29]) + Gs[9] * (20.25 * mk[4] - 81.0 * mk[10] + 40.5 * mk[11] + 40.5 * mk[12] + 81.0 * mk[20] - 81.0 * mk[21] - 81.0 * mk[22] + 20.25 * mk[23] + 40.5 * mk[24] + 20.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[252] = v_;
    }
    {
      const double M_ = 20.25 * m[25] - 20.25 * m[40] + 40.5 * m[43] - 20.25 * m[44] - 40.5 * m[61] - 20.25 * m[64] + 101.25 * m[65] + 20.25 * m[68] - 20.25 * m[69] - 40.5 * m[70];
      const double K_ = Gs[4] * (20.25 * mk[9] - 81.0 * mk[15] + 40.5 * mk[18] - 20.25 * mk[19] - 101.25 * mk[25] - 81.0 * mk[28] + 222.75 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[6] * (40.5 * mk[6] - 101.25 * mk[12] + 81.0 * mk[14] - 101.25 * mk[15] - 141.75 * mk[22] - 101.25 * mk[24] + 627.75 * mk[25] + 40.5 * mk[27] - 101.25 * mk[28] - 141.75 * mk[29]) + Gs[9] * (20.25 * mk[4] - 20.25 * mk[10] + 40.5 * mk[11] - 81.0 * mk[12] - 40.5 * mk[20] - 20.25 * mk[21] + 222.75 * mk[22] + 20.25 * mk[23] - 81.0 * mk[24] - 101.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[253] = v_;
      out[272] = v_;
    }
    {
      const double M_ = 20.25 * m[28] - 20.25 * m[43] - 20.25 * m[47] + 40.5 * m[48] - 40.5 * m[64] + 101.25 * m[68] - 20.25 * m[69] - 40.5 * m[73] - 20.25 * m[74] + 20.25 * m[75];
      const double K_ = Gs[5] * (20.25 * mk[9] - 81.0 * mk[15] - 81.0 * mk[18] + 40.5 * mk[19] - 101.25 * mk[25] + 526.5 * mk[28] - 81.0 * mk[29] - 101.25 * mk[32] - 81.0 * mk[33] + 20.25 * mk[34]) + Gs[6] * (20.25 * mk[8] - 81.0 * mk[14] - 20.25 * mk[17] + 40.5 * mk[18] - 101.25 * mk[24] + 222.75 * mk[27] - 81.0 * mk[28] - 40.5 * mk[31] - 20.25 * mk[32] + 20.25 * mk[33]) + Gs[8] * (20.25 * mk[6] - 20.25 * mk[12] - 81.0 * mk[14] + 40.5 * mk[15] - 40.5 * mk[22] + 222.75 * mk[24] - 20.25 * mk[25] - 101.25 * mk[27] - 81.0 * mk[28] + 20.25 * mk[29]) + Gs[9] * (20.25 * mk[5] - 20.25 * mk[11] - 20.25 * mk[13] + 40.5 * mk[14] - 40.5 * mk[21] + 101.25 * mk[23] - 20.25 * mk[24] - 40.5 * mk[26] - 20.25 * mk[27] + 20.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[254] = v_;
      out[292] = v_;
    }
    {
      const double M_ = 20.25 * m[28] - 20.25 * m[43] + 40.5 * m[47] - 20.25 * m[48] - 40.5 * m[64] - 20.25 * m[68] + 101.25 * m[69] + 20.25 * m[73] - 20.25 * m[74] - 40.5 * m[75];
      const double K_ = Gs[5] * (20.25 * mk[9] - 81.0 * mk[15] + 40.5 * mk[18] - 20.25 * mk[19] - 101.25 * mk[25] - 81.0 * mk[28] + 222.75 * mk[29] + 20.25 * mk[32] - 20.25 * mk[33] - 40.5 * mk[34]) + Gs[6] * (20.25 * mk[8] - 81.0 * mk[14] + 40.5 * mk[17] - 81.0 * mk[18] - 101.25 * mk[24] - 81.0 * mk[27] + 526.5 * mk[28] + 20.25 * mk[31] - 81.0 * mk[32] - 101.25 * mk[33]) + Gs[8] * (20.25 * mk[6] - 20.25 * mk[12] + 40.5 * mk[14] - 20.25 * mk[15] - 40.5 * mk[22] - 20.25 * mk[24] + 101.25 * mk[25] + 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[29]) + Gs[9] * (20.25 * mk[5] - 20.25 * mk[11] + 40.5 * mk[13] - 81.0 * mk[14] - 40.5 * mk[21] - 20.25 * mk[23] + 222.75 * mk[24] + 20.25 * mk[26] - 81.0 * mk[27] - 101.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[255] = v_;
      out[312] = v_;
    }
    {
      const double M_ = -121.5 * m[24] + 243.0 * m[39] - 121.5 * m[42] - 121.5 * m[43];
      const double K_ = Gs[1] * (-121.5 * mk[14] + 607.5 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[3] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]) + Gs[4] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[5] * (-121.5 * mk[6] + 607.5 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[6] * (-121.5 * mk[5] + 243.0 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]) + Gs[8] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[256] = v_;
      out[332] = v_;
    }
    {
      const double M_ = -121.5 * m[25] + 243.0 * m[40] - 121.5 * m[43] - 121.5 * m[44];
      const double K_ = Gs[1] * (-121.5 * mk[15] + 607.5 * mk[25] - 121.5 * mk[28] - 121.5 * mk[29]) + Gs[3] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[4] * (-121.5 * mk[9] + 607.5 * mk[15] - 121.5 * mk[18] - 121.5 * mk[19]) + Gs[6] * (-243.0 * mk[6] + 850.5 * mk[12] - 243.0 * mk[14] - 243.0 * mk[15]) + Gs[9] * (-121.5 * mk[4] + 243.0 * mk[10] - 121.5 * mk[11] - 121.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[257] = v_;
      out[352] = v_;
    }
    {
      const double M_ = -121.5 * m[28] + 243.0 * m[43] - 121.5 * m[47] - 121.5 * m[48];
      const double K_ = Gs[1] * (-121.5 * mk[18] + 607.5 * mk[28] - 121.5 * mk[32] - 121.5 * mk[33]) + Gs[3] * (-121.5 * mk[14] + 243.0 * mk[24] - 121.5 * mk[27] - 121.5 * mk[28]) + Gs[5] * (-121.5 * mk[9] + 607.5 * mk[15] - 121.5 * mk[18] - 121.5 * mk[19]) + Gs[6] * (-121.5 * mk[8] + 607.5 * mk[14] - 121.5 * mk[17] - 121.5 * mk[18]) + Gs[8] * (-121.5 * mk[6] + 243.0 * mk[12] - 121.5 * mk[14] - 121.5 * mk[15]) + Gs[9] * (-121.5 * mk[5] + 243.0 * mk[11] - 121.5 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[258] = v_;
      out[372] = v_;
    }
    {
      const double M_ = -121.5 * m[43] + 243.0 * m[64] - 121.5 * m[68] - 121.5 * m[69];
      const double K_ = Gs[4] * (-121.5 * mk[18] + 607.5 * mk[28] - 121.5 * mk[32] - 121.5 * mk[33]) + Gs[5] * (-121.5 * mk[15] + 607.5 * mk[25] - 121.5 * mk[28] - 121.5 * mk[29]) + Gs[6] * (-243.0 * mk[14] + 850.5 * mk[24] - 243.0 * mk[27] - 243.0 * mk[28]) + Gs[8] * (-121.5 * mk[12] + 243.0 * mk[22] - 121.5 * mk[24] - 121.5 * mk[25]) + Gs[9] * (-121.5 * mk[11] + 243.0 * mk[21] - 121.5 * mk[23] - 121.5 * mk[24]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[259] = v_;
      out[392] = v_;
    }
    {
      const double M_ = 20.25 * m[25] + 40.5 * m[40] + 40.5 * m[43] - 81.0 * m[44] + 20.25 * m[61] + 40.5 * m[64] - 81.0 * m[65] + 20.25 * m[68] - 81.0 * m[69] + 81.0 * m[70];
      const double K_ = Gs[4] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[6] * (40.5 * mk[6] + 81.0 * mk[12] + 81.0 * mk[14] - 283.5 * mk[15] + 40.5 * mk[22] + 81.0 * mk[24] - 283.5 * mk[25] + 40.5 * mk[27] - 283.5 * mk[28] + 405.0 * mk[29]) + Gs[9] * (20.25 * mk[4] + 40.5 * mk[10] + 40.5 * mk[11] - 202.5 * mk[12] + 20.25 * mk[20] + 40.5 * mk[21] - 202.5 * mk[22] + 20.25 * mk[23] - 202.5 * mk[24] + 506.25 * mk[25]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[273] = v_;
    }
    {
      const double M_ = 20.25 * m[28] + 40.5 * m[43] - 20.25 * m[47] - 20.25 * m[48] + 20.25 * m[64] - 20.25 * m[68] - 20.25 * m[69] - 40.5 * m[73] + 101.25 * m[74] - 40.5 * m[75];
      const double K_ = Gs[5] * (20.25 * mk[9] + 40.5 * mk[15] - 81.0 * mk[18] - 20.25 * mk[19] + 20.25 * mk[25] - 81.0 * mk[28] - 20.25 * mk[29] - 101.25 * mk[32] + 222.75 * mk[33] - 40.5 * mk[34]) + Gs[6] * (20.25 * mk[8] + 40.5 * mk[14] - 20.25 * mk[17] - 20.25 * mk[18] + 20.25 * mk[24] - 20.25 * mk[27] - 20.25 * mk[28] - 40.5 * mk[31] + 101.25 * mk[32] - 40.5 * mk[33]) + Gs[8] * (20.25 * mk[6] + 40.5 * mk[12] - 81.0 * mk[14] - 81.0 * mk[15] + 20.25 * mk[22] - 81.0 * mk[24] - 81.0 * mk[25] - 101.25 * mk[27] + 526.5 * mk[28] - 101.25 * mk[29]) + Gs[9] * (20.25 * mk[5] + 40.5 * mk[11] - 20.25 * mk[13] - 81.0 * mk[14] + 20.25 * mk[21] - 20.25 * mk[23] - 81.0 * mk[24] - 40.5 * mk[26] + 222.75 * mk[27] - 101.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[274] = v_;
      out[293] = v_;
    }
    {
      const double M_ = 20.25 * m[28] + 40.5 * m[43] + 40.5 * m[47] - 81.0 * m[48] + 20.25 * m[64] + 40.5 * m[68] - 81.0 * m[69] + 20.25 * m[73] - 81.0 * m[74] + 81.0 * m[75];
      const double K_ = Gs[5] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[6] * (20.25 * mk[8] + 40.5 * mk[14] + 40.5 * mk[17] - 141.75 * mk[18] + 20.25 * mk[24] + 40.5 * mk[27] - 141.75 * mk[28] + 20.25 * mk[31] - 141.75 * mk[32] + 202.5 * mk[33]) + Gs[8] * (20.25 * mk[6] + 40.5 * mk[12] + 40.5 * mk[14] - 141.75 * mk[15] + 20.25 * mk[22] + 40.5 * mk[24] - 141.75 * mk[25] + 20.25 * mk[27] - 141.75 * mk[28] + 202.5 * mk[29]) + Gs[9] * (20.25 * mk[5] + 40.5 * mk[11] + 40.5 * mk[13] - 202.5 * mk[14] + 20.25 * mk[21] + 40.5 * mk[23] - 202.5 * mk[24] + 20.25 * mk[26] - 202.5 * mk[27] + 506.25 * mk[28]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[275] = v_;
      out[313] = v_;
    }
    {
      const double M_ = -121.5 * m[24] - 121.5 * m[39] - 121.5 * m[42] + 243.0 * m[43];
      const double K_ = Gs[1] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 243.0 * mk[28]) + Gs[3] * (-121.5 * mk[11] - 121.5 * mk[21] - 121.5 * mk[23] + 607.5 * mk[24]) + Gs[4] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 243.0 * mk[18]) + Gs[5] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 243.0 * mk[15]) + Gs[6] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]) + Gs[8] * (-121.5 * mk[4] - 121.5 * mk[10] - 121.5 * mk[11] + 607.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[276] = v_;
      out[333] = v_;
    }
    {
      const double M_ = -121.5 * m[25] - 121.5 * m[40] - 121.5 * m[43] + 243.0 * m[44];
      const double K_ = Gs[1] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[3] * (-121.5 * mk[12] - 121.5 * mk[22] - 121.5 * mk[24] + 607.5 * mk[25]) + Gs[4] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[6] * (-243.0 * mk[6] - 243.0 * mk[12] - 243.0 * mk[14] + 850.5 * mk[15]) + Gs[9] * (-121.5 * mk[4] - 121.5 * mk[10] - 121.5 * mk[11] + 607.5 * mk[12]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[277] = v_;
      out[353] = v_;
    }
    {
      const double M_ = -121.5 * m[28] - 121.5 * m[43] - 121.5 * m[47] + 243.0 * m[48];
      const double K_ = Gs[1] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[3] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 607.5 * mk[28]) + Gs[5] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[6] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 243.0 * mk[18]) + Gs[8] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 607.5 * mk[15]) + Gs[9] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[278] = v_;
      out[373] = v_;
    }
    {
      const double M_ = -121.5 * m[43] - 121.5 * m[64] - 121.5 * m[68] + 243.0 * m[69];
      const double K_ = Gs[4] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[5] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[6] * (-243.0 * mk[14] - 243.0 * mk[24] - 243.0 * mk[27] + 850.5 * mk[28]) + Gs[8] * (-121.5 * mk[12] - 121.5 * mk[22] - 121.5 * mk[24] + 607.5 * mk[25]) + Gs[9] * (-121.5 * mk[11] - 121.5 * mk[21] - 121.5 * mk[23] + 607.5 * mk[24]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[279] = v_;
      out[393] = v_;
    }
    {
      const double M_ = 20.25 * m[32] + 40.5 * m[47] - 81.0 * m[52] + 40.5 * m[53] + 20.25 * m[68] - 81.0 * m[73] + 40.5 * m[74] + 81.0 * m[79] - 81.0 * m[80] + 20.25 * m[81];
      const double K_ = Gs[7] * (20.25 * mk[9] + 40.5 * mk[15] - 202.5 * mk[18] + 40.5 * mk[19] + 20.25 * mk[25] - 202.5 * mk[28] + 40.5 * mk[29] + 506.25 * mk[32] - 202.5 * mk[33] + 20.25 * mk[34]) + Gs[8] * (40.5 * mk[8] + 81.0 * mk[14] - 283.5 * mk[17] + 81.0 * mk[18] + 40.5 * mk[24] - 283.5 * mk[27] + 81.0 * mk[28] + 405.0 * mk[31] - 283.5 * mk[32] + 40.5 * mk[33]) + Gs[9] * (20.25 * mk[7] + 40.5 * mk[13] - 81.0 * mk[16] + 40.5 * mk[17] + 20.25 * mk[23] - 81.0 * mk[26] + 40.5 * mk[27] + 81.0 * mk[30] - 81.0 * mk[31] + 20.25 * mk[32]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[294] = v_;
    }
    {
      const double M_ = 20.25 * m[32] + 40.5 * m[47] - 20.25 * m[52] - 20.25 * m[53] + 20.25 * m[68] - 20.25 * m[73] - 20.25 * m[74] - 40.5 * m[79] + 101.25 * m[80] - 40.5 * m[81];
      const double K_ = Gs[7] * (20.25 * mk[9] + 40.5 * mk[15] - 81.0 * mk[18] - 20.25 * mk[19] + 20.25 * mk[25] - 81.0 * mk[28] - 20.25 * mk[29] - 101.25 * mk[32] + 222.75 * mk[33] - 40.5 * mk[34]) + Gs[8] * (40.5 * mk[8] + 81.0 * mk[14] - 101.25 * mk[17] - 101.25 * mk[18] + 40.5 * mk[24] - 101.25 * mk[27] - 101.25 * mk[28] - 141.75 * mk[31] + 627.75 * mk[32] - 141.75 * mk[33]) + Gs[9] * (20.25 * mk[7] + 40.5 * mk[13] - 20.25 * mk[16] - 81.0 * mk[17] + 20.25 * mk[23] - 20.25 * mk[26] - 81.0 * mk[27] - 40.5 * mk[30] + 222.75 * mk[31] - 101.25 * mk[32]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[295] = v_;
      out[314] = v_;
    }
    {
      const double M_ = -121.5 * m[27] - 121.5 * m[42] + 243.0 * m[46] - 121.5 * m[47];
      const double K_ = Gs[2] * (-121.5 * mk[14] - 121.5 * mk[24] + 607.5 * mk[27] - 121.5 * mk[28]) + Gs[3] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]) + Gs[5] * (-121.5 * mk[8] - 121.5 * mk[14] + 607.5 * mk[17] - 121.5 * mk[18]) + Gs[6] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]) + Gs[7] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[8] * (-121.5 * mk[5] - 121.5 * mk[11] + 243.0 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[296] = v_;
      out[334] = v_;
    }
    {
      const double M_ = -121.5 * m[28] - 121.5 * m[43] + 243.0 * m[47] - 121.5 * m[48];
      const double K_ = Gs[2] * (-121.5 * mk[15] - 121.5 * mk[25] + 607.5 * mk[28] - 121.5 * mk[29]) + Gs[3] * (-121.5 * mk[14] - 121.5 * mk[24] + 243.0 * mk[27] - 121.5 * mk[28]) + Gs[5] * (-121.5 * mk[9] - 121.5 * mk[15] + 607.5 * mk[18] - 121.5 * mk[19]) + Gs[6] * (-121.5 * mk[8] - 121.5 * mk[14] + 243.0 * mk[17] - 121.5 * mk[18]) + Gs[8] * (-121.5 * mk[6] - 121.5 * mk[12] + 607.5 * mk[14] - 121.5 * mk[15]) + Gs[9] * (-121.5 * mk[5] - 121.5 * mk[11] + 243.0 * mk[13] - 121.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[297] = v_;
      out[354] = v_;
    }
    {
      const double M_ = -121.5 * m[32] - 121.5 * m[47] + 243.0 * m[52] - 121.5 * m[53];
      const double K_ = Gs[2] * (-121.5 * mk[18] - 121.5 * mk[28] + 607.5 * mk[32] - 121.5 * mk[33]) + Gs[3] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[7] * (-121.5 * mk[9] - 121.5 * mk[15] + 607.5 * mk[18] - 121.5 * mk[19]) + Gs[8] * (-243.0 * mk[8] - 243.0 * mk[14] + 850.5 * mk[17] - 243.0 * mk[18]) + Gs[9] * (-121.5 * mk[7] - 121.5 * mk[13] + 243.0 * mk[16] - 121.5 * mk[17]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[298] = v_;
      out[374] = v_;
    }
    {
      const double M_ = -121.5 * m[47] - 121.5 * m[68] + 243.0 * m[73] - 121.5 * m[74];
      const double K_ = Gs[5] * (-121.5 * mk[18] - 121.5 * mk[28] + 607.5 * mk[32] - 121.5 * mk[33]) + Gs[6] * (-121.5 * mk[17] - 121.5 * mk[27] + 243.0 * mk[31] - 121.5 * mk[32]) + Gs[7] * (-121.5 * mk[15] - 121.5 * mk[25] + 607.5 * mk[28] - 121.5 * mk[29]) + Gs[8] * (-243.0 * mk[14] - 243.0 * mk[24] + 850.5 * mk[27] - 243.0 * mk[28]) + Gs[9] * (-121.5 * mk[13] - 121.5 * mk[23] + 243.0 * mk[26] - 121.5 * mk[27]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[299] = v_;
      out[394] = v_;
    }
    {
      const double M_ = 20.25 * m[32] + 40.5 * m[47] + 40.5 * m[52] - 81.0 * m[53] + 20.25 * m[68] + 40.5 * m[73] - 81.0 * m[74] + 20.25 * m[79] - 81.0 * m[80] + 81.0 * m[81];
      const double K_ = Gs[7] * (20.25 * mk[9] + 40.5 * mk[15] + 40.5 * mk[18] - 81.0 * mk[19] + 20.25 * mk[25] + 40.5 * mk[28] - 81.0 * mk[29] + 20.25 * mk[32] - 81.0 * mk[33] + 81.0 * mk[34]) + Gs[8] * (40.5 * mk[8] + 81.0 * mk[14] + 81.0 * mk[17] - 283.5 * mk[18] + 40.5 * mk[24] + 81.0 * mk[27] - 283.5 * mk[28] + 40.5 * mk[31] - 283.5 * mk[32] + 405.0 * mk[33]) + Gs[9] * (20.25 * mk[7] + 40.5 * mk[13] + 40.5 * mk[16] - 202.5 * mk[17] + 20.25 * mk[23] + 40.5 * mk[26] - 202.5 * mk[27] + 20.25 * mk[30] - 202.5 * mk[31] + 506.25 * mk[32]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[315] = v_;
    }
    {
      const double M_ = -121.5 * m[27] - 121.5 * m[42] - 121.5 * m[46] + 243.0 * m[47];
      const double K_ = Gs[2] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 243.0 * mk[28]) + Gs[3] * (-121.5 * mk[13] - 121.5 * mk[23] - 121.5 * mk[26] + 607.5 * mk[27]) + Gs[5] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 243.0 * mk[18]) + Gs[6] * (-121.5 * mk[7] - 121.5 * mk[13] - 121.5 * mk[16] + 607.5 * mk[17]) + Gs[7] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 243.0 * mk[15]) + Gs[8] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[316] = v_;
      out[335] = v_;
    }
    {
      const double M_ = -121.5 * m[28] - 121.5 * m[43] - 121.5 * m[47] + 243.0 * m[48];
      const double K_ = Gs[2] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[3] * (-121.5 * mk[14] - 121.5 * mk[24] - 121.5 * mk[27] + 607.5 * mk[28]) + Gs[5] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[6] * (-121.5 * mk[8] - 121.5 * mk[14] - 121.5 * mk[17] + 607.5 * mk[18]) + Gs[8] * (-121.5 * mk[6] - 121.5 * mk[12] - 121.5 * mk[14] + 243.0 * mk[15]) + Gs[9] * (-121.5 * mk[5] - 121.5 * mk[11] - 121.5 * mk[13] + 607.5 * mk[14]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[317] = v_;
      out[355] = v_;
    }
    {
      const double M_ = -121.5 * m[32] - 121.5 * m[47] - 121.5 * m[52] + 243.0 * m[53];
      const double K_ = Gs[2] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[3] * (-121.5 * mk[17] - 121.5 * mk[27] - 121.5 * mk[31] + 607.5 * mk[32]) + Gs[7] * (-121.5 * mk[9] - 121.5 * mk[15] - 121.5 * mk[18] + 243.0 * mk[19]) + Gs[8] * (-243.0 * mk[8] - 243.0 * mk[14] - 243.0 * mk[17] + 850.5 * mk[18]) + Gs[9] * (-121.5 * mk[7] - 121.5 * mk[13] - 121.5 * mk[16] + 607.5 * mk[17]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[318] = v_;
      out[375] = v_;
    }
    {
      const double M_ = -121.5 * m[47] - 121.5 * m[68] - 121.5 * m[73] + 243.0 * m[74];
      const double K_ = Gs[5] * (-121.5 * mk[18] - 121.5 * mk[28] - 121.5 * mk[32] + 243.0 * mk[33]) + Gs[6] * (-121.5 * mk[17] - 121.5 * mk[27] - 121.5 * mk[31] + 607.5 * mk[32]) + Gs[7] * (-121.5 * mk[15] - 121.5 * mk[25] - 121.5 * mk[28] + 243.0 * mk[29]) + Gs[8] * (-243.0 * mk[14] - 243.0 * mk[24] - 243.0 * mk[27] + 850.5 * mk[28]) + Gs[9] * (-121.5 * mk[13] - 121.5 * mk[23] - 121.5 * mk[26] + 607.5 * mk[27]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[319] = v_;
      out[395] = v_;
    }
    {
      const double M_ = 729.0 * m[23];
      const double K_ = Gs[0] * (729.0 * mk[23]) + Gs[1] * (1458.0 * mk[13]) + Gs[2] * (1458.0 * mk[11]) + Gs[4] * (729.0 * mk[7]) + Gs[5] * (1458.0 * mk[5]) + Gs[7] * (729.0 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[336] = v_;
    }
    {
      const double M_ = 729.0 * m[24];
      const double K_ = Gs[0] * (729.0 * mk[24]) + Gs[1] * (1458.0 * mk[14]) + Gs[2] * (729.0 * mk[12]) + Gs[3] * (729.0 * mk[11]) + Gs[4] * (729.0 * mk[8]) + Gs[5] * (729.0 * mk[6]) + Gs[6] * (729.0 * mk[5]) + Gs[8] * (729.0 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[337] = v_;
      out[356] = v_;
    }
    {
      const double M_ = 729.0 * m[27];
      const double K_ = Gs[0] * (729.0 * mk[27]) + Gs[1] * (729.0 * mk[17]) + Gs[2] * (1458.0 * mk[14]) + Gs[3] * (729.0 * mk[13]) + Gs[5] * (729.0 * mk[8]) + Gs[6] * (729.0 * mk[7]) + Gs[7] * (729.0 * mk[6]) + Gs[8] * (729.0 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[338] = v_;
      out[376] = v_;
    }
    {
      const double M_ = 729.0 * m[42];
      const double K_ = Gs[1] * (729.0 * mk[27]) + Gs[2] * (729.0 * mk[24]) + Gs[3] * (729.0 * mk[23]) + Gs[4] * (729.0 * mk[17]) + Gs[5] * (1458.0 * mk[14]) + Gs[6] * (729.0 * mk[13]) + Gs[7] * (729.0 * mk[12]) + Gs[8] * (729.0 * mk[11]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[339] = v_;
      out[396] = v_;
    }
    {
      const double M_ = 729.0 * m[25];
      const double K_ = Gs[0] * (729.0 * mk[25]) + Gs[1] * (1458.0 * mk[15]) + Gs[3] * (1458.0 * mk[12]) + Gs[4] * (729.0 * mk[9]) + Gs[6] * (1458.0 * mk[6]) + Gs[9] * (729.0 * mk[4]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[357] = v_;
    }
    {
      const double M_ = 729.0 * m[28];
      const double K_ = Gs[0] * (729.0 * mk[28]) + Gs[1] * (729.0 * mk[18]) + Gs[2] * (729.0 * mk[15]) + Gs[3] * (1458.0 * mk[14]) + Gs[5] * (729.0 * mk[9]) + Gs[6] * (729.0 * mk[8]) + Gs[8] * (729.0 * mk[6]) + Gs[9] * (729.0 * mk[5]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[358] = v_;
      out[377] = v_;
    }
    {
      const double M_ = 729.0 * m[43];
      const double K_ = Gs[1] * (729.0 * mk[28]) + Gs[2] * (729.0 * mk[25]) + Gs[3] * (729.0 * mk[24]) + Gs[4] * (729.0 * mk[18]) + Gs[5] * (729.0 * mk[15]) + Gs[6] * (1458.0 * mk[14]) + Gs[8] * (729.0 * mk[12]) + Gs[9] * (729.0 * mk[11]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[359] = v_;
      out[397] = v_;
    }
    {
      const double M_ = 729.0 * m[32];
      const double K_ = Gs[0] * (729.0 * mk[32]) + Gs[2] * (1458.0 * mk[18]) + Gs[3] * (1458.0 * mk[17]) + Gs[7] * (729.0 * mk[9]) + Gs[8] * (1458.0 * mk[8]) + Gs[9] * (729.0 * mk[7]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[378] = v_;
    }
    {
      const double M_ = 729.0 * m[47];
      const double K_ = Gs[1] * (729.0 * mk[32]) + Gs[2] * (729.0 * mk[28]) + Gs[3] * (729.0 * mk[27]) + Gs[5] * (729.0 * mk[18]) + Gs[6] * (729.0 * mk[17]) + Gs[7] * (729.0 * mk[15]) + Gs[8] * (1458.0 * mk[14]) + Gs[9] * (729.0 * mk[13]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[379] = v_;
      out[398] = v_;
    }
    {
      const double M_ = 729.0 * m[68];
      const double K_ = Gs[4] * (729.0 * mk[32]) + Gs[5] * (1458.0 * mk[28]) + Gs[6] * (1458.0 * mk[27]) + Gs[7] * (729.0 * mk[25]) + Gs[8] * (1458.0 * mk[24]) + Gs[9] * (729.0 * mk[23]);
      const T v_ = (T)(sm * M_ + sk * K_);
      out[399] = v_;
    }
  }
  // out[a] = s * sum_i w_i phi_a(x_i)  (source term of a linear form)
  template <typename T>
  XG_DEV static void vec(const double *m, double s, T *out) {
    out[0] = (T)(s * (m[0] + 0.5 * m[1] + 0.5 * m[2] + 0.5 * m[3] - 3.5 * m[4] - 7.0 * m[5] - 7.0 * m[6] - 3.5 * m[7] - 7.0 * m[8] - 3.5 * m[9] - 3.5 * m[10] - 10.5 * m[11] - 10.5 * m[12] - 10.5 * m[13] - 21.0 * m[14] - 10.5 * m[15] - 3.5 * m[16] - 10.5 * m[17] - 10.5 * m[18] - 3.5 * m[19] + 0.5 * m[20] + 2.0 * m[21] + 2.0 * m[22] + 3.0 * m[23] + 6.0 * m[24] + 3.0 * m[25] + 2.0 * m[26] + 6.0 * m[27] + 6.0 * m[28] + 2.0 * m[29] + 0.5 * m[30] + 2.0 * m[31] + 3.0 * m[32] + 2.0 * m[33] + 0.5 * m[34] + m[35] + 5.0 * m[36] + 5.0 * m[37] + 10.0 * m[38] + 20.0 * m[39] + 10.0 * m[40] + 10.0 * m[41] + 30.0 * m[42] + 30.0 * m[43] + 10.0 * m[44] + 5.0 * m[45] + 20.0 * m[46] + 30.0 * m[47] + 20.0 * m[48] + 5.0 * m[49] + m[50] + 5.0 * m[51] + 10.0 * m[52] + 10.0 * m[53] + 5.0 * m[54] + m[55]));
    out[1] = (T)(s * (m[1] + 0.5 * m[4] + 5.0 * m[5] + 5.0 * m[6] - 3.5 * m[10] + 2.0 * m[11] + 2.0 * m[12] + 10.0 * m[13] + 20.0 * m[14] + 10.0 * m[15] - 3.5 * m[20] - 10.5 * m[21] - 10.5 * m[22] + 3.0 * m[23] + 6.0 * m[24] + 3.0 * m[25] + 10.0 * m[26] + 30.0 * m[27] + 30.0 * m[28] + 10.0 * m[29] + 0.5 * m[35] - 7.0 * m[36] - 7.0 * m[37] - 10.5 * m[38] - 21.0 * m[39] - 10.5 * m[40] + 2.0 * m[41] + 6.0 * m[42] + 6.0 * m[43] + 2.0 * m[44] + 5.0 * m[45] + 20.0 * m[46] + 30.0 * m[47] + 20.0 * m[48] + 5.0 * m[49] + m[56] + 0.5 * m[57] + 0.5 * m[58] - 3.5 * m[59] - 7.0 * m[60] - 3.5 * m[61] - 3.5 * m[62] - 10.5 * m[63] - 10.5 * m[64] - 3.5 * m[65] + 0.5 * m[66] + 2.0 * m[67] + 3.0 * m[68] + 2.0 * m[69] + 0.5 * m[70] + m[71] + 5.0 * m[72] + 10.0 * m[73] + 10.0 * m[74] + 5.0 * m[75] + m[76]));
    out[2] = (T)(s * (m[2] + 5.0 * m[5] + 0.5 * m[7] + 5.0 * m[8] + 10.0 * m[11] + 2.0 * m[13] + 20.0 * m[14] - 3.5 * m[16] + 2.0 * m[17] + 10.0 * m[18] + 10.0 * m[21] + 3.0 * m[23] + 30.0 * m[24] - 10.5 * m[26] + 6.0 * m[27] + 30.0 * m[28] - 3.5 * m[30] - 10.5 * m[31] + 3.0 * m[32] + 10.0 * m[33] + 5.0 * m[36] + 2.0 * m[38] + 20.0 * m[39] - 10.5 * m[41] + 6.0 * m[42] + 30.0 * m[43] - 7.0 * m[45] - 21.0 * m[46] + 6.0 * m[47] + 20.0 * m[48] + 0.5 * m[50] - 7.0 * m[51] - 10.5 * m[52] + 2.0 * m[53] + 5.0 * m[54] + m[57] + 0.5 * m[59] + 5.0 * m[60] - 3.5 * m[62] + 2.0 * m[63] + 10.0 * m[64] - 3.5 * m[66] - 10.5 * m[67] + 3.0 * m[68] + 10.0 * m[69] + 0.5 * m[71] - 7.0 * m[72] - 10.5 * m[73] + 2.0 * m[74] + 5.0 * m[75] + m[77] + 0.5 * m[78] - 3.5 * m[79] - 3.5 * m[80] + 0.5 * m[81] + m[82]));
    out[3] = (T)(s * (m[3] + 5.0 * m[6] + 5.0 * m[8] + 0.5 * m[9] + 10.0 * m[12] + 20.0 * m[14] + 2.0 * m[15] + 10.0 * m[17] + 2.0 * m[18] - 3.5 * m[19] + 10.0 * m[22] + 30.0 * m[24] + 3.0 * m[25] + 30.0 * m[27] + 6.0 * m[28] - 10.5 * m[29] + 10.0 * m[31] + 3.0 * m[32] - 10.5 * m[33] - 3.5 * m[34] + 5.0 * m[37] + 20.0 * m[39] + 2.0 * m[40] + 30.0 * m[42] + 6.0 * m[43] - 10.5 * m[44] + 20.0 * m[46] + 6.0 * m[47] - 21.0 * m[48] - 7.0 * m[49] + 5.0 * m[51] + 2.0 * m[52] - 10.5 * m[53] - 7.0 * m[54] + 0.5 * m[55] + m[58] + 5.0 * m[60] + 0.5 * m[61] + 10.0 * m[63] + 2.0 * m[64] - 3.5 * m[65] + 10.0 * m[67] + 3.0 * m[68] - 10.5 * m[69] - 3.5 * m[70] + 5.0 * m[72] + 2.0 * m[73] - 10.5 * m[74] - 7.0 * m[75] + 0.5 * m[76] + m[78] + 0.5 * m[79] - 3.5 * m[80] - 3.5 * m[81] + 0.5 * m[82] + m[83]));
    out[4] = (T)(s * (9.0 * m[1] + 22.5 * m[4] + 22.5 * m[5] + 22.5 * m[6] + 13.5 * m[10] + 27.0 * m[11] + 27.0 * m[12] + 13.5 * m[13] + 27.0 * m[14] + 13.5 * m[15] - 4.5 * m[20] - 13.5 * m[21] - 13.5 * m[22] - 13.5 * m[23] - 27.0 * m[24] - 13.5 * m[25] - 4.5 * m[26] - 13.5 * m[27] - 13.5 * m[28] - 4.5 * m[29] - 4.5 * m[35] - 18.0 * m[36] - 18.0 * m[37] - 27.0 * m[38] - 54.0 * m[39] - 27.0 * m[40] - 18.0 * m[41] - 54.0 * m[42] - 54.0 * m[43] - 18.0 * m[44] - 4.5 * m[45] - 18.0 * m[46] - 27.0 * m[47] - 18.0 * m[48] - 4.5 * m[49]));
    out[5] = (T)(s * (-4.5 * m[1] - 4.5 * m[4] - 18.0 * m[5] - 18.0 * m[6] + 13.5 * m[10] - 13.5 * m[11] - 13.5 * m[12] - 27.0 * m[13] - 54.0 * m[14] - 27.0 * m[15] + 22.5 * m[20] + 27.0 * m[21] + 27.0 * m[22] - 13.5 * m[23] - 27.0 * m[24] - 13.5 * m[25] - 18.0 * m[26] - 54.0 * m[27] - 54.0 * m[28] - 18.0 * m[29] + 9.0 * m[35] + 22.5 * m[36] + 22.5 * m[37] + 13.5 * m[38] + 27.0 * m[39] + 13.5 * m[40] - 4.5 * m[41] - 13.5 * m[42] - 13.5 * m[43] - 4.5 * m[44] - 4.5 * m[45] - 18.0 * m[46] - 27.0 * m[47] - 18.0 * m[48] - 4.5 * m[49]));
    out[6] = (T)(s * (9.0 * m[2] + 22.5 * m[5] + 22.5 * m[7] + 22.5 * m[8] + 13.5 * m[11] + 27.0 * m[13] + 27.0 * m[14] + 13.5 * m[16] + 27.0 * m[17] + 13.5 * m[18] - 4.5 * m[21] - 13.5 * m[23] - 13.5 * m[24] - 13.5 * m[26] - 27.0 * m[27] - 13.5 * m[28] - 4.5 * m[30] - 13.5 * m[31] - 13.5 * m[32] - 4.5 * m[33] - 4.5 * m[36] - 18.0 * m[38] - 18.0 * m[39] - 27.0 * m[41] - 54.0 * m[42] - 27.0 * m[43] - 18.0 * m[45] - 54.0 * m[46] - 54.0 * m[47] - 18.0 * m[48] - 4.5 * m[50] - 18.0 * m[51] - 27.0 * m[52] - 18.0 * m[53] - 4.5 * m[54]));
    out[7] = (T)(s * (-4.5 * m[2] - 18.0 * m[5] - 4.5 * m[7] - 18.0 * m[8] - 27.0 * m[11] - 13.5 * m[13] - 54.0 * m[14] + 13.5 * m[16] - 13.5 * m[17] - 27.0 * m[18] - 18.0 * m[21] - 13.5 * m[23] - 54.0 * m[24] + 27.0 * m[26] - 27.0 * m[27] - 54.0 * m[28] + 22.5 * m[30] + 27.0 * m[31] - 13.5 * m[32] - 18.0 * m[33] - 4.5 * m[36] - 4.5 * m[38] - 18.0 * m[39] + 13.5 * m[41] - 13.5 * m[42] - 27.0 * m[43] + 22.5 * m[45] + 27.0 * m[46] - 13.5 * m[47] - 18.0 * m[48] + 9.0 * m[50] + 22.5 * m[51] + 13.5 * m[52] - 4.5 * m[53] - 4.5 * m[54]));
    out[8] = (T)(s * (9.0 * m[3] + 22.5 * m[6] + 22.5 * m[8] + 22.5 * m[9] + 13.5 * m[12] + 27.0 * m[14] + 27.0 * m[15] + 13.5 * m[17] + 27.0 * m[18] + 13.5 * m[19] - 4.5 * m[22] - 13.5 * m[24] - 13.5 * m[25] - 13.5 * m[27] - 27.0 * m[28] - 13.5 * m[29] - 4.5 * m[31] - 13.5 * m[32] - 13.5 * m[33] - 4.5 * m[34] - 4.5 * m[37] - 18.0 * m[39] - 18.0 * m[40] - 27.0 * m[42] - 54.0 * m[43] - 27.0 * m[44] - 18.0 * m[46] - 54.0 * m[47] - 54.0 * m[48] - 18.0 * m[49] - 4.5 * m[51] - 18.0 * m[52] - 27.0 * m[53] - 18.0 * m[54] - 4.5 * m[55]));
    out[9] = (T)(s * (-4.5 * m[3] - 18.0 * m[6] - 18.0 * m[8] - 4.5 * m[9] - 27.0 * m[12] - 54.0 * m[14] - 13.5 * m[15] - 27.0 * m[17] - 13.5 * m[18] + 13.5 * m[19] - 18.0 * m[22] - 54.0 * m[24] - 13.5 * m[25] - 54.0 * m[27] - 27.0 * m[28] + 27.0 * m[29] - 18.0 * m[31] - 13.5 * m[32] + 27.0 * m[33] + 22.5 * m[34] - 4.5 * m[37] - 18.0 * m[39] - 4.5 * m[40] - 27.0 * m[42] - 13.5 * m[43] + 13.5 * m[44] - 18.0 * m[46] - 13.5 * m[47] + 27.0 * m[48] + 22.5 * m[49] - 4.5 * m[51] - 4.5 * m[52] + 13.5 * m[53] + 22.5 * m[54] + 9.0 * m[55]));
    out[10] = (T)(s * (-4.5 * m[5] - 4.5 * m[11] - 18.0 * m[13] - 18.0 * m[14] + 13.5 * m[21] - 13.5 * m[23] - 13.5 * m[24] - 27.0 * m[26] - 54.0 * m[27] - 27.0 * m[28] + 22.5 * m[36] + 27.0 * m[38] + 27.0 * m[39] - 13.5 * m[41] - 27.0 * m[42] - 13.5 * m[43] - 18.0 * m[45] - 54.0 * m[46] - 54.0 * m[47] - 18.0 * m[48] + 9.0 * m[57] + 22.5 * m[59] + 22.5 * m[60] + 13.5 * m[62] + 27.0 * m[63] + 13.5 * m[64] - 4.5 * m[66] - 13.5 * m[67] - 13.5 * m[68] - 4.5 * m[69] - 4.5 * m[71] - 18.0 * m[72] - 27.0 * m[73] - 18.0 * m[74] - 4.5 * m[75]));
    out[11] = (T)(s * (-4.5 * m[5] - 18.0 * m[11] - 4.5 * m[13] - 18.0 * m[14] - 27.0 * m[21] - 13.5 * m[23] - 54.0 * m[24] + 13.5 * m[26] - 13.5 * m[27] - 27.0 * m[28] - 18.0 * m[36] - 13.5 * m[38] - 54.0 * m[39] + 27.0 * m[41] - 27.0 * m[42] - 54.0 * m[43] + 22.5 * m[45] + 27.0 * m[46] - 13.5 * m[47] - 18.0 * m[48] - 4.5 * m[57] - 4.5 * m[59] - 18.0 * m[60] + 13.5 * m[62] - 13.5 * m[63] - 27.0 * m[64] + 22.5 * m[66] + 27.0 * m[67] - 13.5 * m[68] - 18.0 * m[69] + 9.0 * m[71] + 22.5 * m[72] + 13.5 * m[73] - 4.5 * m[74] - 4.5 * m[75]));
    out[12] = (T)(s * (-4.5 * m[6] - 4.5 * m[12] - 18.0 * m[14] - 18.0 * m[15] + 13.5 * m[22] - 13.5 * m[24] - 13.5 * m[25] - 27.0 * m[27] - 54.0 * m[28] - 27.0 * m[29] + 22.5 * m[37] + 27.0 * m[39] + 27.0 * m[40] - 13.5 * m[42] - 27.0 * m[43] - 13.5 * m[44] - 18.0 * m[46] - 54.0 * m[47] - 54.0 * m[48] - 18.0 * m[49] + 9.0 * m[58] + 22.5 * m[60] + 22.5 * m[61] + 13.5 * m[63] + 27.0 * m[64] + 13.5 * m[65] - 4.5 * m[67] - 13.5 * m[68] - 13.5 * m[69] - 4.5 * m[70] - 4.5 * m[72] - 18.0 * m[73] - 27.0 * m[74] - 18.0 * m[75] - 4.5 * m[76]));
    out[13] = (T)(s * (-4.5 * m[6] - 18.0 * m[12] - 18.0 * m[14] - 4.5 * m[15] - 27.0 * m[22] - 54.0 * m[24] - 13.5 * m[25] - 27.0 * m[27] - 13.5 * m[28] + 13.5 * m[29] - 18.0 * m[37] - 54.0 * m[39] - 13.5 * m[40] - 54.0 * m[42] - 27.0 * m[43] + 27.0 * m[44] - 18.0 * m[46] - 13.5 * m[47] + 27.0 * m[48] + 22.5 * m[49] - 4.5 * m[58] - 18.0 * m[60] - 4.5 * m[61] - 27.0 * m[63] - 13.5 * m[64] + 13.5 * m[65] - 18.0 * m[67] - 13.5 * m[68] + 27.0 * m[69] + 22.5 * m[70] - 4.5 * m[72] - 4.5 * m[73] + 13.5 * m[74] + 22.5 * m[75] + 9.0 * m[76]));
    out[14] = (T)(s * (-4.5 * m[8] - 18.0 * m[14] - 4.5 * m[17] - 18.0 * m[18] - 27.0 * m[24] - 13.5 * m[27] - 54.0 * m[28] + 13.5 * m[31] - 13.5 * m[32] - 27.0 * m[33] - 18.0 * m[39] - 13.5 * m[42] - 54.0 * m[43] + 27.0 * m[46] - 27.0 * m[47] - 54.0 * m[48] + 22.5 * m[51] + 27.0 * m[52] - 13.5 * m[53] - 18.0 * m[54] - 4.5 * m[60] - 4.5 * m[63] - 18.0 * m[64] + 13.5 * m[67] - 13.5 * m[68] - 27.0 * m[69] + 22.5 * m[72] + 27.0 * m[73] - 13.5 * m[74] - 18.0 * m[75] + 9.0 * m[78] + 22.5 * m[79] + 13.5 * m[80] - 4.5 * m[81] - 4.5 * m[82]));
    out[15] = (T)(s * (-4.5 * m[8] - 18.0 * m[14] - 18.0 * m[17] - 4.5 * m[18] - 27.0 * m[24] - 54.0 * m[27] - 13.5 * m[28] - 27.0 * m[31] - 13.5 * m[32] + 13.5 * m[33] - 18.0 * m[39] - 54.0 * m[42] - 13.5 * m[43] - 54.0 * m[46] - 27.0 * m[47] + 27.0 * m[48] - 18.0 * m[51] - 13.5 * m[52] + 27.0 * m[53] + 22.5 * m[54] - 4.5 * m[60] - 18.0 * m[63] - 4.5 * m[64] - 27.0 * m[67] - 13.5 * m[68] + 13.5 * m[69] - 18.0 * m[72] - 13.5 * m[73] + 27.0 * m[74] + 22.5 * m[75] - 4.5 * m[78] - 4.5 * m[79] + 13.5 * m[80] + 22.5 * m[81] + 9.0 * m[82]));
    out[16] = (T)(s * (27.0 * m[5] + 81.0 * m[11] + 81.0 * m[13] + 81.0 * m[14] + 81.0 * m[21] + 162.0 * m[23] + 162.0 * m[24] + 81.0 * m[26] + 162.0 * m[27] + 81.0 * m[28] + 27.0 * m[36] + 81.0 * m[38] + 81.0 * m[39] + 81.0 * m[41] + 162.0 * m[42] + 81.0 * m[43] + 27.0 * m[45] + 81.0 * m[46] + 81.0 * m[47] + 27.0 * m[48]));
    out[17] = (T)(s * (27.0 * m[6] + 81.0 * m[12] + 81.0 * m[14] + 81.0 * m[15] + 81.0 * m[22] + 162.0 * m[24] + 162.0 * m[25] + 81.0 * m[27] + 162.0 * m[28] + 81.0 * m[29] + 27.0 * m[37] + 81.0 * m[39] + 81.0 * m[40] + 81.0 * m[42] + 162.0 * m[43] + 81.0 * m[44] + 27.0 * m[46] + 81.0 * m[47] + 81.0 * m[48] + 27.0 * m[49]));
    out[18] = (T)(s * (27.0 * m[8] + 81.0 * m[14] + 81.0 * m[17] + 81.0 * m[18] + 81.0 * m[24] + 162.0 * m[27] + 162.0 * m[28] + 81.0 * m[31] + 162.0 * m[32] + 81.0 * m[33] + 27.0 * m[39] + 81.0 * m[42] + 81.0 * m[43] + 81.0 * m[46] + 162.0 * m[47] + 81.0 * m[48] + 27.0 * m[51] + 81.0 * m[52] + 81.0 * m[53] + 27.0 * m[54]));
    out[19] = (T)(s * (27.0 * m[14] + 81.0 * m[24] + 81.0 * m[27] + 81.0 * m[28] + 81.0 * m[39] + 162.0 * m[42] + 162.0 * m[43] + 81.0 * m[46] + 162.0 * m[47] + 81.0 * m[48] + 27.0 * m[60] + 81.0 * m[63] + 81.0 * m[64] + 81.0 * m[67] + 162.0 * m[68] + 81.0 * m[69] + 27.0 * m[72] + 81.0 * m[73] + 81.0 * m[74] + 27.0 * m[75]));
  }
};  // 9054 coefficient terms
// centred affine moments (y = lam - 1/4) -> homogeneous degree-2 moments, D = 3:
// m[alpha] = sum_slot xg_aff31[slot][alpha % 64][alpha / 64] n[slot]
#ifndef XG_AFF_STORAGE
#define XG_AFF_STORAGE static __device__
#endif
XG_AFF_STORAGE const float xg_aff31[10][64][2] __attribute__((aligned(16))) = {
    {{1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.5, 0}, {0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0.25, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
};
// beta! / (|beta| + k)! of Moments<3,1>::aser_*, k = 3 and 2
XG_AFF_STORAGE const double xg_aser31[10][2] = {
    {0.016666666666666666, 0.08333333333333333},
    {0.008333333333333333, 0.041666666666666664},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.041666666666666664, 0.16666666666666666},
    {0.16666666666666666, 0.5},
};
// centred affine moments (y = lam - 1/4) -> homogeneous degree-4 moments, D = 3:
// m[alpha] = sum_slot xg_aff32[slot][alpha % 64][alpha / 64] n[slot]
#ifndef XG_AFF_STORAGE
#define XG_AFF_STORAGE static __device__
#endif
XG_AFF_STORAGE const float xg_aff32[35][64][2] __attribute__((aligned(16))) = {
    {{1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{1.0, 0}, {0.25, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0.75, 0}, {0, 0}, {-0.75, 0}, {0.5, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0.75, 0}, {-0.75, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0.25, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.375, 0}, {0.1875, 0}, {0.1875, 0}, {0, 0}, {0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.125, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.1875, 0}, {0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0.75, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {0, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0.1875, 0}, {0, 0}, {-0.1875, 0}, {0.25, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {-0.125, 0}, {-0.125, 0}, {0.1875, 0}, {0.125, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0, 0}, {-0.125, 0}, {-0.125, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0.125, 0}, {0.375, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0.75, 0}, {-0.5, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {-0.75, 0}, {0.5, 0}, {0.75, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {0, 0}, {0.125, 0}, {-0.125, 0}, {0.25, 0}, {-0.0625, 0}, {-0.125, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0, 0}, {-0.125, 0}, {0, 0}, {0.375, 0}, {0, 0}, {-0.1875, 0}, {-0.125, 0}, {0.1875, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.0625, 0}, {0.046875, 0}, {0.046875, 0}, {0.03125, 0}, {0.03125, 0}, {0.03125, 0}, {0.015625, 0}, {0.03125, 0}, {0.015625, 0}, {0, 0}, {0.015625, 0}, {0.015625, 0}, {0, 0}, {0.015625, 0}, {0, 0}, {-0.015625, 0}, {0.015625, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {-0.046875, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {-0.046875, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {0, 0}, {0.75, 0}, {-0.75, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0.25, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.1875, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.1875, 0}, {0.375, 0}, {0.1875, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.125, 0}, {0, 0}, {-0.0625, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.1875, 0}, {0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0.75, 0}, {-0.5, 0}, {0.25, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {0.5, 0}, {0.75, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0, 0}, {0.125, 0}, {-0.125, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {-0.125, 0}, {0, 0}, {0.375, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {0.25, 0}, {-0.0625, 0}, {-0.125, 0}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0}, {0.1875, 0}, {0, 0}, {-0.1875, 0}, {-0.125, 0}, {0.1875, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0.015625, 0}, {0, 0}, {-0.015625, 0}, {0.03125, 0}, {0.015625, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {0.046875, 0}, {0.03125, 0}, {0.015625, 0}, {0.015625, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {-0.046875, 0}, {0.0625, 0}, {0.046875, 0}, {0.03125, 0}, {0.03125, 0}, {0.015625, 0}, {0, 0}, {0.015625, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {0, 0}, {-0.015625, 0}, {-0.03125, 0}, {-0.046875, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {1.0, 0}, {-0.5, 0}, {0, 0}, {0.5, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0}, {0.1875, 0}, {0.375, 0}, {0, 0}, {-0.125, 0}, {0, 0}, {0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {0.046875, 0}, {0.015625, 0}, {-0.015625, 0}, {-0.046875, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {0.046875, 0}, {0.015625, 0}, {-0.015625, 0}, {-0.046875, 0}, {0.0625, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.00390625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
};
// beta! / (|beta| + k)! of Moments<3,2>::aser_*, k = 3 and 2
XG_AFF_STORAGE const double xg_aser32[35][2] = {
    {0.004761904761904762, 0.03333333333333333},
    {0.0011904761904761906, 0.008333333333333333},
    {0.0011904761904761906, 0.008333333333333333},
    {0.008333333333333333, 0.05},
    {0.0007936507936507937, 0.005555555555555556},
    {0.0003968253968253968, 0.002777777777777778},
    {0.002777777777777778, 0.016666666666666666},
    {0.0007936507936507937, 0.005555555555555556},
    {0.002777777777777778, 0.016666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.0011904761904761906, 0.008333333333333333},
    {0.0003968253968253968, 0.002777777777777778},
    {0.002777777777777778, 0.016666666666666666},
    {0.0003968253968253968, 0.002777777777777778},
    {0.001388888888888889, 0.008333333333333333},
    {0.008333333333333333, 0.041666666666666664},
    {0.0011904761904761906, 0.008333333333333333},
    {0.002777777777777778, 0.016666666666666666},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.004761904761904762, 0.03333333333333333},
    {0.0011904761904761906, 0.008333333333333333},
    {0.008333333333333333, 0.05},
    {0.0007936507936507937, 0.005555555555555556},
    {0.002777777777777778, 0.016666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.0011904761904761906, 0.008333333333333333},
    {0.002777777777777778, 0.016666666666666666},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.004761904761904762, 0.03333333333333333},
    {0.008333333333333333, 0.05},
    {0.016666666666666666, 0.08333333333333333},
    {0.041666666666666664, 0.16666666666666666},
    {0.16666666666666666, 0.5},
};
// centred affine moments (y = lam - 1/4) -> homogeneous degree-6 moments, D = 3:
// m[alpha] = sum_slot xg_aff33[slot][alpha % 64][alpha / 64] n[slot]
#ifndef XG_AFF_STORAGE
#define XG_AFF_STORAGE static __device__
#endif
XG_AFF_STORAGE const float xg_aff33[84][64][2] __attribute__((aligned(16))) = {
    {{1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, -1.0}, {-3.0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{1.5, 0}, {0.25, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, -0.25}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0.25, -0.25}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 1.0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {-1.0, -5.0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 1.0}, {0, -5.0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {2.0, -5.0}, {-6.0, 30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {-20.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {1.25, 0}, {0, 0}, {-1.25, 0}, {0.5, 0}, {0.25, 0}, {-1.0, 0.5}, {0, 0}, {-0.25, 0}, {1.5, 0}, {0, 0}, {0, 0.25}, {-0.5, 0}, {0, 0}, {-0.25, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0.5, -1.25}, {-0.75, -7.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {3.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 1.0}, {2.0, -5.0}, {-3.0, 15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {1.25, 0}, {-1.25, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.5, 0}, {-1.0, 0}, {1.5, 0}, {0, 0}, {0, 0.25}, {0, -1.25}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {-0.5, 0.5}, {0.75, 0}, {-0.75, -7.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {0.25, 0}, {3.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.9375, 0}, {0.3125, 0}, {0.3125, 0}, {-0.3125, 0}, {0.0625, 0}, {0.0625, 0}, {-0.1875, 0.0625}, {0.0625, 0}, {-0.1875, 0}, {-0.0625, 0}, {0, 0}, {0, 0.0625}, {-0.0625, 0.3125}, {0, 0}, {-0.0625, 0}, {0.0625, 0}, {0, 0}, {-0.0625, 0.0625}, {0.0625, 0.3125}, {0.1875, 0.9375}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {-0.1875, 0}, {-0.3125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, -1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, -10.0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 20.0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 4.0}, {-1.0, -20.0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {1.0, -10.0}, {-3.0, 60.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {6.0, 0}, {-30.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, -0.75}, {0, 0}, {0, 0}, {1.0, 0}, {0, -0.25}, {-1.0, 1.0}, {0, 0}, {0, 0}, {1.0, 0}, {0.75, 0}, {0.25, 1.0}, {-1.0, 2.5}, {0, 0}, {-0.25, 0}, {1.25, 0}, {0, 0}, {0, 0}, {0.25, -2.5}, {-1.5, -15.0}, {0, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.5, 0}, {5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 4.0}, {0, -10.0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 4.0}, {2.0, -20.0}, {-3.0, 60.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {-30.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, -0.5}, {-1.0, 2.0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, -0.5}, {0.5, 1.0}, {-0.5, 0}, {0.5, 0}, {-1.0, 0}, {1.5, 0}, {0, 0}, {-0.5, 2.0}, {1.5, 0}, {-3.0, -30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.5, 0}, {1.0, 0}, {10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0.625, -0.1875}, {0, 0}, {-0.625, 0}, {0.5, 0}, {0.25, -0.125}, {-0.375, -0.25}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0.1875, -0.0625}, {0.125, 0}, {-0.3125, 0.625}, {0.0625, 0}, {-0.1875, 0}, {0.125, 0}, {0, 0}, {-0.0625, 0.25}, {0.25, 1.25}, {0.375, 3.75}, {0, 0}, {0, 0}, {-0.1875, 0}, {0, 0}, {-0.125, 0}, {0.125, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0.125, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0.125, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {-0.5, 0}, {-0.625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, -1.0}, {-1.0, 4.0}, {1.0, -10.0}, {-1.0, 20.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, -0.25}, {0, 1.0}, {0, -2.5}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0.75, -0.75}, {-1.0, 1.0}, {1.25, 2.5}, {-1.5, -15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {-0.75, 0}, {1.0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {1.5, 0}, {0, 0}, {0, 0}, {0.75, 0}, {-1.0, 0}, {-0.5, 0}, {5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0.625, 0}, {-0.625, 0}, {0, 0}, {0.25, -0.0625}, {-0.25, 0.25}, {0.5, 0}, {-0.375, 0}, {0.25, 0}, {0, -0.125}, {0.0625, 0}, {-0.0625, 1.25}, {0.125, 0}, {-0.1875, 0}, {0.25, 0}, {0.1875, -0.1875}, {-0.3125, -0.25}, {0.125, 0.625}, {0.375, 3.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0, 0}, {-0.125, 0}, {0.125, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0.125, 0}, {0.125, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0.125, 0}, {-0.0625, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {0.0625, 0}, {-0.375, 0}, {-0.625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.3125, 0}, {0.15625, -0.015625}, {0.15625, 0}, {0, 0}, {0.0625, 0}, {0.0625, -0.015625}, {-0.03125, -0.0625}, {0.0625, 0}, {-0.03125, 0}, {-0.0625, 0}, {0.015625, -0.015625}, {0.015625, -0.0625}, {-0.03125, -0.15625}, {0.015625, 0}, {-0.03125, 0}, {-0.03125, 0}, {0.015625, -0.015625}, {-0.03125, -0.0625}, {-0.03125, -0.15625}, {0, -0.3125}, {0, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {0.03125, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {0.03125, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0.03125, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0.03125, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -10.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 15.0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}},
    {{0, 1.0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 6.0}, {0, -30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -10.0}, {0, 60.0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {4.0, 0}, {-20.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.25}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0}, {0, -0.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.75, 0}, {0, 1.5}, {-0.75, 5.0}, {0, 0}, {0, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0, -2.5}, {-0.75, -15.0}, {1.0, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {-0.25, 0}, {1.25, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {2.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, -30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 6.0}, {0, -30.0}, {0, 90.0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {12.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-3.0, 0}, {12.0, 0}, {-30.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.75}, {0, -2.25}, {0, 0}, {0, 0}, {0, 0.5}, {0, -1.5}, {0, 3.0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.5}, {0.75, 1.5}, {-0.75, 7.5}, {0, 0}, {-0.75, 0}, {1.5, 0}, {0, 0}, {0, 3.0}, {0.75, 0}, {-2.25, -45.0}, {0, 0}, {0.75, 0}, {-0.75, 0}, {0.5, 0}, {-1.0, 0}, {1.5, 0}, {0, 0}, {-0.5, 0}, {1.25, 0}, {-2.25, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.5, 0}, {3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}, {1.5, 0}, {0, 0}, {-0.5, 0}, {1.25, 0}, {-2.25, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.5, 0}, {1.5, 0}, {7.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.1875}, {0, 0}, {0, 0}, {0, 0}, {0.375, 0.0625}, {0, -0.1875}, {-0.375, -0.75}, {0, 0}, {0, 0}, {0.375, 0}, {0.5625, -0.1875}, {0.1875, -0.375}, {-0.375, 0}, {0, 0}, {-0.1875, 0}, {0.1875, 0}, {0, 0}, {0, 0.375}, {0.1875, 1.875}, {0, 5.625}, {0.375, 0}, {0.1875, 0}, {-0.375, 0}, {0.0625, 0}, {-0.1875, 0}, {0.1875, 0}, {0, 0}, {-0.0625, 0}, {0.1875, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.1875, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {-0.375, 0}, {0, 0}, {-0.1875, 0}, {0.1875, 0}, {0, 0}, {-0.0625, 0}, {0.1875, 0}, {0.1875, 0}, {0, 0}, {0, 0}, {0.125, 0}, {0, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.375, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, -10.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, -30.0}, {0, 60.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {-6.0, 0}, {12.0, 0}, {-20.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.5}, {0, -1.5}, {0, 3.0}, {0, 0}, {0, 0}, {0, 0.75}, {0, -1.5}, {0, 1.5}, {0, 0}, {0.75, 0}, {-0.75, 0}, {0.75, 0}, {0, -2.25}, {-0.75, 3.0}, {1.5, 7.5}, {-2.25, -45.0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0.75, 0}, {-1.0, 0}, {1.25, 0}, {-1.5, 0}, {0, 0}, {-0.75, 0}, {1.5, 0}, {-2.25, 0}, {3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {-0.75, 0}, {1.25, 0}, {-1.5, 0}, {1.5, 0}, {0, 0}, {0, 0}, {1.5, 0}, {-2.25, 0}, {0, 0}, {7.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.1875}, {0, -0.5625}, {0, 0}, {0, 0}, {0, 0.25}, {0.375, -0.1875}, {-0.375, -0.75}, {0, 0}, {-0.375, 0}, {0.75, 0.1875}, {0, -0.1875}, {0.375, -0.375}, {-0.375, 1.875}, {0.375, 0}, {-0.375, 0}, {0.375, 0}, {0, -0.5625}, {-0.375, -0.75}, {0.375, 1.875}, {0, 11.25}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {0.25, 0}, {-0.3125, 0}, {0.375, 0}, {0.1875, 0}, {-0.3125, 0}, {0.25, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0.375, 0}, {0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0.375, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0.25, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0.375, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.046875}, {0.15625, 0.09375}, {0, 0}, {-0.15625, 0}, {0.1875, 0.03125}, {0.09375, 0.046875}, {-0.0625, 0}, {0, 0}, {-0.09375, 0}, {-0.0625, 0.015625}, {0.140625, 0}, {0.09375, -0.09375}, {-0.046875, -0.3125}, {0.046875, 0}, {-0.046875, 0}, {-0.03125, 0}, {0, -0.046875}, {-0.046875, -0.1875}, {0, -0.46875}, {0.09375, -0.9375}, {0.0625, 0}, {0.046875, 0}, {-0.0625, 0}, {0.03125, 0}, {-0.046875, 0}, {-0.03125, 0}, {0.015625, 0}, {-0.03125, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {-0.015625, 0}, {0.03125, 0}, {0.09375, 0}, {0.125, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {-0.046875, 0}, {-0.015625, 0}, {0, 0}, {-0.03125, 0}, {0, 0}, {0.046875, 0}, {0, 0}, {-0.015625, 0}, {0.015625, 0}, {0.046875, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0.03125, 0}, {0.046875, 0}, {0, 0}, {-0.15625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, -10.0}, {0, 15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.25}, {0, -0.75}, {0, 1.5}, {0, -2.5}, {0, 0}, {0, 0}, {0, 1.0}, {0.75, -1.5}, {-0.75, 0}, {0.75, 5.0}, {-0.75, -15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {1.25, 0}, {-0.75, 0}, {-0.5, 0}, {2.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.0625}, {0, -0.1875}, {0, 0.375}, {0.375, 0}, {-0.375, 0}, {0.375, 0.1875}, {0, -0.1875}, {0, -0.375}, {0, 1.875}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0.375}, {0.5625, 0}, {-0.375, -0.75}, {0.1875, 0}, {0, 5.625}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0}, {-0.1875, 0}, {0.375, 0}, {-0.375, 0}, {0.1875, 0}, {0.1875, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {-0.1875, 0}, {0, 0}, {-0.1875, 0}, {0.1875, 0}, {0, 0}, {-0.375, 0}, {0, 0}, {-0.375, 0}, {0.1875, 0}, {0.1875, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.015625}, {0, -0.046875}, {0.15625, 0}, {-0.15625, 0}, {0, 0.03125}, {0.09375, 0}, {-0.09375, -0.1875}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0.046875}, {0, 0.046875}, {0.046875, -0.09375}, {-0.046875, -0.46875}, {0.09375, 0}, {-0.046875, 0}, {0, 0.0625}, {0.140625, 0.09375}, {-0.046875, 0}, {-0.03125, -0.3125}, {0.09375, -0.9375}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.03125, 0}, {-0.03125, 0}, {0.03125, 0}, {0.046875, 0}, {-0.046875, 0}, {0, 0}, {0.09375, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.03125, 0}, {0.0625, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {0.015625, 0}, {0.046875, 0}, {0, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {-0.015625, 0}, {0.046875, 0}, {0.03125, 0}, {-0.15625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0.05859375, 0.00390625}, {0.0390625, 0.01171875}, {0.0390625, 0}, {0.01953125, 0}, {0.0234375, 0.00390625}, {0.0234375, 0.01171875}, {0.0078125, 0.0234375}, {0.0234375, 0}, {0.0078125, 0}, {-0.00390625, 0.00390625}, {0.01171875, 0.01171875}, {0.01171875, 0.0234375}, {0, 0.0390625}, {0.01171875, 0}, {0, 0}, {-0.0078125, 0.00390625}, {0.01171875, 0.01171875}, {0, 0.0234375}, {-0.0078125, 0.0390625}, {-0.01171875, 0.05859375}, {0.00390625, 0}, {0.00390625, 0}, {-0.00390625, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {-0.0078125, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {-0.0078125, 0}, {-0.00390625, 0}, {0, 0}, {0, 0}, {-0.00390625, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {0.0078125, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {0.0078125, 0}, {0.01953125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -5.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {2.0, 0}, {0, 0}, {0, 0}},
    {{0, 2.0}, {0, -6.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 4.0}, {0, -20.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -5.0}, {0, 30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}},
    {{0, 0.5}, {0, -0.75}, {0, 0}, {0, 0}, {0, 0}, {0, -0.75}, {0, -1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, 3.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.25}, {0, -7.5}, {0.5, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {1.25, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {-0.25, 0}, {0.75, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.25, 0}, {0, 0}, {-0.25, 0}, {1.5, 0}, {0, 0}, {0, 0}},
    {{0, 2.0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 2.0}, {0, -6.0}, {0, 12.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, -30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 4.0}, {0, -20.0}, {0, 60.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {4.0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}},
    {{0, 1.5}, {0, -3.0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.5}, {0, 1.0}, {0, 10.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 2.0}, {0, 0}, {0, -30.0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {2.0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0.5, 0}, {-1.0, 0}, {1.5, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {-0.5, 0}},
    {{0, 0.25}, {0, 0.375}, {0, 0}, {0, 0}, {0, 0.125}, {0, 0}, {0, -0.5}, {0, 0}, {0, 0}, {0, 0}, {0.1875, -0.1875}, {0, -0.5}, {-0.1875, -0.625}, {0, 0}, {0, 0}, {0.1875, 0}, {0, 0}, {0, 0.25}, {0, 1.25}, {-0.1875, 3.75}, {0.5, 0}, {0.125, 0}, {-0.3125, 0}, {0, 0}, {-0.125, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0.125, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.125, 0}, {-0.25, 0}, {0.625, 0}, {0.25, 0}, {-0.375, 0}, {0.0625, 0}, {-0.1875, 0}, {0.125, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0.625, 0}, {0, 0}, {0, 0}, {-0.625, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {-0.0625, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 2.0}, {0, -6.0}, {0, 12.0}, {0, -20.0}, {0, 0}, {0, 0}, {0, 0}, {0, -3.0}, {0, 12.0}, {0, -30.0}, {0, 60.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-3.0, 0}, {6.0, 0}, {-10.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 1.5}, {0, -2.25}, {0, 0}, {0, -0.75}, {0, 1.5}, {0, -2.25}, {0, 3.0}, {0, 0}, {0, 0}, {0, 1.5}, {0, -2.25}, {0, 0}, {0, 7.5}, {0, 0}, {0, 0}, {0, 0}, {0, -2.25}, {0, 3.0}, {0, 7.5}, {0, -45.0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {-1.5, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-1.5, 0}, {3.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.75, 0}, {-0.75, 0}, {0.75, 0}, {0.75, 0}, {-1.0, 0}, {1.25, 0}, {-1.5, 0}, {0, 0}, {-0.75, 0}, {1.25, 0}, {-1.5, 0}, {1.5, 0}, {0, 0}, {0, 0}, {0.75, 0}, {-1.5, 0}, {1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.75, 0}},
    {{0, 0.375}, {0, 0}, {0, 0}, {0, -0.1875}, {0, 0.375}, {0, 0}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0.375}, {0, 0}, {0.1875, -0.75}, {-0.1875, 0}, {0, 0}, {-0.1875, 0}, {0.375, 0}, {0, -0.5625}, {0, -0.75}, {0.1875, 1.875}, {-0.5625, 11.25}, {0, 0}, {0.375, 0}, {-0.375, 0}, {0.25, 0}, {-0.3125, 0}, {0.375, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.1875, 0}, {-0.75, 0}, {0, 0}, {0.375, 0}, {-0.375, 0}, {0.375, 0}, {-0.375, 0}, {0.375, 0}, {0.1875, 0}, {-0.3125, 0}, {0.25, 0}, {0, 0}, {0, 0}, {-0.1875, 0}, {0.25, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {-0.375, 0}, {1.875, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.375, 0}, {0.75, 0}, {0, 0}, {-0.375, 0}},
    {{0, 0}, {0, 0.09375}, {0, 0}, {0, -0.015625}, {0.0625, 0.03125}, {0, 0.09375}, {-0.0625, 0.125}, {0, 0}, {0, 0}, {0.0625, 0.03125}, {0.140625, 0.046875}, {0.046875, 0}, {-0.0625, -0.15625}, {0, 0}, {-0.046875, 0}, {-0.015625, 0}, {0, -0.046875}, {0, -0.1875}, {0.046875, -0.46875}, {0.09375, -0.9375}, {0.1875, 0}, {0.09375, 0}, {-0.046875, 0}, {0.03125, 0}, {-0.046875, 0}, {-0.03125, 0}, {0, 0}, {-0.03125, 0}, {0, 0}, {0.046875, 0}, {0, 0}, {0, 0}, {0.03125, 0}, {0.046875, 0}, {0, 0}, {0.15625, 0}, {0.09375, 0}, {-0.0625, 0}, {0.046875, 0}, {-0.046875, 0}, {-0.03125, 0}, {0.015625, 0}, {-0.03125, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {-0.015625, 0}, {0.015625, 0}, {0.046875, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0, 0}, {-0.09375, 0}, {-0.3125, 0}, {0, 0}, {0, 0}, {-0.15625, 0}, {0, 0}, {-0.09375, 0}, {-0.0625, 0}, {0, 0}, {-0.046875, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, -5.0}, {0, 0}, {0, 0}, {0, 2.0}, {0, -6.0}, {0, 12.0}, {0, -20.0}, {0, 30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {-3.0, 0}, {4.0, 0}, {-5.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, -0.5}, {0, 1.0}, {0, -1.5}, {0, 2.0}, {0, 0}, {0, -1.0}, {0, 1.5}, {0, -1.5}, {0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 2.0}, {0, -3.0}, {0, 0}, {0, 10.0}, {0, -30.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {-0.5, 0}, {0, 0}, {-0.5, 0}, {1.0, 0}, {-1.5, 0}, {2.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {-0.5, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {1.5, 0}, {-1.5, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.375}, {0, -0.5625}, {0, 0}, {0, -0.375}, {0, 0.375}, {0, 0}, {0, -0.75}, {0, 0}, {0, -0.375}, {0, 0.375}, {0, 0}, {0, -0.75}, {0, 1.875}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0.75}, {0, 0}, {-0.1875, -1.5}, {0.375, 0}, {-0.5625, 11.25}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0.375, 0}, {-0.3125, 0}, {0.25, 0}, {-0.1875, 0}, {0, 0}, {-0.375, 0}, {0.375, 0}, {0, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0}, {0.375, 0}, {-0.3125, 0}, {0.25, 0}, {-0.1875, 0}, {0.375, 0}, {-0.375, 0}, {0.25, 0}, {0, 0}, {-0.375, 0}, {0, 0}, {-0.375, 0}, {0.375, 0}, {0, 0}, {-0.75, 0}, {1.875, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.1875, 0}},
    {{0, 0.03125}, {0, 0.1875}, {0, 0}, {0, -0.09375}, {0, 0}, {0.0625, 0.09375}, {-0.0625, 0}, {0, 0}, {-0.0625, -0.0625}, {0.125, 0.03125}, {0, 0.09375}, {0.09375, -0.0625}, {-0.09375, -0.625}, {0.09375, 0}, {-0.0625, 0}, {0.03125, 0.125}, {0, 0.1875}, {-0.09375, 0}, {0.03125, -0.625}, {0.1875, -1.875}, {0, 0}, {0.09375, 0}, {-0.09375, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {0.09375, 0}, {-0.0625, 0}, {0, 0}, {0.09375, 0}, {0, 0}, {-0.09375, 0}, {0, 0}, {0.09375, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.09375, 0}, {-0.0625, 0}, {0.03125, 0}, {0.09375, 0}, {-0.0625, 0}, {0, 0}, {0.09375, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {0.03125, 0}, {0.09375, 0}, {-0.0625, 0}, {-0.625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0, 0}, {-0.09375, 0}},
    {{0, -0.015625}, {0.01953125, -0.01171875}, {0, 0}, {-0.01953125, -0.0078125}, {0.03125, -0.0078125}, {0.015625, 0}, {-0.00390625, 0.015625}, {0, 0}, {-0.015625, -0.00390625}, {-0.0234375, 0}, {0.03515625, 0.01171875}, {0.0234375, 0.03125}, {0.00390625, 0.05859375}, {0.01171875, 0}, {-0.00390625, 0}, {-0.01171875, 0.0078125}, {0, 0.0234375}, {-0.01171875, 0.046875}, {-0.015625, 0.078125}, {-0.01171875, 0.1171875}, {0.03125, 0}, {0.0234375, 0}, {0.00390625, 0}, {0.015625, 0}, {0, 0}, {-0.0078125, 0}, {0.0078125, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {-0.00390625, 0}, {0, 0}, {-0.0078125, 0}, {-0.0078125, 0}, {0, 0}, {0.015625, 0}, {0.01953125, 0}, {0.015625, 0}, {-0.00390625, 0}, {0.01171875, 0}, {-0.00390625, 0}, {-0.01171875, 0}, {0.0078125, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {-0.00390625, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0.00390625, 0}, {0.01953125, 0}, {0, 0}, {-0.00390625, 0}, {0, 0}, {0.01171875, 0}, {0.03125, 0}, {0.05859375, 0}, {0, 0}, {0, 0}, {-0.01953125, 0}, {0, 0}, {-0.015625, 0}, {-0.0234375, 0}, {0, 0}, {-0.01171875, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, -5.0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -0.25}, {0, 0.5}, {0, -0.75}, {0, 1.0}, {0, -1.25}, {0, 0}, {0, -1.25}, {0, 1.5}, {0, -0.75}, {0, -1.0}, {0, 3.75}, {0, -7.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {-0.5, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {1.25, 0}, {-1.0, 0}, {0.75, 0}, {-0.5, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, -0.0625}, {0, 0.125}, {0, -0.1875}, {0, 0.25}, {0, 0}, {0, -0.25}, {0, 0.25}, {0, 0}, {0, -0.5}, {0, 1.25}, {0, 0}, {0, -0.625}, {0, 0.25}, {0.1875, 0.375}, {-0.1875, -0.5}, {0.1875, -0.625}, {-0.1875, 3.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.125, 0}, {-0.125, 0}, {0.125, 0}, {-0.125, 0}, {0.5, 0}, {-0.3125, 0}, {0.125, 0}, {0.0625, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0.25, 0}, {-0.1875, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {0.625, 0}, {-0.375, 0}, {0.125, 0}, {0.125, 0}, {-0.375, 0}, {0.625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.03125}, {0, -0.046875}, {0, 0}, {0, -0.046875}, {0, 0.03125}, {0, 0.046875}, {0, -0.1875}, {0.0625, 0}, {-0.0625, -0.09375}, {0.0625, 0}, {0, 0.09375}, {0, 0}, {0, -0.46875}, {0.046875, 0}, {-0.046875, -0.15625}, {0.046875, -0.0625}, {0.140625, 0.09375}, {-0.0625, 0.125}, {-0.015625, -0.15625}, {0.09375, -0.9375}, {0, 0}, {0, 0}, {0, 0}, {0.03125, 0}, {-0.03125, 0}, {0.03125, 0}, {0.09375, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {0.1875, 0}, {-0.046875, 0}, {-0.03125, 0}, {0.046875, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.015625, 0}, {0.046875, 0}, {-0.03125, 0}, {0.015625, 0}, {0, 0}, {0.09375, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {-0.09375, 0}, {0.15625, 0}, {-0.0625, 0}, {-0.03125, 0}, {0.0625, 0}, {0.03125, 0}, {-0.3125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.015625, 0}},
    {{0, 0}, {0, 0.0234375}, {0.01953125, 0}, {-0.01953125, -0.01171875}, {0, -0.0078125}, {0.015625, 0.01171875}, {-0.015625, 0.046875}, {0.03125, 0}, {-0.00390625, -0.015625}, {-0.0234375, -0.015625}, {0, 0}, {0.01171875, 0.03125}, {-0.01171875, 0.078125}, {0.0234375, 0}, {-0.00390625, -0.01953125}, {-0.015625, -0.0234375}, {0.03515625, -0.01171875}, {0.00390625, 0.015625}, {-0.01171875, 0.05859375}, {-0.01171875, 0.1171875}, {0, 0}, {0.0078125, 0}, {-0.0078125, 0}, {0.015625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0.0234375, 0}, {0, 0}, {-0.0078125, 0}, {0, 0}, {0.03125, 0}, {0.00390625, 0}, {-0.0078125, 0}, {-0.00390625, 0}, {0.015625, 0}, {0, 0}, {0.00390625, 0}, {-0.00390625, 0}, {0.0078125, 0}, {-0.00390625, 0}, {0, 0}, {0.01171875, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0.01171875, 0}, {0.015625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0.00390625, 0}, {0.03125, 0}, {0.01953125, 0}, {-0.00390625, 0}, {-0.01171875, 0}, {-0.00390625, 0}, {0.01953125, 0}, {0.05859375, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.00390625, 0}, {0.0078125, 0}, {0, 0}, {-0.0078125, 0}},
    {{0.005859375, -0.001953125}, {0.0048828125, -0.0029296875}, {0.0048828125, 0}, {0.00390625, -0.0009765625}, {0.00390625, -0.001953125}, {0.00390625, -0.0029296875}, {0.0029296875, -0.00390625}, {0.00390625, 0}, {0.0029296875, -0.0009765625}, {0.001953125, -0.001953125}, {0.0029296875, -0.0029296875}, {0.0029296875, -0.00390625}, {0.001953125, -0.0048828125}, {0.0029296875, 0}, {0.001953125, -0.0009765625}, {0.0009765625, -0.001953125}, {0.0029296875, -0.0029296875}, {0.001953125, -0.00390625}, {0.0009765625, -0.0048828125}, {0, -0.005859375}, {0.001953125, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {0.0009765625, 0}, {0.0009765625, 0}, {0, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {-0.0029296875, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {-0.0029296875, 0}, {-0.00390625, 0}, {0, 0}, {0, 0}, {-0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {0, 0}, {-0.0009765625, 0}},
    {{0, 0}, {0, -1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {0, 0}, {0, 0}},
    {{0, 1.0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -5.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {0, 0}, {-1.0, 0}, {2.0, 0}, {0, 0}, {0, 0}},
    {{0, 0.25}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -0.25}, {0, -0.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.25}, {0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, -0.25}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.5, 0}, {0.25, 0}, {-1.0, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}},
    {{0, 2.0}, {0, -3.0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 4.0}, {0, -10.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -5.0}, {0, 15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0, 0}, {-1.0, 0}},
    {{0, 0.75}, {0, -0.75}, {0, 0}, {0, 0}, {0, 0.5}, {0, -0.5}, {0, -1.0}, {0, 0}, {0, 0}, {0, 0}, {0, -0.5}, {0, 0.25}, {0, 3.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.5}, {0, 0}, {0, -7.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-1.25, 0}, {0, 0}, {1.25, 0}, {-1.25, 0}, {0.5, 0}, {-1.0, 0}, {1.5, 0}, {0, 0}, {-0.5, 0}},
    {{0, 0.0625}, {0, 0.1875}, {0, 0}, {0, 0}, {0, 0.0625}, {0, 0.0625}, {0, -0.0625}, {0, 0}, {0, 0}, {0, 0}, {0, -0.0625}, {0, -0.1875}, {0, -0.3125}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.0625}, {0, 0.3125}, {0, 0.9375}, {0.0625, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.3125, 0}, {0.0625, 0}, {-0.1875, 0}, {0, 0}, {-0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {0.3125, 0}, {0.9375, 0}, {0.3125, 0}, {-0.3125, 0}, {0.0625, 0}, {-0.1875, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}},
    {{0, 1.0}, {0, -1.0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, -10.0}, {0, 0}, {0, 0}, {0, 0}, {0, -1.0}, {0, 4.0}, {0, -10.0}, {0, 20.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}},
    {{0, 1.25}, {0, -1.5}, {0, 0}, {0, -0.75}, {0, 1.0}, {0, -0.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0.75}, {0, -1.0}, {0, -0.5}, {0, 5.0}, {0, 0}, {0, 0}, {0, 0}, {0, -0.75}, {0, 1.0}, {0, 2.5}, {0, -15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {1.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {1.0, 0}, {-2.5, 0}, {0, 0}, {0, 0}, {0, 0}, {1.0, 0}, {-1.0, 0}, {1.0, 0}, {0.75, 0}, {-1.0, 0}},
    {{0, 0.125}, {0, 0.375}, {0, 0}, {0, -0.1875}, {0, 0.125}, {0, 0.125}, {0, -0.5}, {0, 0}, {0, 0}, {0, 0.1875}, {0, 0.0625}, {0, -0.375}, {0, -0.625}, {0, 0}, {0, 0}, {0, 0}, {0, -0.1875}, {0, -0.25}, {0, 0.625}, {0, 3.75}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.0625, 0}, {0.25, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.125, 0}, {-0.1875, 0}, {0.25, 0}, {0, 0}, {-0.125, 0}, {0.125, 0}, {0, 0}, {0, 0}, {0, 0}, {0.125, 0}, {-0.0625, 0}, {-0.5, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.125, 0}, {0, 0}, {1.25, 0}, {0, 0}, {0.625, 0}, {-0.625, 0}, {0.5, 0}, {-0.375, 0}, {0.25, 0}, {0.1875, 0}, {-0.3125, 0}},
    {{0, -0.03125}, {0, 0}, {0, 0}, {0, -0.015625}, {0, 0}, {0, 0.03125}, {0, 0.0625}, {0, 0}, {0, 0}, {0, 0.015625}, {0.015625, 0.03125}, {0, 0.03125}, {-0.015625, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0, -0.015625}, {0, -0.0625}, {0, -0.15625}, {-0.015625, -0.3125}, {0.0625, 0}, {0.015625, 0}, {-0.03125, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {-0.0625, 0}, {0.15625, 0}, {0.0625, 0}, {-0.03125, 0}, {0.015625, 0}, {-0.03125, 0}, {-0.03125, 0}, {0, 0}, {-0.015625, 0}, {0, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {0.03125, 0}, {0.03125, 0}, {0, 0}, {0, 0}, {0, 0}, {-0.015625, 0}, {-0.0625, 0}, {-0.15625, 0}, {0.3125, 0}, {0.15625, 0}, {0, 0}, {0.0625, 0}, {-0.03125, 0}, {-0.0625, 0}, {0.015625, 0}, {-0.03125, 0}},
    {{0, 0}, {0, 0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, -5.0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -3.0}, {0, 6.0}, {0, -10.0}, {0, 15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.75}, {0, -0.75}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, 0}, {0, -1.0}, {0, 1.25}, {0, -0.75}, {0, -0.5}, {0, 2.5}, {0, 0}, {0, 0}, {0, 1.0}, {0, -1.5}, {0, 0}, {0, 5.0}, {0, -15.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {1.0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.75, 0}, {1.5, 0}, {-2.5, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.75, 0}, {-0.75, 0}},
    {{0, 0.1875}, {0, 0}, {0, 0.375}, {0, -0.375}, {0, 0.1875}, {0, 0.1875}, {0, -0.75}, {0, 0}, {0, -0.375}, {0, 0.1875}, {0, 0.1875}, {0, -0.375}, {0, 0}, {0, 0}, {0, 0}, {0, 0.375}, {0, 0}, {0, -0.75}, {0, 0}, {0, 5.625}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.1875, 0}, {0.375, 0}, {0, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0}, {0.1875, 0}, {-0.1875, 0}, {0.1875, 0}, {-0.1875, 0}, {0, 0}, {-0.1875, 0}, {0.1875, 0}, {0, 0}, {-0.375, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}, {-0.375, 0}, {1.875, 0}, {0, 0}, {0, 0}, {0, 0}, {0.375, 0}, {-0.375, 0}, {0.375, 0}, {0.5625, 0}, {-0.375, 0}},
    {{0, -0.03125}, {0, 0.09375}, {0, 0.0625}, {0, -0.0625}, {0, -0.03125}, {0, 0.0625}, {0, 0.125}, {0, 0}, {0, -0.0625}, {0, -0.015625}, {0, 0.046875}, {0.015625, 0.03125}, {-0.015625, -0.15625}, {0, 0}, {-0.015625, 0}, {0.03125, 0.0625}, {0, 0.09375}, {0, 0}, {0.015625, -0.3125}, {-0.046875, -0.9375}, {0, 0}, {0.046875, 0}, {-0.046875, 0}, {0.03125, 0}, {-0.03125, 0}, {0.03125, 0}, {0, 0}, {-0.03125, 0}, {0.015625, 0}, {0.046875, 0}, {0, 0}, {0, 0}, {0.03125, 0}, {0, 0}, {-0.1875, 0}, {0, 0}, {0.09375, 0}, {-0.09375, 0}, {0.09375, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {-0.046875, 0}, {0, 0}, {0.09375, 0}, {0, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {0, 0}, {0, 0}, {0, 0}, {0.046875, 0}, {0.046875, 0}, {-0.09375, 0}, {-0.46875, 0}, {0, 0}, {0.15625, 0}, {-0.15625, 0}, {0.1875, 0}, {-0.0625, 0}, {-0.0625, 0}, {0.140625, 0}, {-0.046875, 0}},
    {{0, -0.0078125}, {0, -0.01171875}, {0, 0.00390625}, {0, -0.00390625}, {0.00390625, -0.0078125}, {0, -0.0078125}, {-0.00390625, -0.00390625}, {0, 0}, {0, -0.00390625}, {0.00390625, -0.00390625}, {0.01171875, 0}, {0.00390625, 0.0078125}, {-0.00390625, 0.01953125}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0.00390625}, {0, 0.01171875}, {0, 0.0234375}, {0.00390625, 0.0390625}, {0.01171875, 0.05859375}, {0.0234375, 0}, {0.01171875, 0}, {0, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {0.01171875, 0}, {0.0234375, 0}, {0.0390625, 0}, {0.0234375, 0}, {0.0078125, 0}, {0.01171875, 0}, {0, 0}, {-0.0078125, 0}, {0.00390625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {-0.0078125, 0}, {0, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0, 0}, {0.0078125, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {0.01171875, 0}, {0.0234375, 0}, {0.0390625, 0}, {0.05859375, 0}, {0.0390625, 0}, {0.01953125, 0}, {0.0234375, 0}, {0.0078125, 0}, {-0.00390625, 0}, {0.01171875, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 0}, {0, -1.0}, {0, 2.0}, {0, -3.0}, {0, 4.0}, {0, -5.0}, {0, 6.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0.5}, {0, -0.5}, {0, 0.5}, {0, -0.5}, {0, 0.5}, {0, 1.25}, {0, -1.0}, {0, 0.75}, {0, -0.5}, {0, 0.25}, {0, 0}, {0, 0}, {0, -1.25}, {0, 1.5}, {0, -0.75}, {0, -1.0}, {0, 3.75}, {0, -7.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {-0.25, 0}, {0.5, 0}, {-0.75, 0}, {1.0, 0}, {-1.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.1875}, {0, -0.1875}, {0, 0.5}, {0, -0.3125}, {0, 0.125}, {0, 0.0625}, {0, -0.25}, {0, 0.625}, {0, -0.375}, {0, 0.125}, {0, 0.125}, {0, -0.375}, {0, 0.625}, {0, 0}, {0, -0.625}, {0, 0.25}, {0, 0.375}, {0, -0.5}, {0, -0.625}, {0, 3.75}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0, 0}, {-0.0625, 0}, {0.125, 0}, {-0.1875, 0}, {0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.125, 0}, {-0.125, 0}, {0.125, 0}, {-0.125, 0}, {0.25, 0}, {-0.1875, 0}, {0.125, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {-0.25, 0}, {0.25, 0}, {0, 0}, {-0.5, 0}, {1.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.1875, 0}, {-0.1875, 0}},
    {{0, -0.015625}, {0, 0.09375}, {0, 0.1875}, {0, -0.046875}, {0, -0.03125}, {0, 0.046875}, {0, 0}, {0, 0.15625}, {0, -0.0625}, {0, -0.03125}, {0, 0.0625}, {0, 0.03125}, {0, -0.3125}, {0.015625, 0}, {-0.015625, -0.15625}, {0.015625, -0.0625}, {0, 0.09375}, {-0.015625, 0.125}, {0.03125, -0.15625}, {-0.046875, -0.9375}, {0, 0}, {0, 0}, {0, 0}, {0.03125, 0}, {-0.03125, 0}, {0.03125, 0}, {0.046875, 0}, {-0.03125, 0}, {0.015625, 0}, {0, 0}, {0, 0}, {-0.046875, 0}, {0.03125, 0}, {0.046875, 0}, {-0.1875, 0}, {0, 0}, {0, 0}, {0, 0}, {0.046875, 0}, {-0.046875, 0}, {0.046875, 0}, {0.09375, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {0.09375, 0}, {-0.046875, 0}, {0, 0}, {0.046875, 0}, {-0.09375, 0}, {0, 0}, {-0.09375, 0}, {0, 0}, {0.09375, 0}, {0, 0}, {-0.46875, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0.140625, 0}, {-0.0625, 0}},
    {{0, -0.01171875}, {0, -0.01171875}, {0, 0.03125}, {0, 0.00390625}, {0, -0.0078125}, {0.00390625, -0.00390625}, {-0.00390625, 0.015625}, {0, 0.01953125}, {-0.00390625, -0.00390625}, {0.0078125, -0.01171875}, {0, -0.00390625}, {0.0078125, 0.01953125}, {-0.0078125, 0.05859375}, {0.0078125, 0}, {-0.00390625, -0.01953125}, {0, -0.0234375}, {0, -0.01171875}, {-0.0078125, 0.015625}, {0, 0.05859375}, {0.0234375, 0.1171875}, {0, 0}, {0.01171875, 0}, {-0.01171875, 0}, {0.015625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0.01171875, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0.01171875, 0}, {0, 0}, {-0.01171875, 0}, {-0.0078125, 0}, {0.01171875, 0}, {0.046875, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.0234375, 0}, {-0.00390625, 0}, {-0.015625, 0}, {0.0234375, 0}, {0, 0}, {-0.0078125, 0}, {0, 0}, {0.015625, 0}, {-0.00390625, 0}, {-0.0078125, 0}, {0.00390625, 0}, {0.03125, 0}, {0, 0}, {-0.015625, 0}, {-0.015625, 0}, {0, 0}, {0.03125, 0}, {0.078125, 0}, {0, 0}, {0.01953125, 0}, {-0.01953125, 0}, {0.03125, 0}, {-0.00390625, 0}, {-0.0234375, 0}, {0.03515625, 0}, {0.00390625, 0}},
    {{0, 0.0009765625}, {0.0009765625, 0}, {0, 0.001953125}, {-0.0009765625, 0.0009765625}, {0.001953125, 0}, {0.0009765625, -0.0009765625}, {0, -0.001953125}, {0, 0.0009765625}, {-0.0009765625, 0}, {-0.001953125, -0.0009765625}, {0.0029296875, -0.001953125}, {0.001953125, -0.0029296875}, {0.0009765625, -0.00390625}, {0.0009765625, 0}, {0, -0.0009765625}, {-0.0009765625, -0.001953125}, {0, -0.0029296875}, {-0.0009765625, -0.00390625}, {-0.001953125, -0.0048828125}, {-0.0029296875, -0.005859375}, {0.00390625, 0}, {0.0029296875, 0}, {0.001953125, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {-0.0029296875, 0}, {-0.00390625, 0}, {0.0048828125, 0}, {0.00390625, 0}, {0.0029296875, 0}, {0.0029296875, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0.001953125, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {0.0009765625, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {-0.0029296875, 0}, {0, 0}, {-0.0009765625, 0}, {-0.001953125, 0}, {-0.0029296875, 0}, {-0.00390625, 0}, {-0.0048828125, 0}, {0.005859375, 0}, {0.0048828125, 0}, {0.00390625, 0}, {0.00390625, 0}, {0.0029296875, 0}, {0.001953125, 0}, {0.0029296875, 0}, {0.001953125, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, -1.0}, {0, 1.0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0.25}, {0, -0.25}, {0, 0.25}, {0, -0.25}, {0, 0.25}, {0, -0.25}, {0, 1.5}, {0, -1.0}, {0, 0.5}, {0, 0}, {0, -0.5}, {0, 1.0}, {0, -1.5}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0.25, 0}, {-0.25, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0}, {0, 0}, {0, 0.0625}, {0, -0.0625}, {0, 0.0625}, {0, -0.0625}, {0, 0.0625}, {0, 0.3125}, {0, -0.1875}, {0, 0.0625}, {0, 0.0625}, {0, -0.1875}, {0, 0.3125}, {0, 0.9375}, {0, -0.3125}, {0, -0.0625}, {0, 0.1875}, {0, -0.0625}, {0, -0.3125}, {0, 0.9375}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {-0.0625, 0}, {0.0625, 0}, {0.3125, 0}, {-0.1875, 0}, {0.0625, 0}, {0.0625, 0}, {-0.1875, 0}, {0.3125, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}},
    {{0, 0.015625}, {0, -0.015625}, {0, 0.0625}, {0, -0.03125}, {0, 0}, {0, 0.03125}, {0, -0.0625}, {0, 0.15625}, {0, -0.03125}, {0, -0.03125}, {0, 0.03125}, {0, 0.03125}, {0, -0.15625}, {0, 0.3125}, {0, 0}, {0, -0.0625}, {0.015625, 0}, {-0.015625, 0.0625}, {0.015625, 0}, {-0.015625, -0.3125}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.015625, 0}, {-0.015625, 0}, {0.0625, 0}, {-0.03125, 0}, {0, 0}, {0.03125, 0}, {-0.0625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}, {0.015625, 0}, {-0.015625, 0}, {0.0625, 0}, {-0.03125, 0}, {0, 0}, {0.03125, 0}, {-0.0625, 0}, {0.15625, 0}, {-0.03125, 0}, {-0.03125, 0}, {0.03125, 0}, {0.03125, 0}, {-0.15625, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0, 0}, {0.015625, 0}, {-0.015625, 0}},
    {{0, -0.00390625}, {0, 0.01171875}, {0, 0.0234375}, {0, 0}, {0, -0.0078125}, {0, 0}, {0, 0.0234375}, {0.00390625, 0.0390625}, {-0.00390625, 0.0078125}, {0.00390625, -0.0078125}, {0, -0.0078125}, {0, 0.0078125}, {0, 0.0390625}, {0.00390625, 0.05859375}, {-0.00390625, 0.01953125}, {0.00390625, -0.00390625}, {0.01171875, -0.01171875}, {-0.00390625, -0.00390625}, {-0.00390625, 0.01953125}, {0.01171875, 0.05859375}, {0, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {-0.00390625, 0}, {0.00390625, 0}, {0.01171875, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0.01171875, 0}, {0.0234375, 0}, {0, 0}, {-0.0078125, 0}, {0, 0}, {0.0234375, 0}, {0, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {-0.00390625, 0}, {0.00390625, 0}, {0.01171875, 0}, {-0.00390625, 0}, {-0.00390625, 0}, {0.01171875, 0}, {0.0234375, 0}, {0, 0}, {-0.0078125, 0}, {0, 0}, {0.0234375, 0}, {0.0390625, 0}, {0.0078125, 0}, {-0.0078125, 0}, {-0.0078125, 0}, {0.0078125, 0}, {0.0390625, 0}, {0, 0}, {0, 0}, {0, 0}, {0.00390625, 0}, {-0.00390625, 0}, {0.00390625, 0}, {0.01171875, 0}, {-0.00390625, 0}},
    {{0, -0.0009765625}, {0, -0.0029296875}, {0.0009765625, 0.00390625}, {-0.0009765625, 0.001953125}, {0, 0}, {0.0009765625, -0.001953125}, {-0.0009765625, -0.00390625}, {0.001953125, 0.0048828125}, {0, 0.0029296875}, {-0.001953125, 0.0009765625}, {0, -0.0009765625}, {0.0009765625, -0.0029296875}, {-0.0009765625, -0.0048828125}, {0.001953125, 0.005859375}, {0, 0.00390625}, {-0.001953125, 0.001953125}, {0.0029296875, 0}, {0.0009765625, -0.001953125}, {-0.0009765625, -0.00390625}, {-0.0029296875, -0.005859375}, {0, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {0.001953125, 0}, {0, 0}, {-0.001953125, 0}, {0.0029296875, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {-0.0029296875, 0}, {0.00390625, 0}, {0.001953125, 0}, {0, 0}, {-0.001953125, 0}, {-0.00390625, 0}, {0, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {0.001953125, 0}, {0, 0}, {-0.001953125, 0}, {0.0029296875, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {-0.0029296875, 0}, {0.00390625, 0}, {0.001953125, 0}, {0, 0}, {-0.001953125, 0}, {-0.00390625, 0}, {0.0048828125, 0}, {0.0029296875, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {-0.0029296875, 0}, {-0.0048828125, 0}, {0, 0}, {0.0009765625, 0}, {-0.0009765625, 0}, {0.001953125, 0}, {0, 0}, {-0.001953125, 0}, {0.0029296875, 0}, {0.0009765625, 0}},
    {{0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0.000244140625}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}, {0.000244140625, 0}},
};
// beta! / (|beta| + k)! of Moments<3,3>::aser_*, k = 3 and 2
XG_AFF_STORAGE const double xg_aser33[84][2] = {
    {0.001984126984126984, 0.017857142857142856},
    {0.00033068783068783067, 0.002976190476190476},
    {0.00033068783068783067, 0.002976190476190476},
    {0.002976190476190476, 0.023809523809523808},
    {0.00013227513227513228, 0.0011904761904761906},
    {6.613756613756614e-05, 0.0005952380952380953},
    {0.0005952380952380953, 0.004761904761904762},
    {0.00013227513227513228, 0.0011904761904761906},
    {0.0005952380952380953, 0.004761904761904762},
    {0.004761904761904762, 0.03333333333333333},
    {9.92063492063492e-05, 0.0008928571428571428},
    {3.306878306878307e-05, 0.00029761904761904765},
    {0.00029761904761904765, 0.002380952380952381},
    {3.306878306878307e-05, 0.00029761904761904765},
    {0.00014880952380952382, 0.0011904761904761906},
    {0.0011904761904761906, 0.008333333333333333},
    {9.92063492063492e-05, 0.0008928571428571428},
    {0.00029761904761904765, 0.002380952380952381},
    {0.0011904761904761906, 0.008333333333333333},
    {0.008333333333333333, 0.05},
    {0.00013227513227513228, 0.0011904761904761906},
    {3.306878306878307e-05, 0.00029761904761904765},
    {0.00029761904761904765, 0.002380952380952381},
    {2.2045855379188714e-05, 0.0001984126984126984},
    {9.92063492063492e-05, 0.0007936507936507937},
    {0.0007936507936507937, 0.005555555555555556},
    {3.306878306878307e-05, 0.00029761904761904765},
    {9.92063492063492e-05, 0.0007936507936507937},
    {0.0003968253968253968, 0.002777777777777778},
    {0.002777777777777778, 0.016666666666666666},
    {0.00013227513227513228, 0.0011904761904761906},
    {0.00029761904761904765, 0.002380952380952381},
    {0.0007936507936507937, 0.005555555555555556},
    {0.002777777777777778, 0.016666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.00033068783068783067, 0.002976190476190476},
    {6.613756613756614e-05, 0.0005952380952380953},
    {0.0005952380952380953, 0.004761904761904762},
    {3.306878306878307e-05, 0.00029761904761904765},
    {0.00014880952380952382, 0.0011904761904761906},
    {0.0011904761904761906, 0.008333333333333333},
    {3.306878306878307e-05, 0.00029761904761904765},
    {9.92063492063492e-05, 0.0007936507936507937},
    {0.0003968253968253968, 0.002777777777777778},
    {0.002777777777777778, 0.016666666666666666},
    {6.613756613756614e-05, 0.0005952380952380953},
    {0.00014880952380952382, 0.0011904761904761906},
    {0.0003968253968253968, 0.002777777777777778},
    {0.001388888888888889, 0.008333333333333333},
    {0.008333333333333333, 0.041666666666666664},
    {0.00033068783068783067, 0.002976190476190476},
    {0.0005952380952380953, 0.004761904761904762},
    {0.0011904761904761906, 0.008333333333333333},
    {0.002777777777777778, 0.016666666666666666},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.001984126984126984, 0.017857142857142856},
    {0.00033068783068783067, 0.002976190476190476},
    {0.002976190476190476, 0.023809523809523808},
    {0.00013227513227513228, 0.0011904761904761906},
    {0.0005952380952380953, 0.004761904761904762},
    {0.004761904761904762, 0.03333333333333333},
    {9.92063492063492e-05, 0.0008928571428571428},
    {0.00029761904761904765, 0.002380952380952381},
    {0.0011904761904761906, 0.008333333333333333},
    {0.008333333333333333, 0.05},
    {0.00013227513227513228, 0.0011904761904761906},
    {0.00029761904761904765, 0.002380952380952381},
    {0.0007936507936507937, 0.005555555555555556},
    {0.002777777777777778, 0.016666666666666666},
    {0.016666666666666666, 0.08333333333333333},
    {0.00033068783068783067, 0.002976190476190476},
    {0.0005952380952380953, 0.004761904761904762},
    {0.0011904761904761906, 0.008333333333333333},
    {0.002777777777777778, 0.016666666666666666},
    {0.008333333333333333, 0.041666666666666664},
    {0.041666666666666664, 0.16666666666666666},
    {0.001984126984126984, 0.017857142857142856},
    {0.002976190476190476, 0.023809523809523808},
    {0.004761904761904762, 0.03333333333333333},
    {0.008333333333333333, 0.05},
    {0.016666666666666666, 0.08333333333333333},
    {0.041666666666666664, 0.16666666666666666},
    {0.16666666666666666, 0.5},
};
#ifndef XG_MOM_NO_NODAL  // host builds of the identities leave the device table out
// degree-4 Lagrange basis of the reference simplex (D = 3) in homogeneous
// monomials: W_k = sum_alpha nodal34[k][alpha] m_alpha
static __device__ const double nodal34[35][35] = {
    {1.0, -4.333333333333333, -4.333333333333333, -4.333333333333333, 4.333333333333333, 8.666666666666666, 8.666666666666666, 4.333333333333333, 8.666666666666666, 4.333333333333333, -1.0, -3.0, -3.0, -3.0, -6.0, -3.0, -1.0, -3.0, -3.0, -1.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, -1.0, 0.0, 0.0, 4.333333333333333, -3.0, -3.0, 0.0, 0.0, 0.0, -4.333333333333333, 8.666666666666666, 8.666666666666666, -3.0, -6.0, -3.0, 0.0, 0.0, 0.0, 0.0, 1.0, -4.333333333333333, -4.333333333333333, 4.333333333333333, 8.666666666666666, 4.333333333333333, -1.0, -3.0, -3.0, -1.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, -1.0, 0.0, 0.0, -3.0, 0.0, 4.333333333333333, -3.0, 0.0, 0.0, -3.0, 0.0, 8.666666666666666, -6.0, 0.0, -4.333333333333333, 8.666666666666666, -3.0, 0.0, 0.0, -1.0, 0.0, 4.333333333333333, -3.0, 0.0, -4.333333333333333, 8.666666666666666, -3.0, 0.0, 1.0, -4.333333333333333, 4.333333333333333, -1.0, 0.0},
    {0.0, 0.0, 0.0, -1.0, 0.0, 0.0, -3.0, 0.0, -3.0, 4.333333333333333, 0.0, 0.0, -3.0, 0.0, -6.0, 8.666666666666666, 0.0, -3.0, 8.666666666666666, -4.333333333333333, 0.0, 0.0, -1.0, 0.0, -3.0, 4.333333333333333, 0.0, -3.0, 8.666666666666666, -4.333333333333333, 0.0, -1.0, 4.333333333333333, -4.333333333333333, 1.0},
    {0.0, 16.0, 0.0, 0.0, -21.333333333333332, -21.333333333333332, -21.333333333333332, 0.0, 0.0, 0.0, 5.333333333333333, 10.666666666666666, 10.666666666666666, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, -12.0, 0.0, 0.0, 40.0, -8.0, -8.0, 0.0, 0.0, 0.0, -12.0, -8.0, -8.0, 4.0, 8.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 5.333333333333333, 0.0, 0.0, -21.333333333333332, 10.666666666666666, 10.666666666666666, 0.0, 0.0, 0.0, 16.0, -21.333333333333332, -21.333333333333332, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 16.0, 0.0, 0.0, -21.333333333333332, 0.0, -21.333333333333332, -21.333333333333332, 0.0, 0.0, 5.333333333333333, 0.0, 10.666666666666666, 10.666666666666666, 0.0, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, -12.0, 0.0, 0.0, -8.0, 0.0, 40.0, -8.0, 0.0, 0.0, 4.0, 0.0, -8.0, 8.0, 0.0, -12.0, -8.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 5.333333333333333, 0.0, 0.0, 10.666666666666666, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 0.0, 5.333333333333333, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 16.0, -21.333333333333332, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 16.0, 0.0, 0.0, -21.333333333333332, 0.0, -21.333333333333332, -21.333333333333332, 0.0, 0.0, 5.333333333333333, 0.0, 10.666666666666666, 10.666666666666666, 0.0, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, -12.0, 0.0, 0.0, -8.0, 0.0, -8.0, 40.0, 0.0, 0.0, 4.0, 0.0, 8.0, -8.0, 0.0, 4.0, -8.0, -12.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 10.666666666666666, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 0.0, 5.333333333333333, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 5.333333333333333, -21.333333333333332, 16.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, -21.333333333333332, 0.0, 10.666666666666666, 10.666666666666666, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 16.0, 0.0, -21.333333333333332, -21.333333333333332, 0.0, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, -8.0, 0.0, -8.0, 8.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -12.0, 0.0, 40.0, -8.0, 0.0, -12.0, -8.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 10.666666666666666, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 16.0, -21.333333333333332, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, -21.333333333333332, 0.0, 10.666666666666666, 10.666666666666666, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 16.0, 0.0, -21.333333333333332, -21.333333333333332, 0.0, 5.333333333333333, 10.666666666666666, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, -8.0, 0.0, 8.0, -8.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -12.0, 0.0, -8.0, 40.0, 0.0, 4.0, -8.0, -12.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 10.666666666666666, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 5.333333333333333, -21.333333333333332, 16.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 10.666666666666666, 0.0, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, -21.333333333333332, 10.666666666666666, 0.0, 0.0, 16.0, -21.333333333333332, 5.333333333333333, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 4.0, 0.0, 0.0, 0.0, 0.0, 0.0, 8.0, 0.0, 0.0, -8.0, -8.0, 0.0, 0.0, 0.0, 0.0, 0.0, 4.0, 0.0, 0.0, -8.0, -8.0, 0.0, 0.0, -12.0, 40.0, -12.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 0.0, 0.0, 0.0, 10.666666666666666, 0.0, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 0.0, 0.0, 0.0, 0.0, 5.333333333333333, 0.0, 0.0, 10.666666666666666, -21.333333333333332, 0.0, 0.0, 5.333333333333333, -21.333333333333332, 16.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 96.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, -32.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 96.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, -32.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 96.0, 0.0, 0.0, -32.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 96.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, -32.0, 0.0, 0.0, -32.0, 96.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
    {0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 256.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0, 0.0},
};
#endif
}  // namespace xg
