// xg_device.hpp -- device building blocks of the cut-element hot path (gfx950).
//
//  * Lagrange lattice tables (compile time), H1 shape functions of degree P.
//  * FP64 element geometry, straight-cut decomposition (topology as small
//    integer index lists into {reference vertices, cut points}).
//  * Base-rule access (rules_table.h, generated by gen_rules.py).
//
// FP64 geometry follows cutint/straightcutrule.cpp operation by operation
// and is compiled with -ffp-contract=off, so that marking decisions and
// sub-simplex counts are bit-exact with an IEEE FP64 evaluation of the same
// algorithm.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rules_table.h"

#define XG_DEV __device__ __forceinline__

namespace xg {

enum { NEG = 0, POS = 1, IF = 2 };

// ---------------------------------------------------------------- lattice
constexpr int binom(int n, int k) {
  if (k < 0 || k > n) return 0;
  int r = 1;
  for (int i = 1; i <= k; ++i) r = r * (n - k + i) / i;
  return r;
}

constexpr int ndof(int D, int P) { return binom(P + D, D); }

// Multi-indices alpha (|alpha| = P) of the degree-P Lagrange lattice in dof
// order: vertex nodes, edge nodes, face nodes, interior nodes.  Support sets
// by size then lexicographically; within one support set alpha descending
// lexicographically.
template <int D, int P>
struct Lattice {
  static constexpr int N = ndof(D, P);
  int a[N][4];
  constexpr Lattice() : a{} {
    int all[ndof(D, P)][4] = {};
    int na = 0;
    for (int a0 = P; a0 >= 0; --a0)
      for (int a1 = (D >= 1 ? P - a0 : 0); a1 >= 0; --a1)
        for (int a2 = (D >= 2 ? P - a0 - a1 : 0); a2 >= 0; --a2) {
          int rest = P - a0 - a1 - a2;
          if (D < 3 && rest != 0) continue;
          all[na][0] = a0;
          all[na][1] = a1;
          all[na][2] = a2;
          all[na][3] = D >= 3 ? rest : 0;
          ++na;
        }
    int cnt = 0;
    for (int s = 1; s <= D + 1; ++s) {
      int sup[4] = {0, 1, 2, 3};
      while (true) {
        int mask = 0;
        for (int i = 0; i < s; ++i) mask |= 1 << sup[i];
        for (int k = 0; k < na; ++k) {
          int m = 0;
          for (int i = 0; i <= D; ++i)
            if (all[k][i] > 0) m |= 1 << i;
          if (m == mask) {
            for (int i = 0; i < 4; ++i) a[cnt][i] = all[k][i];
            ++cnt;
          }
        }
        int i = s - 1;
        while (i >= 0 && sup[i] == D + 1 - s + i) --i;
        if (i < 0) break;
        ++sup[i];
        for (int j = i + 1; j < s; ++j) sup[j] = sup[j - 1] + 1;
      }
    }
  }
};

// H1 Lagrange shape functions of degree P at barycentric coordinates lam
// (lam[k] is the coordinate of reference vertex k, lam[D] = 1 - sum xi).
// phi[N]; dphi[N][D] = d phi / d xi (reference gradient).
template <int D, int P, typename T>
XG_DEV void h1_shape(const T *lam, T *phi, T (*dphi)[D]) {
  constexpr Lattice<D, P> L{};
  constexpr int N = Lattice<D, P>::N;
  T Lv[D + 1][P + 1], dLv[D + 1][P + 1];
#pragma unroll
  for (int k = 0; k <= D; ++k) {
    Lv[k][0] = T(1);
    dLv[k][0] = T(0);
#pragma unroll
    for (int m = 1; m <= P; ++m) {
      const T f = (T(P) * lam[k] - T(m - 1)) / T(m);
      const T df = T(P) / T(m);
      dLv[k][m] = dLv[k][m - 1] * f + Lv[k][m - 1] * df;
      Lv[k][m] = Lv[k][m - 1] * f;
    }
  }
#pragma unroll
  for (int n = 0; n < N; ++n) {
    T val = T(1);
#pragma unroll
    for (int k = 0; k <= D; ++k) val *= Lv[k][L.a[n][k]];
    phi[n] = val;
    if (dphi) {
      T dl[D + 1];
#pragma unroll
      for (int k = 0; k <= D; ++k) {
        T pr = dLv[k][L.a[n][k]];
#pragma unroll
        for (int j = 0; j <= D; ++j)
          if (j != k) pr *= Lv[j][L.a[n][j]];
        dl[k] = pr;
      }
#pragma unroll
      for (int d = 0; d < D; ++d) dphi[n][d] = dl[d] - dl[D];
    }
  }
}

// value of the degree-LO Lagrange interpolant with nodal values cl (dof
// order of Lattice<3,LO>) at reference coordinates x (FP64, fixed order)
template <int LO>
XG_DEV double lagrange_eval3(const double *cl, const double *x) {
  constexpr int NL = ndof(3, LO);
  double lam[4];
  double s = 1.0;
#pragma unroll
  for (int m = 0; m < 3; ++m) {
    lam[m] = x[m];
    s -= x[m];
  }
  lam[3] = s;
  double phi[NL];
  h1_shape<3, LO, double>(lam, phi, (double(*)[3]) nullptr);
  double v = 0.0;
#pragma unroll
  for (int k = 0; k < NL; ++k) v += phi[k] * cl[k];
  return v;
}

// the same on the reference triangle (dof order of Lattice<2,LO>)
template <int LO>
XG_DEV double lagrange_eval2(const double *cl, const double *x) {
  constexpr int NL = ndof(2, LO);
  double lam[3];
  double s = 1.0;
#pragma unroll
  for (int m = 0; m < 2; ++m) {
    lam[m] = x[m];
    s -= x[m];
  }
  lam[2] = s;
  double phi[NL];
  h1_shape<2, LO, double>(lam, phi, (double(*)[2]) nullptr);
  double v = 0.0;
#pragma unroll
  for (int k = 0; k < NL; ++k) v += phi[k] * cl[k];
  return v;
}

// ---------------------------------------------------------------- geometry
// Determinant(col1,col2,col3) in the expansion of xdecompose.hpp:91-99
XG_DEV double det3(const double *c1, const double *c2, const double *c3) {
  return c1[0] * (c2[1] * c3[2] - c2[2] * c3[1]) + c1[1] * (c2[2] * c3[0] - c2[0] * c3[2]) +
         c1[2] * (c2[0] * c3[1] - c2[1] * c3[0]);
}

XG_DEV double norm3(const double *a) { return sqrt(a[0] * a[0] + a[1] * a[1] + a[2] * a[2]); }

// F (row-major, column c = V_c - V_D), F^{-1}, |det F|.  V: (D+1) x 3.
template <int D>
XG_DEV void jacobian(const double (*V)[3], double *F, double *Finv, double &absdet) {
#pragma unroll
  for (int r = 0; r < D; ++r)
#pragma unroll
    for (int c = 0; c < D; ++c) F[r * D + c] = V[c][r] - V[D][r];
  double det;
  if constexpr (D == 1) {
    det = F[0];
    Finv[0] = 1.0 / det;
  } else if constexpr (D == 2) {
    det = F[0] * F[3] - F[1] * F[2];
    Finv[0] = F[3] / det;
    Finv[1] = -F[1] / det;
    Finv[2] = -F[2] / det;
    Finv[3] = F[0] / det;
  } else {
    const double a = F[0], b = F[1], c = F[2], d = F[3], e = F[4], f = F[5], g = F[6], h = F[7],
                 i = F[8];
    const double A = e * i - f * h, B = -(d * i - f * g), C = d * h - e * g;
    det = a * A + b * B + c * C;
    // one reciprocal instead of nine FP64 divisions (F^{-1} only enters
    // gradients and interface weights, never a marking decision)
    const double id = 1.0 / det;
    Finv[0] = A * id;
    Finv[1] = -(b * i - c * h) * id;
    Finv[2] = (b * f - c * e) * id;
    Finv[3] = B * id;
    Finv[4] = (a * i - c * g) * id;
    Finv[5] = -(a * f - c * d) * id;
    Finv[6] = C * id;
    Finv[7] = -(a * h - b * g) * id;
    Finv[8] = (a * e - b * d) * id;
  }
  absdet = fabs(det);
}

// ------------------------------------------------------ straight cut topology
// CheckIfStraightCut (straightcutrule.cpp:11-24) with epsilon = 0
template <int D>
XG_DEV int check_if_straight_cut(const double *l) {
  bool haspos = false, hasneg = false;
#pragma unroll
  for (int i = 0; i <= D; ++i) {
    haspos |= l[i] > 0.0;
    hasneg |= l[i] < 0.0;
  }
  if (haspos == hasneg) return IF;
  return hasneg ? NEG : POS;
}

// Decomposition of a cut simplex (LevelsetCutSimplex::Decompose,
// straightcutrule.cpp:131-196) as index lists into the point array
//   pts[0..D]       = reference vertices,
//   pts[D+1+k]      = k-th cut point (edges i<j in lexicographic order with
//                     (l_i >= 0) != (l_j >= 0), CalcIFPolytopEUsingLset :41-64).
// Returns the number of sub-simplices (0 = error), each with nv = D+1
// vertices (D for dt == IF).  *err = 1 when the reference would throw.
struct Decomp {
  int ns;         // number of sub-simplices
  int nv;         // vertices per sub-simplex
  int nc;         // number of cut points
  int8_t v[3][4]; // vertex indices
  int8_t ce[4][2];// cut edges (i, j)
};

template <int D>
XG_DEV bool decompose(const double *l, int dt, Decomp &dc) {
  const int C0 = D + 1;
  int nc = 0;
  bool ok = true;
#pragma unroll
  for (int i = 0; i <= D; ++i)
#pragma unroll
    for (int j = i + 1; j <= D; ++j)
      if ((l[i] >= 0.0) != (l[j] >= 0.0)) {
        // the pair itself must be a straight cut (no exact zero next to a
        // negative value), straightcutrule.cpp:45-49
        const bool hp = (l[i] > 0.0) || (l[j] > 0.0);
        const bool hn = (l[i] < 0.0) || (l[j] < 0.0);
        ok = ok && hp && hn;
        dc.ce[nc][0] = (int8_t)i;
        dc.ce[nc][1] = (int8_t)j;
        ++nc;
      }
  dc.nc = nc;
  dc.ns = 0;
  if (!ok) return false;
  if (dt == IF) {
    dc.nv = D;
    if (nc == D) {
      for (int k = 0; k < D; ++k) dc.v[0][k] = (int8_t)(C0 + k);
      dc.ns = 1;
    } else if (D == 3 && nc == 4) {
      dc.v[0][0] = C0 + 0; dc.v[0][1] = C0 + 1; dc.v[0][2] = C0 + 3;
      dc.v[1][0] = C0 + 0; dc.v[1][1] = C0 + 2; dc.v[1][2] = C0 + 3;
      dc.ns = 2;
    } else
      return false;
    return true;
  }
  dc.nv = D + 1;
  int R[4], nr = 0;
#pragma unroll
  for (int i = 0; i <= D; ++i)
    if ((dt == POS && l[i] >= 0.0) || (dt == NEG && l[i] < 0.0)) R[nr++] = i;
  if (nr == 1) {
    for (int k = 0; k < nc; ++k) dc.v[0][k] = (int8_t)(C0 + k);
    dc.v[0][nc] = (int8_t)R[0];
    dc.ns = (nc == D) ? 1 : 0;
    return nc == D;
  }
  if (nr == 2 && D == 2) {
    dc.v[0][0] = R[0]; dc.v[0][1] = R[1]; dc.v[0][2] = C0 + 1;
    dc.v[1][0] = C0 + 0; dc.v[1][1] = C0 + 1; dc.v[1][2] = R[0];
    dc.ns = 2;
    return true;
  }
  if (nr == 2 && D == 3) {
    dc.v[0][0] = R[1]; dc.v[0][1] = C0 + 1; dc.v[0][2] = C0 + 2; dc.v[0][3] = C0 + 3;
    dc.v[1][0] = R[0]; dc.v[1][1] = R[1]; dc.v[1][2] = C0 + 1; dc.v[1][3] = C0 + 2;
    dc.v[2][0] = C0 + 0; dc.v[2][1] = C0 + 1; dc.v[2][2] = C0 + 2; dc.v[2][3] = R[0];
    dc.ns = 3;
    return true;
  }
  if (nr == 3 && D == 3) {
    dc.v[0][0] = C0 + 0; dc.v[0][1] = C0 + 1; dc.v[0][2] = C0 + 2; dc.v[0][3] = R[2];
    dc.v[1][0] = R[0]; dc.v[1][1] = R[1]; dc.v[1][2] = R[2]; dc.v[1][3] = C0 + 1;
    dc.v[2][0] = C0 + 0; dc.v[2][1] = C0 + 1; dc.v[2][2] = R[0]; dc.v[2][3] = R[2];
    dc.ns = 3;
    return true;
  }
  return false;
}

// The decomposition depends only on D, dt and the sign mask
// m = sum_i [l_i >= 0] << i, so it is tabulated at compile time (same
// construction as decompose()).  Kernels whose element is wave-uniform read
// the entry with scalar loads instead of rebuilding it in registers.
struct DecompEntry {
  int8_t ns, nv, nc, ok;
  int8_t v[3][4];
  int8_t ce[4][2];
};

constexpr DecompEntry make_decomp_entry(int D, int dt, int mask) {
  DecompEntry E{};
  const int C0 = D + 1;
  int nc = 0;
  for (int i = 0; i <= D; ++i)
    for (int j = i + 1; j <= D; ++j)
      if (((mask >> i) & 1) != ((mask >> j) & 1)) {
        E.ce[nc][0] = (int8_t)i;
        E.ce[nc][1] = (int8_t)j;
        ++nc;
      }
  E.nc = (int8_t)nc;
  E.ok = 0;
  if (dt == IF) {
    E.nv = (int8_t)D;
    if (nc == D && nc > 0) {
      for (int k = 0; k < D; ++k) E.v[0][k] = (int8_t)(C0 + k);
      E.ns = 1;
      E.ok = 1;
    } else if (D == 3 && nc == 4) {
      E.v[0][0] = C0 + 0; E.v[0][1] = C0 + 1; E.v[0][2] = C0 + 3;
      E.v[1][0] = C0 + 0; E.v[1][1] = C0 + 2; E.v[1][2] = C0 + 3;
      E.ns = 2;
      E.ok = 1;
    }
    return E;
  }
  E.nv = (int8_t)(D + 1);
  int R[4] = {0, 0, 0, 0}, nr = 0;
  for (int i = 0; i <= D; ++i) {
    const bool pos = (mask >> i) & 1;
    if ((dt == POS && pos) || (dt == NEG && !pos)) R[nr++] = i;
  }
  if (nr == 1 && nc == D) {
    for (int k = 0; k < nc; ++k) E.v[0][k] = (int8_t)(C0 + k);
    E.v[0][nc] = (int8_t)R[0];
    E.ns = 1;
    E.ok = 1;
  } else if (nr == 2 && D == 2) {
    E.v[0][0] = R[0]; E.v[0][1] = R[1]; E.v[0][2] = C0 + 1;
    E.v[1][0] = C0 + 0; E.v[1][1] = C0 + 1; E.v[1][2] = R[0];
    E.ns = 2;
    E.ok = 1;
  } else if (nr == 2 && D == 3) {
    E.v[0][0] = R[1]; E.v[0][1] = C0 + 1; E.v[0][2] = C0 + 2; E.v[0][3] = C0 + 3;
    E.v[1][0] = R[0]; E.v[1][1] = R[1]; E.v[1][2] = C0 + 1; E.v[1][3] = C0 + 2;
    E.v[2][0] = C0 + 0; E.v[2][1] = C0 + 1; E.v[2][2] = C0 + 2; E.v[2][3] = R[0];
    E.ns = 3;
    E.ok = 1;
  } else if (nr == 3 && D == 3) {
    E.v[0][0] = C0 + 0; E.v[0][1] = C0 + 1; E.v[0][2] = C0 + 2; E.v[0][3] = R[2];
    E.v[1][0] = R[0]; E.v[1][1] = R[1]; E.v[1][2] = R[2]; E.v[1][3] = C0 + 1;
    E.v[2][0] = C0 + 0; E.v[2][1] = C0 + 1; E.v[2][2] = R[0]; E.v[2][3] = R[2];
    E.ns = 3;
    E.ok = 1;
  }
  return E;
}

struct DecompTable {
  DecompEntry e[3][3][16];  // [D-1][dt][mask]
  constexpr DecompTable() : e{} {
    for (int D = 1; D <= 3; ++D)
      for (int dt = 0; dt < 3; ++dt)
        for (int m = 0; m < (1 << (D + 1)); ++m) e[D - 1][dt][m] = make_decomp_entry(D, dt, m);
  }
};

static __device__ const DecompTable xg_decomp_d{};

template <int D>
XG_DEV int sign_mask(const double *l) {
  int m = 0;
#pragma unroll
  for (int i = 0; i <= D; ++i) m |= (l[i] >= 0.0 ? 1 : 0) << i;
  return m;
}

// the reference throws for an exact zero next to a negative value
// (straightcutrule.cpp:45-49) and for an all-zero element (:148, :193)
template <int D>
XG_DEV bool cut_is_valid(const double *l) {
  bool hz = false, hn = false, hp = false;
#pragma unroll
  for (int i = 0; i <= D; ++i) {
    hz |= l[i] == 0.0;
    hn |= l[i] < 0.0;
    hp |= l[i] > 0.0;
  }
  return !(hz && hn) && (hp || hn);
}

// point array: reference vertices then cut points (FP64, exact order of
// straightcutrule.cpp:50: p_i + (l_i/(l_i-l_j)) * (p_j - p_i))
template <int D>
XG_DEV void cut_point_array(const double *l, const Decomp &dc, double (*P)[3]) {
  // reference vertex k < D is e_k, vertex D is the origin
#pragma unroll
  for (int k = 0; k <= D; ++k)
#pragma unroll
    for (int d = 0; d < 3; ++d) P[k][d] = (d == k && k < D) ? 1.0 : 0.0;
  for (int c = 0; c < dc.nc; ++c) {
    const int i = dc.ce[c][0], j = dc.ce[c][1];
    const double t = l[i] / (l[i] - l[j]);
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double pi = (d == i && i < D) ? 1.0 : 0.0;
      const double pj = (d == j && j < D) ? 1.0 : 0.0;
      P[D + 1 + c][d] = pi + t * (pj - pi);
    }
  }
}

// SimpleX::GetVolume (straightcutrule.cpp:66-72) of a sub-simplex with nv
// vertices given by index list idx into P
XG_DEV double simplex_volume(int nv, const int8_t *idx, const double (*P)[3]) {
  const double *p0 = P[idx[0]];
  if (nv == 1) return 1.0;
  if (nv == 2) {
    const double *p1 = P[idx[1]];
    double a[3] = {p1[0] - p0[0], p1[1] - p0[1], p1[2] - p0[2]};
    return norm3(a);
  }
  if (nv == 3) {
    const double *p1 = P[idx[1]], *p2 = P[idx[2]];
    double a[3], b[3], c[3];
    for (int d = 0; d < 3; ++d) {
      a[d] = p2[d] - p0[d];
      b[d] = p1[d] - p0[d];
    }
    c[0] = a[1] * b[2] - a[2] * b[1];
    c[1] = a[2] * b[0] - a[0] * b[2];
    c[2] = a[0] * b[1] - a[1] * b[0];
    return norm3(c);
  }
  const double *p1 = P[idx[1]], *p2 = P[idx[2]], *p3 = P[idx[3]];
  double a[3], b[3], c[3];
  for (int d = 0; d < 3; ++d) {
    a[d] = p3[d] - p0[d];
    b[d] = p2[d] - p0[d];
    c[d] = p1[d] - p0[d];
  }
  return fabs(det3(a, b, c));
}

// interface weight factor |F^{-T} n_ref| with n_ref = grad(l)/|grad(l)|
// (TransformQuadUntrafoToIRInterface, straightcutrule.cpp:558-578)
template <int D>
XG_DEV double interface_factor(const double *l, const double *Finv) {
  double g[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int m = 0; m < D; ++m) g[m] = l[m] - l[D];
  const double gn = norm3(g);
#pragma unroll
  for (int m = 0; m < 3; ++m) g[m] /= gn;
  double nrm[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int r = 0; r < D; ++r) {
    double acc = 0.0;
#pragma unroll
    for (int c = 0; c < D; ++c) acc += Finv[c * D + r] * g[c];
    nrm[r] = acc;
  }
  return norm3(nrm);
}

// ---------------------------------------------- simplex cut helpers
// CheckIfStraightCut (straightcutrule.cpp:11-24, epsilon 0) of n values
XG_DEV int straight_cut(const double *v, int n) {
  bool hp = false, hn = false;
  for (int i = 0; i < n; ++i) {
    hp |= v[i] > 0.0;
    hn |= v[i] < 0.0;
  }
  if (hp == hn) return IF;
  return hn ? NEG : POS;
}

XG_DEV double simplex_measure(int dim, const double (*P)[3]) {
  if (dim == 0) return 1.0;
  if (dim == 1) {
    double a[3] = {P[1][0] - P[0][0], P[1][1] - P[0][1], P[1][2] - P[0][2]};
    return norm3(a);
  }
  double a[3], b[3];
  for (int d = 0; d < 3; ++d) {
    a[d] = P[2][d] - P[0][d];
    b[d] = P[1][d] - P[0][d];
  }
  if (dim == 2) {
    double c[3] = {a[1] * b[2] - a[2] * b[1], a[2] * b[0] - a[0] * b[2], a[0] * b[1] - a[1] * b[0]};
    return norm3(c);
  }
  double c[3] = {P[3][0] - P[0][0], P[3][1] - P[0][1], P[3][2] - P[0][2]};
  return fabs(det3(c, a, b));
}

// children of simplex P (dimension dim, vertex values v) cut by a level set
// with target domain type dt (LevelsetCutSimplex::Decompose through the
// decomposition table); returns the number of children (0 where the table
// has no entry: the reference throws)
XG_DEV int children(int dim, const double (*P)[3], const double *v, int dt, double (*out)[4][3],
                                        bool &bad) {
  int mask = 0;
  for (int i = 0; i <= dim; ++i) mask |= (v[i] >= 0.0 ? 1 : 0) << i;
  const DecompEntry &E = xg_decomp_d.e[dim - 1][dt][mask];
  if (!E.ok) {
    bad = true;
    return 0;
  }
  double C[4][3];
  for (int c = 0; c < E.nc; ++c) {
    const int a = E.ce[c][0], b = E.ce[c][1];
    // CalcIFPolytopEUsingLset: a zero next to a negative value throws
    if ((v[a] == 0.0 && v[b] < 0.0) || (v[b] == 0.0 && v[a] < 0.0)) bad = true;
    const double t = v[a] / (v[a] - v[b]);
    for (int d = 0; d < 3; ++d) C[c][d] = P[a][d] + t * (P[b][d] - P[a][d]);
  }
  for (int s = 0; s < E.ns; ++s)
    for (int k = 0; k < E.nv; ++k) {
      const int code = E.v[s][k];
      for (int d = 0; d < 3; ++d) out[s][k][d] = code <= dim ? P[code][d] : C[code - (dim + 1)][d];
    }
  return E.ns;
}

// polynomial integrand sum_t c[t] x^ex[t][0] y^ex[t][1] z^ex[t][2], passed by
// value to the integration kernels
struct Poly {
  int n;
  double c[32];
  int ex[32][3];
};

// ------------------------------------------------------------------- rules
XG_DEV int rule_n1d(int order) { return order / 2 + 1; }
XG_DEV int rule_off(int D, int order) { return xg_rule_off_d[D][rule_n1d(order)]; }
XG_DEV int rule_cnt(int D, int order) { return xg_rule_cnt_d[D][rule_n1d(order)]; }

}  // namespace xg
