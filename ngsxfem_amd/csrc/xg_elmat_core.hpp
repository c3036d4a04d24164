// xg_elmat_core.hpp -- device building blocks of the element-matrix kernels
// (shared by the single-mesh kernels in xg_elmat.hip and the batched
// persistent kernels in xg_batch.hip).  See xg_elmat.hip for the mapping.
#pragma once
#include "xg_device.hpp"

typedef float floatx4 __attribute__((ext_vector_type(4)));
typedef double doublex4 __attribute__((ext_vector_type(4)));

namespace xg {
namespace ecore {


template <typename T>
struct Mfma;
template <>
struct Mfma<float> {
  using acc_t = floatx4;
  static __device__ __forceinline__ acc_t run(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  // output row of accumulator element v in lane group c = lane / 16
  static __device__ __forceinline__ int row(int c, int v) { return 4 * c + v; }
};
template <>
struct Mfma<double> {
  using acc_t = doublex4;
  static __device__ __forceinline__ acc_t run(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  // the FP64 variant interleaves the rows: element v of lane group c is row c + 4 v
  static __device__ __forceinline__ int row(int c, int v) { return c + 4 * v; }
};

__device__ __forceinline__ void wave_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int D, int P, typename T>
struct Cfg {
  static constexpr int N = ndof(D, P);
  static constexpr int NB = (N + 15) / 16;
  static constexpr int CH = (sizeof(T) == 4) ? (NB == 1 ? 64 : 32) : (NB == 1 ? 32 : 16);
  static constexpr int PAD = CH + 1;
  static constexpr int ROWS = N;                      // LDS rows per component (real dofs only)
  static constexpr int SB_SIZE = 4 * ROWS * PAD;      // shape/gradient table per wave
  static constexpr int WAVES = 2;  // 128-thread blocks, <= 35 KB LDS per block
  static constexpr size_t LDS_PER_WAVE = sizeof(T) * (SB_SIZE + CH);
};

// Point sources.  point(g, x, w) gives the reference coordinates x (FP64) and
// the reference weight w of point g; the element kernels multiply by |det F|.
//
// StagedSrc: the straight cut rule built on the fly.  The topology comes from
// the decomposition table (staged in LDS once per block: from global memory its
// wave-uniform entries were a chain of three dependent loads per element and
// domain type), the FP64 sub-simplex vertices are computed by one lane each;
// a lane then maps its point with x = ow V0 + sum_m xi_m V_{m+1}
// (straightcutrule.cpp:80-100) and takes the sub-simplex volume from the same
// vertices, so that no second pass over LDS stands between them.
constexpr int PIPE_NQMAX = 125;  // base rule points (order <= 8 tets)

struct StageLds {
  double V[3][4][3];  // sub-simplex vertices (mapping order, FP64)
};

// What the kernels need of an element, computed by one lane for each of a run
// of elements and read by the whole wave from LDS (every lane computing it for
// the wave's one element took half of the FP64 issue slots at P2)
struct ElemRec {
  double g[4][3];  // gradients of the barycentrics (row m < D: row m of F^{-1})
  double absdet;
  double ifac, t[4];      // cut elements: interface factor, cut parameters in edge order
  int eldom, msk, bad, pad;  // straight-cut domain, sign mask, the reference throws
};
constexpr int EL_RUN = 8;  // elements per run at most
// elements per run: more only while 16,384 waves remain (four for each of the
// 4 x 1024 that run at once: with one or two the last ones run alone; 38,000
// elements in runs of 8 took 139 us, in runs of 2 127)
inline int el_run(int nel) {  // host
  int r = 1;
  while (r < EL_RUN && nel / (2 * r) >= 16384) r *= 2;
  return r;
}

// (l == nullptr: geometry only; cutting: the interface factor is wanted)
template <int D>
__device__ __forceinline__ void elem_rec(ElemRec &R, const double (*V)[3], const double *l, bool with_if) {
  double F[D * D], Finv[D * D], absdet;
  jacobian<D>(V, F, Finv, absdet);
  double s[3] = {0.0, 0.0, 0.0};
#pragma unroll
  for (int m = 0; m < D; ++m)
#pragma unroll
    for (int r = 0; r < 3; ++r) {
      const double v = r < D ? Finv[m * D + r] : 0.0;
      R.g[m][r] = v;
      s[r] -= v;
    }
#pragma unroll
  for (int r = 0; r < 3; ++r) R.g[D][r] = s[r];
  R.absdet = absdet;
  if (!l) return;
  const int eldom = check_if_straight_cut<D>(l), msk = sign_mask<D>(l);
  R.eldom = eldom;
  R.msk = msk;
  R.bad = eldom == IF && !cut_is_valid<D>(l) ? 1 : 0;
  if (eldom != IF) return;
  int c = 0;
#pragma unroll
  for (int a = 0; a <= D; ++a)
#pragma unroll
    for (int b = a + 1; b <= D; ++b)
      if (((msk >> a) & 1) != ((msk >> b) & 1)) R.t[c++] = l[a] / (l[a] - l[b]);
  R.ifac = with_if ? interface_factor<D>(l, Finv) : 1.0;
}

// block-shared tables of the fused kernels: the decomposition entries of
// dimension D and the base rules of dimensions D and D - 1
template <int D>
struct StageTab {
  alignas(8) DecompEntry e[3][16];
};
inline size_t stage_rule_bytes(int D, int order) {  // host
  return sizeof(double) * 4 * (size_t)(xg_rule_cnt[D][order / 2 + 1] + xg_rule_cnt[D - 1][order / 2 + 1]);
}
// every thread of the block; the caller's block barrier follows
template <int D>
__device__ __forceinline__ void stage_tables(StageTab<D> &tab, double (*rule)[4], int order) {
  constexpr int W = sizeof(DecompEntry) / 8 * 48;
  const char *src = reinterpret_cast<const char *>(&xg_decomp_d.e[D - 1][0][0]);
  for (int k = threadIdx.x; k < W; k += blockDim.x)
    __builtin_memcpy(reinterpret_cast<uint64_t *>(&tab.e[0][0]) + k, src + 8 * k, 8);
  const int nq_vol = rule_cnt(D, order), nq_if = rule_cnt(D - 1, order);
  const int off_vol = rule_off(D, order), off_if = rule_off(D - 1, order);
  for (int k = threadIdx.x; k < nq_vol + nq_if; k += blockDim.x) {
    const double *r = xg_rule_data_d[k < nq_vol ? off_vol + k : off_if + k - nq_vol];
#pragma unroll
    for (int c = 0; c < 4; ++c) rule[k][c] = r[c];
  }
}

struct StagedSrc {
  const StageLds *st;
  const double (*R)[4];  // base rule (xi0, xi1, xi2, w), in LDS
  int nq, nv1;           // points per sub-simplex, vertices per sub-simplex
  double ifac;           // interface factor
  // point mapping in FP64 (the barycentric lam_D = 1 - sum xi of the element
  // is formed from these coordinates; FP32 here costs ~1e-6 for P3)
  __device__ void point(int g, double *x, double &w) const {
    const int s = (g >= nq) + (g >= 2 * nq);
    const int k = g - s * nq;
    const double *r = R[k];
    const double(*V)[3] = st->V[s];
    double ow = 1.0;
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (m + 1 < nv1) ow -= r[m];
#pragma unroll
    for (int d = 0; d < 3; ++d) x[d] = ow * V[0][d];
#pragma unroll
    for (int m = 0; m < 3; ++m)
      if (m + 1 < nv1)
#pragma unroll
        for (int d = 0; d < 3; ++d) x[d] += r[m] * V[m + 1][d];
    w = r[3] * (simplex_measure(nv1 - 1, V) * ifac);
  }
};

__device__ __forceinline__ void wave_fence() { wave_sync(); }

// Builds the stage for (element, dt); returns the number of points (0 = no
// rule).  Wave-uniform.  *bad set when the reference throws.
template <int D>
__device__ __forceinline__ int build_stage(StageLds *st, const StageTab<D> &tab, const ElemRec &R, int dt, int nq_vol,
                                           int nq_if, StagedSrc &src, bool &bad) {
  const int lane = threadIdx.x & 63;
  const int eldom = __builtin_amdgcn_readfirstlane(R.eldom);
  bad = false;
  src.nq = nq_vol;
  src.nv1 = D + 1;
  src.ifac = 1.0;
  if (eldom != IF) {
    if (eldom != dt) return 0;
    // uncut: the base rule itself = one "sub-simplex" (origin, e_1, .., e_D)
    // of measure 1
    if (lane < (D + 1) * 3) {
      const int m = lane / 3, d = lane % 3;
      st->V[0][m][d] = (m > 0 && d == m - 1) ? 1.0 : 0.0;
    }
    wave_fence();
    return nq_vol;
  }
  const DecompEntry &E = tab.e[dt][__builtin_amdgcn_readfirstlane(R.msk)];
  const int ns = __builtin_amdgcn_readfirstlane((int)E.ns), nv = __builtin_amdgcn_readfirstlane((int)E.nv);
  if (__builtin_amdgcn_readfirstlane(R.bad) || !__builtin_amdgcn_readfirstlane((int)E.ok)) {
    bad = true;
    return 0;
  }
  // vertex q of sub-simplex s: a reference vertex or a cut point (FP64,
  // straightcutrule.cpp:50)
  if (lane < ns * nv) {
    const int s = nv == 4 ? lane >> 2 : (nv == 3 ? lane / 3 : (nv == 2 ? lane >> 1 : lane)), q = lane - s * nv;
    const int code = E.v[s][q], c = code - (D + 1);
    const int i = c >= 0 ? E.ce[c][0] : code, j = c >= 0 ? E.ce[c][1] : code;
    const double t = c >= 0 ? R.t[c] : 0.0;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double pi = (d == i && i < D) ? 1.0 : 0.0;
      const double pj = (d == j && j < D) ? 1.0 : 0.0;
      st->V[s][q][d] = pi + t * (pj - pi);
    }
  }
  if (dt == IF) {
    src.ifac = R.ifac;
    src.nq = nq_if;
  }
  src.nv1 = nv;
  wave_fence();
  return ns * src.nq;
}

// ---------------------------------------------------------------- Gram form
// p <= 2, FP32 and FP64 output.  The contraction over the points runs on
// v_mfma_f64_16x16x4 with K = 4 points: rows = the N shape functions and the
// D + 1 barycentrics, each a product of two linear factors, so a lane (row, point)
// makes its operand from two LDS reads.  The barycentric block G = sum w lam lam^T
// holds everything the stiffness needs, because the gradients are linear in lam:
// grad_r phi_a = sum_k C_r[a][k] lam_k and K = sum_r C_r G C_r^T, 2 D more MFMAs per
// element whose intermediate is already in operand layout.  With K = the 4
// components of one point (value and gradient) the matrix unit ran 4 times as
// often, every point's N (1 + D) values went through LDS, and FP32 values needed
// FP64 sums of groups of points; here all of it is FP64 until the store.
// Bound: LDS reads and FP64 issue, about 90 cycles per 4 points.
// 61 x 53 x 67 cells, P2, NEG + IF, FP32: 257 -> 109 us; rule, coefficient, matrices,
// vectors on 40^3, order 6: 842 -> 371 us with the coefficient and vector kernels.
constexpr int GRAM_PAD = 68;  // doubles per barycentric: rows 8 banks apart
template <int D, int P>
struct Gram {
  static constexpr int N = ndof(D, P);
  static constexpr int QOFF = P == 1 ? 0 : N;  // rows of the barycentrics
  static constexpr size_t BYTES = sizeof(double) * (4 * GRAM_PAD + 64 + 16);
  static_assert(P > 2 || QOFF + D + 1 <= 16, "one 16 x 16 tile");
};

// a lane's row: u = lam_a (al lam_b + be); its gradient coefficients for the
// barycentric k = lane / 16: cp grad lam_p + cq grad lam_q
struct GramLane {
  int a, b, p, q;
  double al, be, cp, cq;
};
template <int D, int P>
__device__ __forceinline__ GramLane gram_lane() {
  constexpr Lattice<D, P> L{};
  constexpr int N = Gram<D, P>::N;
  const int ii = threadIdx.x & 15, k = (threadIdx.x & 63) >> 4;
  GramLane g{0, 0, 0, 0, 0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int n = 0; n < N; ++n) {
    if (ii != n) continue;
    int i = -1, j = -1;  // the lattice point's vertices
#pragma unroll
    for (int m = 0; m <= D; ++m)
      if (L.a[n][m] > 0) {
        if (i < 0) i = m;
        else j = m;
      }
    if (P == 1) {  // lam_i
      g = GramLane{i, i, i, i, 0.0, 1.0, k <= D ? 1.0 : 0.0, 0.0};
    } else if (j < 0) {  // lam_i (2 lam_i - 1), gradient (4 lam_i - sum lam) grad lam_i
      g = GramLane{i, i, i, i, 2.0, -1.0, k <= D ? (k == i ? 3.0 : -1.0) : 0.0, 0.0};
    } else {  // 4 lam_i lam_j, gradient 4 lam_j grad lam_i + 4 lam_i grad lam_j
      g = GramLane{i, j, i, j, 4.0, 0.0, k == j ? 4.0 : 0.0, k == i ? 4.0 : 0.0};
    }
  }
  if (P > 1 && ii >= N && ii <= N + D) g = GramLane{ii - N, ii - N, 0, 0, 0.0, 1.0, 0.0, 0.0};
  return g;
}

// adds up to 64 points, one per lane (x: reference coordinates; past nch: w = 0)
template <int D>
__device__ __forceinline__ void gram_chunk(const double *x, double w, int nch, const GramLane &gl, double *sL,
                                           double *sW, doublex4 &acc) {
  const int lane = threadIdx.x & 63, c = lane >> 4;
  const double *la = sL + gl.a * GRAM_PAD + c, *lb = sL + gl.b * GRAM_PAD + c;
  double lD = 1.0;
#pragma unroll
  for (int m = 0; m < D; ++m) {
    lD -= x[m];
    sL[m * GRAM_PAD + lane] = x[m];
  }
  sL[D * GRAM_PAD + lane] = lD;
  sW[lane] = w;
  wave_sync();
#pragma unroll 4
  for (int p0 = 0; p0 < nch; p0 += 4) {
    const double u = la[p0] * fma(gl.al, lb[p0], gl.be);
    acc = Mfma<double>::run(u, u * sW[p0 + c], acc);
  }
  wave_sync();
}

// the matrix from the products' sums; sQ: 16 doubles
template <int D, int P, typename T>
__device__ __forceinline__ void gram_store(doublex4 acc, const double (*grad)[3], int mask, const GramLane &gl,
                                           double *sQ, T *out) {
  constexpr int N = Gram<D, P>::N, QOFF = Gram<D, P>::QOFF;
  const int lane = threadIdx.x & 63;
  const int c = lane >> 4, ii = lane & 15;
  if (mask & 2) {
    if (D < 3) {
      if (lane < 16) sQ[lane] = 0.0;
      wave_sync();
    }
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int i = Mfma<double>::row(c, v) - QOFF, j = ii - QOFF;
      if (i >= 0 && i <= D && j >= 0 && j <= D) sQ[i * 4 + j] = acc[v];
    }
    wave_sync();
    const double qa = sQ[(ii & 3) * 4 + c];
    double g[3];
#pragma unroll
    for (int r = 0; r < D; ++r) g[r] = fma(gl.cp, grad[gl.p][r], gl.cq * grad[gl.q][r]);
    // rows 4 r + k of t: (G C_r^T)[k][dof]; element r of lane group c is row 4 r + c,
    // which is what the second product's operand wants
    doublex4 t{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < D; ++r) t = Mfma<double>::run((ii >> 2) == r ? qa : 0.0, g[r], t);
    if (!(mask & 1)) acc = doublex4{0, 0, 0, 0};
#pragma unroll
    for (int r = 0; r < D; ++r) acc = Mfma<double>::run(g[r], t[r], acc);
    wave_sync();
  }
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int i = Mfma<double>::row(c, v);
    if (i < N && ii < N) out[i * N + ii] = (T)acc[v];
  }
}

template <int D, int P, typename T, typename SRC>
__device__ __forceinline__ void elmat_gram(const SRC &src, int npts, const double (*grad)[3], double absdet, int mask,
                                           const GramLane &gl, double *lds, T *out) {
  double *sL = lds, *sW = lds + 4 * GRAM_PAD;
  const int lane = threadIdx.x & 63;
  doublex4 acc{0, 0, 0, 0};
  for (int c0 = 0; c0 < npts; c0 += 64) {
    const int nch = min(64, npts - c0);
    double x[3] = {0.0, 0.0, 0.0}, w = 0.0;
    if (lane < nch) src.point(c0 + lane, x, w);
    gram_chunk<D>(x, w * absdet, nch, gl, sL, sW, acc);
  }
  gram_store<D, P, T>(acc, grad, mask, gl, sW + 64, out);
}

// LDS per wave of the element-matrix kernels
template <int D, int P, typename T, int SPLIT>
struct ElLds {
  static constexpr bool GRAM = P <= 2 && !SPLIT;
  static constexpr size_t BYTES = GRAM ? Gram<D, P>::BYTES : Cfg<D, P, T>::LDS_PER_WAVE;
  static constexpr int ZERO = GRAM ? 0 : Cfg<D, P, T>::SB_SIZE;  // padding rows to clear once
};

// one element (or one (element, dt) pair): accumulate and store
template <int D, int P, typename T, typename SRC>
__device__ __forceinline__ void elmat_one(const SRC &src, int npts, const double (*grad)[3], double absdet,
                                          int mask, T *sB, T *sW, T *out) {
  using C = Cfg<D, P, T>;
  using acc_t = typename Mfma<T>::acc_t;
  constexpr int N = C::N, NB = C::NB, CH = C::CH, PAD = C::PAD;
  const int lane = threadIdx.x & 63;
  const int c = lane >> 4, ii = lane & 15;
  acc_t acc[NB][NB];
  double dacc[NB][NB][sizeof(T) == 4 ? 4 : 1];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc[a][b] = acc_t{0, 0, 0, 0};
#pragma unroll
      for (int v = 0; v < (sizeof(T) == 4 ? 4 : 1); ++v) dacc[a][b][v] = 0.0;
    }
  T FinvT[D * D];
#pragma unroll
  for (int k = 0; k < D * D; ++k) FinvT[k] = (T)grad[k / D][k % D];
  const bool m_mass = mask & 1, m_lap = mask & 2;

  for (int c0 = 0; c0 < npts; c0 += CH) {
    const int nch = min(CH, npts - c0);
    if (lane < CH) {
      const int g = c0 + lane;
      T phi[N], dphi[N][D];
      T w = T(0);
      if (g < npts) {
        double x[3], wr;
        src.point(g, x, wr);
        w = (T)(wr * absdet);
        T lam[D + 1];
        double s = 1.0;
#pragma unroll
        for (int m = 0; m < D; ++m) {
          lam[m] = (T)x[m];
          s -= x[m];
        }
        lam[D] = (T)s;
        h1_shape<D, P, T>(lam, phi, dphi);
      } else {
#pragma unroll
        for (int n = 0; n < N; ++n) {
          phi[n] = T(0);
#pragma unroll
          for (int d = 0; d < D; ++d) dphi[n][d] = T(0);
        }
      }
      sW[lane] = w;
#pragma unroll
      for (int n = 0; n < N; ++n) {
        sB[(0 * N + n) * PAD + lane] = m_mass ? phi[n] : T(0);
#pragma unroll
        for (int r = 0; r < D; ++r) {
          T gr = T(0);
#pragma unroll
          for (int cc = 0; cc < D; ++cc) gr += FinvT[cc * D + r] * dphi[n][cc];
          sB[((1 + r) * N + n) * PAD + lane] = m_lap ? gr : T(0);
        }
      }
    }
    wave_sync();
    // contraction over the chunk's points, 8 at a time: all LDS operand loads
    // of a group are issued before its MFMAs (points past npts carry zero
    // weight and zero shape rows, so rounding nch up to 8 adds nothing)
    const int nch8 = min(CH, (nch + 7) & ~7);
    for (int p0 = 0; p0 < nch8; p0 += 8) {
      T av[8][NB], wv[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        wv[u] = sW[p0 + u];
#pragma unroll
        for (int b = 0; b < NB; ++b) {
          const int dof = b * 16 + ii;  // dofs >= N are zero rows of the MFMA tile
          av[u][b] = dof < N ? sB[(c * N + dof) * PAD + p0 + u] : T(0);
        }
      }
#pragma unroll
      for (int u = 0; u < 8; ++u)
#pragma unroll
        for (int bi = 0; bi < NB; ++bi)
#pragma unroll
          for (int bj = bi; bj < NB; ++bj) acc[bi][bj] = Mfma<T>::run(av[u][bi], av[u][bj] * wv[u], acc[bi][bj]);
      if constexpr (sizeof(T) == 4) {
        // the FP32 sums of a group of 8 points join FP64 accumulators, so
        // the rounding of long point sums does not grow with the rule size
#pragma unroll
        for (int bi = 0; bi < NB; ++bi)
#pragma unroll
          for (int bj = bi; bj < NB; ++bj)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
              dacc[bi][bj][v] += (double)acc[bi][bj][v];
              acc[bi][bj][v] = 0.0f;
            }
      }
    }
    wave_sync();
  }
  // D[row][col]: lane holds col lane%16 and rows Mfma<T>::row(lane/16, v)
#pragma unroll
  for (int bi = 0; bi < NB; ++bi)
#pragma unroll
    for (int bj = bi; bj < NB; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gi = bi * 16 + Mfma<T>::row(c, v), gj = bj * 16 + ii;
        if (gi < N && gj < N) {
          const T val = (sizeof(T) == 4) ? (T)dacc[bi][bj][v] : acc[bi][bj][v];
          out[gi * N + gj] = val;
          if (bi < bj) out[gj * N + gi] = val;
        }
      }
}

// ---------------------------------------------------------------- split BF16
// x = hi + mid + lo, each a BF16 (8 significant bits, round to nearest
// even); the two subtractions are exact in FP32, so hi + mid + lo carries 24
// bits of x
typedef short shortx8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ uint32_t bf16_bits(float x) {
  uint32_t u = __float_as_uint(x);
  u += 0x7fffu + ((u >> 16) & 1u);
  return u >> 16;
}
__device__ __forceinline__ float bf16_value(uint32_t h) { return __uint_as_float(h << 16); }

__device__ __forceinline__ void split3(const float *x, shortx8 &hi, shortx8 &mid, shortx8 &lo) {
#pragma unroll
  for (int u = 0; u < 8; ++u) {
    const uint32_t h = bf16_bits(x[u]);
    const float r1 = x[u] - bf16_value(h);
    const uint32_t m = bf16_bits(r1);
    const float r2 = r1 - bf16_value(m);
    hi[u] = (short)h;
    mid[u] = (short)m;
    lo[u] = (short)bf16_bits(r2);
  }
}

__device__ __forceinline__ floatx4 mfma_bf16(const shortx8 &a, const shortx8 &b, floatx4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                 0, 0, 0);
}

// elmat_one with split-BF16 products on v_mfma_f32_16x16x32_bf16: K = 32 =
// 4 components x 8 points, so one MFMA covers a whole group of 8 points.
// Each lane stores sqrt(|w|) * (value or gradient component) in FP32 (the
// weight sign in sW), the contraction lane (dof, component) splits its 8
// values into hi / mid / lo BF16 vectors and runs the six products
// hi.hi + hi.mid + mid.hi + hi.lo + mid.mid + lo.hi (the dropped ones are
// below 2^-26 relative) with FP32 accumulation; the B operand is the A
// operand with the sign of the points of negative weight flipped.  Each
// group's FP32 sums join FP64 accumulators.  Output FP32.
template <int D, int P, typename SRC>
__device__ __forceinline__ void elmat_one_bf16x3(const SRC &src, int npts, const double (*grad)[3], double absdet,
                                                 int mask, float *sB, float *sW, float *out) {
  using C = Cfg<D, P, float>;
  constexpr int N = C::N, NB = C::NB, CH = C::CH, PAD = C::PAD;
  const int lane = threadIdx.x & 63;
  const int c = lane >> 4, ii = lane & 15;
  floatx4 acc[NB][NB];
  double dacc[NB][NB][4];
#pragma unroll
  for (int a = 0; a < NB; ++a)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      acc[a][b] = floatx4{0, 0, 0, 0};
#pragma unroll
      for (int v = 0; v < 4; ++v) dacc[a][b][v] = 0.0;
    }
  float FinvT[D * D];
#pragma unroll
  for (int k = 0; k < D * D; ++k) FinvT[k] = (float)grad[k / D][k % D];
  const bool m_mass = mask & 1, m_lap = mask & 2;

  for (int c0 = 0; c0 < npts; c0 += CH) {
    const int nch = min(CH, npts - c0);
    if (lane < CH) {
      const int g = c0 + lane;
      float phi[N], dphi[N][D];
      float sw = 0.0f, sgn = 1.0f;
      if (g < npts) {
        double x[3], wr;
        src.point(g, x, wr);
        const double wp = wr * absdet;
        sgn = wp < 0.0 ? -1.0f : 1.0f;
        sw = (float)sqrt(fabs(wp));
        float lam[D + 1];
        double s = 1.0;
#pragma unroll
        for (int m = 0; m < D; ++m) {
          lam[m] = (float)x[m];
          s -= x[m];
        }
        lam[D] = (float)s;
        h1_shape<D, P, float>(lam, phi, dphi);
      } else {
#pragma unroll
        for (int n = 0; n < N; ++n) {
          phi[n] = 0.0f;
#pragma unroll
          for (int d = 0; d < D; ++d) dphi[n][d] = 0.0f;
        }
      }
      sW[lane] = sgn;
#pragma unroll
      for (int n = 0; n < N; ++n) {
        sB[(0 * N + n) * PAD + lane] = m_mass ? sw * phi[n] : 0.0f;
#pragma unroll
        for (int r = 0; r < D; ++r) {
          float gr = 0.0f;
#pragma unroll
          for (int cc = 0; cc < D; ++cc) gr += FinvT[cc * D + r] * dphi[n][cc];
          sB[((1 + r) * N + n) * PAD + lane] = m_lap ? sw * gr : 0.0f;
        }
      }
    }
    wave_sync();
    const int nch8 = min(CH, (nch + 7) & ~7);
    for (int p0 = 0; p0 < nch8; p0 += 8) {
      // sign flips of the group's negative-weight points (BF16 sign bit)
      short flip[8];
      bool anyneg = false;
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        const bool neg = sW[p0 + u] < 0.0f;
        flip[u] = neg ? (short)0x8000 : (short)0;
        anyneg |= neg;
      }
      shortx8 ah[NB], am[NB], al[NB];
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        const int dof = b * 16 + ii;  // dofs >= N are zero rows of the MFMA tile
        float xv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) xv[u] = dof < N ? sB[(c * N + dof) * PAD + p0 + u] : 0.0f;
        split3(xv, ah[b], am[b], al[b]);
      }
#pragma unroll
      for (int bi = 0; bi < NB; ++bi)
#pragma unroll
        for (int bj = bi; bj < NB; ++bj) {
          shortx8 bh = ah[bj], bm = am[bj], bl = al[bj];
          if (anyneg) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              bh[u] ^= flip[u];
              bm[u] ^= flip[u];
              bl[u] ^= flip[u];
            }
          }
          floatx4 t = acc[bi][bj];
          t = mfma_bf16(ah[bi], bh, t);
          t = mfma_bf16(ah[bi], bm, t);
          t = mfma_bf16(am[bi], bh, t);
          t = mfma_bf16(ah[bi], bl, t);
          t = mfma_bf16(am[bi], bm, t);
          t = mfma_bf16(al[bi], bh, t);
#pragma unroll
          for (int v = 0; v < 4; ++v) {
            dacc[bi][bj][v] += (double)t[v];
            t[v] = 0.0f;
          }
          acc[bi][bj] = t;
        }
    }
    wave_sync();
  }
#pragma unroll
  for (int bi = 0; bi < NB; ++bi)
#pragma unroll
    for (int bj = bi; bj < NB; ++bj)
#pragma unroll
      for (int v = 0; v < 4; ++v) {
        const int gi = bi * 16 + 4 * c + v, gj = bj * 16 + ii;
        if (gi < N && gj < N) {
          const float val = (float)dacc[bi][bj][v];
          out[gi * N + gj] = val;
          if (bi < bj) out[gj * N + gi] = val;
        }
      }
}

template <int D>
__device__ __forceinline__ void load_geom(const int32_t *__restrict__ el2v, const double *__restrict__ coords,
                                          const double *__restrict__ lset, int e, double (*V)[3], double *l) {
#pragma unroll
  for (int k = 0; k <= D; ++k) {
    const int v = el2v[(size_t)e * (D + 1) + k];
    if (l) l[k] = lset[v];
#pragma unroll
    for (int d = 0; d < 3; ++d) V[k][d] = d < D ? coords[(size_t)v * D + d] : 0.0;
  }
}


}  // namespace ecore
}  // namespace xg
