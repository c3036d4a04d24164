// xg_elmat.hip -- element matrices B^T W B on MFMA, on a materialised rule or
// fused with the straight-cut rule construction.
//
// Reference: xfem/symboliccutbfi.cpp:76-304 (T_CalcElementMatrixAdd, SIMD
// path): for the proxy pairs (u, v) and (grad u, grad v),
//   elmat += B_test^T diag(w_i |det J_i|) B_trial          (AddABt :272-287)
// i.e. elmat = sum_i w_i |J| (phi phi^T + grad phi grad phi^T).
//
// Mapping on CDNA4 (one wavefront per element, a run of elements per wave: the
// geometry of a run is computed one element per lane):
//  * p <= 2 (FP32 and FP64 results): the Gram form of xg_elmat_core.hpp, FP64
//    matrix instructions over 4 points at a time;
//  * p = 3 and split BF16: quadrature points are produced lane-parallel (lane =
//    point, chunks of CH points); each lane evaluates the degree-P Lagrange
//    shapes and physical gradients of its point and stores them in LDS as
//    B[c][dof][point] (c = 0: value, 1..D: gradient components), CH+1 points per
//    row so both the stores (lane = point) and the MFMA operand loads (lane =
//    (c, dof)) are bank-conflict free; the contraction over (point, component)
//    runs on v_mfma_{f32,f64}_16x16x4 with K = the 4 components of one point
//    (blocks bi <= bj only; the lower blocks are mirrored at store time).  The B
//    operand is the A operand scaled by the point's weight.
//  * FP64 is kept for the geometry (cut points, sub-simplex determinants,
//    weights).
#include "xg_device.hpp"
#include "xg_elmat_core.hpp"
#include "xg_internal.hpp"

using namespace xg;

namespace {

using namespace xg::ecore;

// SPLIT = 1: split-BF16 products (T = float, elmat_one_bf16x3)
template <int D, int P, typename T, int SPLIT = 0>
__global__ __launch_bounds__(128) void k_pipeline(int nel, int run, const int32_t *__restrict__ elems,
                                                  const int32_t *__restrict__ el2v,
                                                  const double *__restrict__ coords,
                                                  const double *__restrict__ lset, int order, int ndt, int dts,
                                                  int mask, T *__restrict__ out, int32_t *err) {
  using C = Cfg<D, P, T>;
  extern __shared__ char smem[];
  __shared__ StageLds s_stage[C::WAVES];
  __shared__ StageTab<D> s_tab;
  __shared__ ElemRec s_rec[C::WAVES][EL_RUN];
  const int wv = threadIdx.x >> 6;
  using EL = ElLds<D, P, T, SPLIT>;
  T *sB = reinterpret_cast<T *>(smem) + (size_t)wv * (EL::BYTES / sizeof(T));
  T *sW = sB + C::SB_SIZE;
  const int lane = threadIdx.x & 63;
  // zero the padding rows once (dofs >= N never get written)
  for (int k = lane; k < EL::ZERO; k += 64) sB[k] = T(0);
  GramLane gl{};
  if constexpr (EL::GRAM) gl = gram_lane<D, P>();
  const int nq_vol = rule_cnt(D, order), nq_if = rule_cnt(D - 1, order);
  // base rules of dimension D, then D - 1 (sized by the order)
  double(*s_rule)[4] = reinterpret_cast<double(*)[4]>(smem + C::WAVES * EL::BYTES);
  stage_tables<D>(s_tab, s_rule, order);
  __syncthreads();  // the only block barrier: before the per-wave loops
  const int wid = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int nwaves = (gridDim.x * blockDim.x) >> 6;
  constexpr int NN = C::N * C::N;
  for (long long base = (long long)wid * run; base < nel; base += (long long)nwaves * run) {
    if (lane < run && base + lane < nel) {
      const int e = elems ? elems[base + lane] : (int)base + lane;
      double V[D + 1][3], l[D + 1];
      load_geom<D>(el2v, coords, lset, e, V, l);
      elem_rec<D>(s_rec[wv][lane], V, l, true);
    }
    wave_sync();
    const int m = min((long long)run, nel - base);
    for (int j = 0; j < m; ++j) {
      const ElemRec &R = s_rec[wv][j];
      const double absdet = R.absdet;
      for (int t = 0; t < ndt; ++t) {
        const int dt = (dts >> (2 * t)) & 3;
        bool bad = false;
        StagedSrc src{&s_stage[wv], dt == IF ? s_rule + nq_vol : s_rule, 0, 0, 1.0};
        const int npts = build_stage<D>(&s_stage[wv], s_tab, R, dt, nq_vol, nq_if, src, bad);
        if (bad && lane == 0) atomicOr(err, 1);
        T *o = out + ((size_t)(base + j) * ndt + t) * NN;
        if constexpr (EL::GRAM)
          elmat_gram<D, P, T>(src, npts, R.g, absdet, mask, gl, reinterpret_cast<double *>(sB), o);
        else if constexpr (SPLIT) elmat_one_bf16x3<D, P>(src, npts, R.g, absdet, mask, sB, sW, o);
        else elmat_one<D, P, T>(src, npts, R.g, absdet, mask, sB, sW, o);
      }
    }
    wave_sync();
  }
}

// gradients of the first D barycentrics (the rows of F^{-1}) and |det F|
template <int D>
__device__ __forceinline__ void element_gradients(const int32_t *__restrict__ el2v, const double *__restrict__ coords,
                                                  int e, double (*g)[3], double &absdet) {
  double V[D + 1][3], F[D * D], Finv[D * D];
  load_geom<D>(el2v, coords, nullptr, e, V, nullptr);
  jacobian<D>(V, F, Finv, absdet);
#pragma unroll
  for (int k = 0; k < D * D; ++k) g[k / D][k % D] = Finv[k];
}

template <typename T>
struct CsrSrc {
  const double4 *pts;
  int base;
  __device__ void point(int g, double *x, double &w) const {
    const double4 p = pts[base + g];
    x[0] = p.x;
    x[1] = p.y;
    x[2] = p.z;
    w = p.w;
  }
};

template <int D, int P, typename T, int SPLIT = 0>
__global__ __launch_bounds__(128) void k_elmat_csr(int nel, int run, const int32_t *__restrict__ elems,
                                                   const int32_t *__restrict__ el2v,
                                                   const double *__restrict__ coords,
                                                   const int32_t *__restrict__ offsets,
                                                   const double4 *__restrict__ pts, int mask,
                                                   T *__restrict__ out) {
  using C = Cfg<D, P, T>;
  extern __shared__ char smem[];
  const int wv = threadIdx.x >> 6;
  using EL = ElLds<D, P, T, SPLIT>;
  T *sB = reinterpret_cast<T *>(smem) + (size_t)wv * (EL::BYTES / sizeof(T));
  T *sW = sB + C::SB_SIZE;
  const int lane = threadIdx.x & 63;
  for (int k = lane; k < EL::ZERO; k += 64) sB[k] = T(0);
  wave_sync();
  const int wid = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int nwaves = (gridDim.x * blockDim.x) >> 6;
  constexpr int NN = C::N * C::N;
  if constexpr (!EL::GRAM) {
    // an element at a time, its geometry in the wave's registers (through LDS,
    // as below, P3 and split BF16 were 3 to 8 % slower: 40,000 tetrahedra of order 4,
    // P3 FP32 320 -> 338 us, P2 BF16X3 139 -> 150)
    for (int i = wid; i < nel; i += nwaves) {
      double g[D][3], absdet;
      element_gradients<D>(el2v, coords, elems ? elems[i] : i, g, absdet);
      CsrSrc<T> src{pts, offsets[i]};
      const int npts = offsets[i + 1] - offsets[i];
      T *o = out + (size_t)i * NN;
      if constexpr (SPLIT) elmat_one_bf16x3<D, P>(src, npts, g, absdet, mask, sB, sW, o);
      else elmat_one<D, P, T>(src, npts, g, absdet, mask, sB, sW, o);
    }
    return;
  }
  __shared__ ElemRec s_rec[C::WAVES][EL::GRAM ? EL_RUN : 1];
  GramLane gl{};
  if constexpr (EL::GRAM) gl = gram_lane<D, P>();
  for (long long base = (long long)wid * run; base < nel; base += (long long)nwaves * run) {
    if (lane < run && base + lane < nel) {
      const int e = elems ? elems[base + lane] : (int)base + lane;
      double V[D + 1][3];
      load_geom<D>(el2v, coords, nullptr, e, V, nullptr);
      elem_rec<D>(s_rec[wv][lane], V, nullptr, false);
    }
    wave_sync();
    const int m = min((long long)run, nel - base);
    if constexpr (EL::GRAM) {
      // the offsets of the run, one per lane; a step's points are loaded while
      // the step before runs, across elements too
      const int off = offsets[base + min(lane, m)];
      double *sL = reinterpret_cast<double *>(sB), *sW2 = sL + 4 * GRAM_PAD;
      const int end = __builtin_amdgcn_readlane(off, m);
      int q0 = __builtin_amdgcn_readlane(off, 0);
      auto load = [&](int q, int q1) { return q + lane < q1 ? pts[q + lane] : make_double4(0.0, 0.0, 0.0, 0.0); };
      int j0 = 1;  // (the run's first elements may have no points)
      while (j0 < m && __builtin_amdgcn_readlane(off, j0) == q0) ++j0;
      double4 nx = load(q0, __builtin_amdgcn_readlane(off, j0));
      for (int j = 0; j < m; ++j) {
        const int q1 = __builtin_amdgcn_readlane(off, j + 1);
        const double absdet = s_rec[wv][j].absdet;
        doublex4 acc{0, 0, 0, 0};
        for (; q0 < q1; q0 += 64) {
          const double4 p = nx;
          if (q0 + 64 < q1) nx = load(q0 + 64, q1);
          else if (q1 < end) {
            // the first points of the next element that has any
            int jn = j + 2;
            while (__builtin_amdgcn_readlane(off, jn) == q1) ++jn;
            nx = load(q1, __builtin_amdgcn_readlane(off, jn));
          }
          const double x[3] = {p.x, p.y, p.z};
          gram_chunk<D>(x, p.w * absdet, min(64, q1 - q0), gl, sL, sW2, acc);
        }
        q0 = q1;
        gram_store<D, P, T>(acc, s_rec[wv][j].g, mask, gl, sW2 + 64, out + (size_t)(base + j) * NN);
      }
    }
    wave_sync();
  }
}

// Fixed-node rule: the degree-Q Lagrange lattice nodes of the reference tet
// with per-element weights (learned rule or contracted subdivision rule).
template <int Q, typename T>
struct WeightSrc {
  const double *w;
  __device__ void point(int g, double *x, double &wt) const {
    constexpr Lattice<3, Q> L{};
    x[0] = (double)L.a[g][0] / Q;
    x[1] = (double)L.a[g][1] / Q;
    x[2] = (double)L.a[g][2] / Q;
    wt = w[g];
  }
};

template <int P, int Q, typename T, int SPLIT = 0>
__global__ __launch_bounds__(128) void k_elmat_weights(int nel, int run, const int32_t *__restrict__ elems,
                                                       const int32_t *__restrict__ el2v,
                                                       const double *__restrict__ coords,
                                                       const double *__restrict__ weights, int mask,
                                                       T *__restrict__ out) {
  using C = Cfg<3, P, T>;
  constexpr int NQ = ndof(3, Q);
  extern __shared__ char smem[];
  const int wv = threadIdx.x >> 6;
  using EL = ElLds<3, P, T, SPLIT>;
  T *sB = reinterpret_cast<T *>(smem) + (size_t)wv * (EL::BYTES / sizeof(T));
  T *sW = sB + C::SB_SIZE;
  const int lane = threadIdx.x & 63;
  for (int k = lane; k < EL::ZERO; k += 64) sB[k] = T(0);
  wave_sync();
  const int wid = __builtin_amdgcn_readfirstlane((blockIdx.x * blockDim.x + threadIdx.x) >> 6);
  const int nwaves = (gridDim.x * blockDim.x) >> 6;
  constexpr int NN = C::N * C::N;
  if constexpr (SPLIT) {  // (as in k_elmat_csr)
    for (int i = wid; i < nel; i += nwaves) {
      double g[3][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}}, absdet = 1.0;
      if (coords) element_gradients<3>(el2v, coords, elems ? elems[i] : i, g, absdet);
      WeightSrc<Q, T> src{weights + (size_t)i * NQ};
      elmat_one_bf16x3<3, P>(src, NQ, g, absdet, mask, sB, sW, out + (size_t)i * NN);
    }
    return;
  }
  __shared__ ElemRec s_rec[C::WAVES][EL::GRAM ? EL_RUN : 1];
  GramLane gl{};
  if constexpr (EL::GRAM) gl = gram_lane<3, P>();
  for (long long base = (long long)wid * run; base < nel; base += (long long)nwaves * run) {
    if (lane < run && base + lane < nel) {
      double V[4][3] = {{1, 0, 0}, {0, 1, 0}, {0, 0, 1}, {0, 0, 0}};
      if (coords) {
        const int e = elems ? elems[base + lane] : (int)base + lane;
        load_geom<3>(el2v, coords, nullptr, e, V, nullptr);
      }
      elem_rec<3>(s_rec[wv][lane], V, nullptr, false);
    }
    wave_sync();
    const int m = min((long long)run, nel - base);
    for (int j = 0; j < m; ++j) {
      const long long i = base + j;
      const ElemRec &R = s_rec[wv][j];
      const double absdet = R.absdet;
      WeightSrc<Q, T> src{weights + (size_t)i * NQ};
      constexpr int npts = NQ;
      T *o = out + (size_t)i * NN;
      if constexpr (EL::GRAM)
        elmat_gram<3, P, T>(src, npts, R.g, absdet, mask, gl, reinterpret_cast<double *>(sB), o);
    }
    wave_sync();
  }
}

int grid_waves(int nel, int run) {
  long long blocks = ((long long)nel + 2 * run - 1) / (2 * run);
  if (blocks > 16384) blocks = 16384;
  if (blocks < 1) blocks = 1;
  return (int)blocks;
}

template <int D, int P, typename T, int SPLIT = 0>
int launch_pipeline(xg_ctx *ctx, int order, int nel, const int32_t *elems, const int32_t *el2v,
                    const double *coords, const double *lset, int ndt, int dts, int mask, void *out) {
  using C = Cfg<D, P, T>;
  const size_t lds = ElLds<D, P, T, SPLIT>::BYTES * C::WAVES + stage_rule_bytes(D, order);
  const int run = el_run(nel);
  k_pipeline<D, P, T, SPLIT><<<grid_waves(nel, run), 64 * C::WAVES, lds, ctx->stream>>>(
      nel, run, elems, el2v, coords, lset, order, ndt, dts, mask, (T *)out, ctx->d_err);
  XG_LAUNCH_CHECK();
  return XG_OK;
}

template <int D, int P, typename T, int SPLIT = 0>
int launch_csr(xg_ctx *ctx, int nel, const int32_t *elems, const int32_t *el2v, const double *coords,
               const int32_t *offsets, const double *pts, int mask, void *out) {
  using C = Cfg<D, P, T>;
  const size_t lds = ElLds<D, P, T, SPLIT>::BYTES * C::WAVES;
  const int run = ElLds<D, P, T, SPLIT>::GRAM ? el_run(nel) : 1;
  k_elmat_csr<D, P, T, SPLIT><<<grid_waves(nel, run), 64 * C::WAVES, lds, ctx->stream>>>(
      nel, run, elems, el2v, coords, offsets, reinterpret_cast<const double4 *>(pts), mask, (T *)out);
  XG_LAUNCH_CHECK();
  return XG_OK;
}

#define XG_DISPATCH(D, p, T, CALL)                  \
  do {                                              \
    if (D == 1 && p == 1) return CALL(1, 1, T);     \
    if (D == 1 && p == 2) return CALL(1, 2, T);     \
    if (D == 1 && p == 3) return CALL(1, 3, T);     \
    if (D == 2 && p == 1) return CALL(2, 1, T);     \
    if (D == 2 && p == 2) return CALL(2, 2, T);     \
    if (D == 2 && p == 3) return CALL(2, 3, T);     \
    if (D == 3 && p == 1) return CALL(3, 1, T);     \
    if (D == 3 && p == 2) return CALL(3, 2, T);     \
    if (D == 3 && p == 3) return CALL(3, 3, T);     \
  } while (0)

}  // namespace

extern "C" int xg_cut_pipeline(xg_ctx *ctx, int D, int p, int order, int nel, const int32_t *elems,
                               const int32_t *el2v, const double *coords, const double *lset_v, int ndt,
                               const int *dts, int mask, int precision, void *out) {
  if (!ctx || D < 1 || D > 3 || p < 1 || p > 3 || nel < 0 || ndt < 1 || ndt > 3 || !dts || order < 0 ||
      order / 2 + 1 > XG_RULE_NMAX || mask < 1 || mask > 3)
    return set_error(XG_ERR_ARG, "xg_cut_pipeline: bad argument");
  const bool moments = (precision & XG_METHOD_MOMENTS) != 0;
  precision &= ~XG_METHOD_MOMENTS;
  if (!moments && xg_rule_cnt[D][order / 2 + 1] > PIPE_NQMAX)
    return set_error(XG_ERR_UNSUPPORTED, "xg_cut_pipeline: order too high for the fused kernel (use xg_elmat)");
  int packed = 0;
  for (int t = 0; t < ndt; ++t) {
    if (dts[t] < 0 || dts[t] > 2) return set_error(XG_ERR_ARG, "xg_cut_pipeline: bad domain type");
    packed |= dts[t] << (2 * t);
  }
  if (nel == 0) return XG_OK;
  if (!el2v || !coords || !lset_v || !out) return set_error(XG_ERR_ARG, "xg_cut_pipeline: null pointer");
  if (moments) {
    if (precision != XG_PREC_FP32 && precision != XG_PREC_FP64)
      return set_error(XG_ERR_UNSUPPORTED, "xg_cut_pipeline: moment form writes FP32 or FP64");
    return launch_moment_pipeline(ctx, D, p, order, nel, elems, el2v, coords, lset_v, ndt, packed, mask,
                                  precision == XG_PREC_FP64, out);
  }
#define CALL_P(DD, PP, TT) launch_pipeline<DD, PP, TT>(ctx, order, nel, elems, el2v, coords, lset_v, ndt, packed, mask, out)
  if (precision == XG_PREC_FP32) XG_DISPATCH(D, p, float, CALL_P);
  if (precision == XG_PREC_FP64) XG_DISPATCH(D, p, double, CALL_P);
#undef CALL_P
#define CALL_S(DD, PP, TT) launch_pipeline<DD, PP, TT, 1>(ctx, order, nel, elems, el2v, coords, lset_v, ndt, packed, mask, out)
  if (precision == XG_PREC_BF16X3) XG_DISPATCH(D, p, float, CALL_S);
#undef CALL_S
  return set_error(XG_ERR_UNSUPPORTED, "xg_cut_pipeline: unsupported precision");
}

template <int P, int Q, typename T, int SPLIT = 0>
int launch_weights(xg_ctx *ctx, int nel, const int32_t *elems, const int32_t *el2v, const double *coords,
                   const double *weights, int mask, void *out) {
  using C = Cfg<3, P, T>;
  const size_t lds = ElLds<3, P, T, SPLIT>::BYTES * C::WAVES;
  const int run = SPLIT ? 1 : el_run(nel);
  k_elmat_weights<P, Q, T, SPLIT><<<grid_waves(nel, run), 64 * C::WAVES, lds, ctx->stream>>>(
      nel, run, elems, el2v, coords, weights, mask, (T *)out);
  XG_LAUNCH_CHECK();
  return XG_OK;
}

extern "C" int xg_elmat_weights(xg_ctx *ctx, int p, int q, int nel, const int32_t *elems, const int32_t *el2v,
                                const double *coords, const double *weights, int mask, int precision, void *out) {
  if (!ctx || p < 1 || p > 2 || q != 4 || nel < 0 || mask < 1 || mask > 3)
    return set_error(XG_ERR_ARG, "xg_elmat_weights: bad argument (p <= 2, q == 4)");
  if (nel == 0) return XG_OK;
  if (!weights || !out || (coords && !el2v)) return set_error(XG_ERR_ARG, "xg_elmat_weights: null pointer");
  if (precision == XG_PREC_FP32)
    return p == 1 ? launch_weights<1, 4, float>(ctx, nel, elems, el2v, coords, weights, mask, out)
                  : launch_weights<2, 4, float>(ctx, nel, elems, el2v, coords, weights, mask, out);
  if (precision == XG_PREC_FP64)
    return p == 1 ? launch_weights<1, 4, double>(ctx, nel, elems, el2v, coords, weights, mask, out)
                  : launch_weights<2, 4, double>(ctx, nel, elems, el2v, coords, weights, mask, out);
  if (precision == XG_PREC_BF16X3)
    return p == 1 ? launch_weights<1, 4, float, 1>(ctx, nel, elems, el2v, coords, weights, mask, out)
                  : launch_weights<2, 4, float, 1>(ctx, nel, elems, el2v, coords, weights, mask, out);
  return set_error(XG_ERR_UNSUPPORTED, "xg_elmat_weights: unsupported precision");
}

extern "C" int xg_elmat(xg_ctx *ctx, int D, int p, int nel, const int32_t *elems, const int32_t *el2v,
                        const double *coords, const int32_t *offsets, const double *pts, int mask,
                        int precision, void *out) {
  if (!ctx || D < 1 || D > 3 || p < 1 || p > 3 || nel < 0 || mask < 1 || mask > 3)
    return set_error(XG_ERR_ARG, "xg_elmat: bad argument");
  if (nel == 0) return XG_OK;
  if (!el2v || !coords || !offsets || !pts || !out) return set_error(XG_ERR_ARG, "xg_elmat: null pointer");
#define CALL_C(DD, PP, TT) launch_csr<DD, PP, TT>(ctx, nel, elems, el2v, coords, offsets, pts, mask, out)
  if (precision == XG_PREC_FP32) XG_DISPATCH(D, p, float, CALL_C);
  if (precision == XG_PREC_FP64) XG_DISPATCH(D, p, double, CALL_C);
#undef CALL_C
#define CALL_CS(DD, PP, TT) launch_csr<DD, PP, TT, 1>(ctx, nel, elems, el2v, coords, offsets, pts, mask, out)
  if (precision == XG_PREC_BF16X3) XG_DISPATCH(D, p, float, CALL_CS);
#undef CALL_CS
  return set_error(XG_ERR_UNSUPPORTED, "xg_elmat: unsupported precision");
}
