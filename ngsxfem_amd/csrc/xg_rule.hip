// xg_rule.hip -- materialised straight-cut rules (count + fill) and IntegrateX.
//
// Reference: cutint/straightcutrule.cpp:582-677 (StraightCutIntegrationRule),
//            :80-100 (GetPlainIntegrationRule), :558-578 (interface weights),
//            cutint/python_cutint.cpp:66-98 (IntegrateX sums).
//
// count: one thread per element (topology only, integer work).
// fill : a wavefront per run of elements, lanes = quadrature points; each lane
//        writes one double4 (x, y, z, w), so a wave stores 2 KB contiguously.
#include "xg_device.hpp"
#include "xg_elmat_core.hpp"
#include "xg_internal.hpp"

using namespace xg;

namespace {

template <int D>
__device__ __forceinline__ void load_elem(const int32_t *__restrict__ el2v, const double *__restrict__ lset,
                                          const double *__restrict__ coords, int e, double *l,
                                          double (*V)[3]) {
#pragma unroll
  for (int k = 0; k <= D; ++k) {
    const int v = el2v[(size_t)e * (D + 1) + k];
    l[k] = lset[v];
    if (V) {
#pragma unroll
      for (int d = 0; d < 3; ++d) V[k][d] = d < D ? coords[(size_t)v * D + d] : 0.0;
    }
  }
}

// q / d for 0 <= q < 2^24, d >= 1 (float estimate, one correction step)
__device__ __forceinline__ int small_div(int q, int d, float rd) {
  int c = (int)((float)q * rd);
  const int t = q - c * d;
  if (t >= d) ++c;
  else if (t < 0) --c;
  return c;
}

template <int D>
__global__ void k_rule_count(int nel, const int32_t *__restrict__ elems, const int32_t *__restrict__ el2v,
                             const double *__restrict__ lset, int dt, int order, int32_t *__restrict__ cnt,
                             uint8_t *__restrict__ nsub, int32_t *err) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= nel) return;
  const int e = elems ? elems[i] : i;
  double l[D + 1];
  load_elem<D>(el2v, lset, nullptr, e, l, nullptr);
  const int eldom = check_if_straight_cut<D>(l);
  int n = 0, ns = 0;
  if (eldom != IF) {
    n = (eldom == dt) ? rule_cnt(D, order) : 0;
  } else {
    Decomp dc;
    if (!decompose<D>(l, dt, dc)) {
      atomicOr(err, 1);
    } else {
      ns = dc.ns;
      n = dc.ns * rule_cnt(dc.nv - 1, order);
    }
  }
  cnt[i] = n;
  if (nsub) nsub[i] = (uint8_t)ns;
}

// One wave takes epw (a power of two, <= 64) consecutive elements.
//  A. lane = element: the gathers, the class of the element and, for a cut
//     one, its sign mask, cut parameters and interface factor;
//  B. the uncut elements with points: lanes over (element, base point) pairs,
//     so every lane stores whatever the rule's length;
//  C. the sub-simplices of all cut elements in one list, FILL_SUB at a time:
//     lane = sub-simplex for the vertices and the volume (into LDS), then lanes
//     over (sub-simplex, base point) pairs.
// Bound: the stores (32 B a point).  With one wave per element every element
// without points cost a wave its whole chain of dependent gathers, an uncut
// one filled 27 of 64 lanes at order 4, and the decomposition's indexed
// private arrays lived in scratch memory (353 us at 64^3 cells, order 4); with
// the cut elements of a run in turn, each with its own chain of table, LDS and
// point loads, 157 us; now 101 us for 349 MB.  (Pairs of lanes writing whole
// lines, half a point each: no fewer bytes written, 105 us.)
constexpr int FILL_SUB = 32;

template <int D>
__global__ __launch_bounds__(256) void k_rule_fill(int nel, const int32_t *__restrict__ elems,
                                                   const int32_t *__restrict__ el2v,
                                                   const double *__restrict__ coords,
                                                   const double *__restrict__ lset, int dt, int order, int epw,
                                                   const int32_t *__restrict__ offsets,
                                                   double4 *__restrict__ out) {
  __shared__ int32_t s_base[4][64];
  __shared__ uint8_t s_item[4][192];         // sub-simplices of the run: 4 x lane of the element + number
  __shared__ double s_V[4][FILL_SUB][13];    // vertices (mapping order; 4 x 3, one of padding)
  __shared__ double2 s_w[4][FILL_SUB];       // volume, interface factor
  __shared__ int2 s_out[4][FILL_SUB];        // first point, points
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const long long wid = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + wv);
  const long long nwaves = (long long)gridDim.x * 4;
  const int voff = rule_off(D, order), vcnt = rule_cnt(D, order);
  const float rcnt = 1.0f / (float)vcnt;
  const int Ds = dt == IF ? D - 1 : D, off = rule_off(Ds, order), nq = rule_cnt(Ds, order);
  const float rnq = 1.0f / (float)nq;
  for (long long i0 = wid * epw; i0 < nel; i0 += nwaves * epw) {
    int base = 0, npts = 0, msk = 0;
    bool uncut = false, cut = false;
    double t[4] = {0.0, 0.0, 0.0, 0.0}, ifac = 1.0;
    if (lane < epw && i0 + lane < nel) {
      const int i = (int)i0 + lane;
      base = offsets[i];
      npts = offsets[i + 1] - base;
      if (npts > 0) {
        const int e = elems ? elems[i] : i;
        double l[D + 1];
        load_elem<D>(el2v, lset, nullptr, e, l, nullptr);
        cut = check_if_straight_cut<D>(l) == IF;
        uncut = !cut && npts >= vcnt;
        if (cut) {
          msk = sign_mask<D>(l);
          // the cut points of the sign-changing edges in lexicographic order
          // (p_i + (l_i / (l_i - l_j)) (p_j - p_i), straightcutrule.cpp:50)
          int c = 0;
#pragma unroll
          for (int a = 0; a <= D; ++a)
#pragma unroll
            for (int b = a + 1; b <= D; ++b)
              if (((msk >> a) & 1) != ((msk >> b) & 1)) {
                const double q = l[a] / (l[a] - l[b]);
#pragma unroll
                for (int k = 0; k < 4; ++k) t[k] = c == k ? q : t[k];
                ++c;
              }
          if (dt == IF) {
            double ll[D + 1], V[D + 1][3], F[D * D], Finv[D * D], absdet;
            load_elem<D>(el2v, lset, coords, e, ll, V);
            jacobian<D>(V, F, Finv, absdet);
            ifac = interface_factor<D>(l, Finv);
          }
        }
      }
    }
    const unsigned long long mu = __ballot(uncut), mc = __ballot(cut);
    if (mu) {
      if (uncut) s_base[wv][__popcll(mu & ((1ull << lane) - 1ull))] = base;
      ecore::wave_sync();
      const int total = __popcll(mu) * vcnt;
      for (int g = lane; g < total; g += 64) {
        const int s = small_div(g, vcnt, rcnt), k = g - s * vcnt;
        const double *r = xg_rule_data_d[voff + k];
        out[s_base[wv][s] + k] = make_double4(r[0], D > 1 ? r[1] : 0.0, D > 2 ? r[2] : 0.0, r[3]);
      }
      ecore::wave_sync();
    }
    if (mc) {
      const DecompEntry *tab = xg_decomp_d.e[D - 1][dt];
      const int ns = cut ? tab[msk].ns : 0;
      const unsigned long long below = (1ull << lane) - 1ull;
      const unsigned long long n1 = __ballot(ns > 0), n2 = __ballot(ns > 1), n3 = __ballot(ns > 2);
      const int pos = __popcll(n1 & below) + __popcll(n2 & below) + __popcll(n3 & below);
#pragma unroll
      for (int s = 0; s < 3; ++s)
        if (s < ns) s_item[wv][pos + s] = (uint8_t)(4 * lane + s);
      ecore::wave_sync();
      const int nsub = __popcll(n1) + __popcll(n2) + __popcll(n3);
      for (int b0 = 0; b0 < nsub; b0 += FILL_SUB) {
        const int nb = min(FILL_SUB, nsub - b0);
        const int item = lane < nb ? s_item[wv][b0 + lane] : 0;
        const int src = item >> 2, sub = item & 3;
        const double t0 = __shfl(t[0], src, 64), t1 = __shfl(t[1], src, 64), t2 = __shfl(t[2], src, 64),
                     t3 = __shfl(t[3], src, 64), cif = __shfl(ifac, src, 64);
        const int smsk = __shfl(msk, src, 64), sbase = __shfl(base, src, 64), snp = __shfl(npts, src, 64);
        if (lane < nb) {
          const DecompEntry &E = tab[smsk];
          double W[4][3];
#pragma unroll
          for (int q = 0; q < 4; ++q) {
            if (q > Ds) break;
            const int code = E.v[sub][q], c = code - (D + 1);
            const int a = c >= 0 ? E.ce[c][0] : code, b = c >= 0 ? E.ce[c][1] : code;
            const double tc = c == 1 ? t1 : (c == 2 ? t2 : (c == 3 ? t3 : t0));
#pragma unroll
            for (int d = 0; d < 3; ++d) {
              const double pa = (d == a && a < D) ? 1.0 : 0.0, pb = (d == b && b < D) ? 1.0 : 0.0;
              W[q][d] = c >= 0 ? pa + tc * (pb - pa) : pa;
              s_V[wv][lane][3 * q + d] = W[q][d];
            }
          }
          s_w[wv][lane] = make_double2(simplex_measure(Ds, W), cif);
          s_out[wv][lane] = make_int2(sbase + sub * nq, min(snp - sub * nq, nq));
        }
        ecore::wave_sync();
        const int total = nb * nq;
        for (int g = lane; g < total; g += 64) {
          const int s = small_div(g, nq, rnq), k = g - s * nq;
          const int2 o = s_out[wv][s];
          if (k >= o.y) continue;
          const double *r = xg_rule_data_d[off + k];
          const double *W = s_V[wv][s];
          double ow = 1.0;
#pragma unroll
          for (int q = 0; q < D; ++q)
            if (q < Ds) ow -= r[q];
          double x[3];
#pragma unroll
          for (int d = 0; d < 3; ++d) x[d] = ow * W[d];
#pragma unroll
          for (int q = 0; q < D; ++q)
            if (q < Ds)
#pragma unroll
              for (int d = 0; d < 3; ++d) x[d] += r[q] * W[3 * (q + 1) + d];
          const double2 tw = s_w[wv][s];
          double w = r[3] * tw.x;
          if (dt == IF) w = w * tw.y;
          out[o.x + k] = make_double4(x[0], x[1], x[2], w);
        }
        ecore::wave_sync();
      }
    }
  }
}

// adds the points q, q + G, .. (NP of them) below q1 to s, in this order.  A
// term's coefficient and exponents are scalar loads at addresses that depend on
// the loop, about 300 cycles each time, so a term is taken for NP points at once
template <int D, int G, int NP>
__device__ __forceinline__ double integrate_points(int q, int q1, const double *V, const double *F, double absdet,
                                                   const double4 *__restrict__ pts, const Poly &f, double s) {
  double x[NP][3], w[NP], fv[NP];
#pragma unroll
  for (int i = 0; i < NP; ++i) {
    const double4 p = q + i * G < q1 ? pts[q + i * G] : make_double4(0.0, 0.0, 0.0, 0.0);
    const double xi[3] = {p.x, p.y, p.z};
    w[i] = p.w;
    fv[i] = 0.0;
#pragma unroll
    for (int r = 0; r < 3; ++r) x[i][r] = 0.0;
#pragma unroll
    for (int r = 0; r < D; ++r) {
      double a = V[r];
#pragma unroll
      for (int c = 0; c < D; ++c) a += F[r * D + c] * xi[c];
      x[i][r] = a;
    }
  }
  for (int t = 0; t < f.n; ++t) {
    const double c = f.c[t];
    const int ex[3] = {f.ex[t][0], f.ex[t][1], f.ex[t][2]};
    double m[NP];
#pragma unroll
    for (int i = 0; i < NP; ++i) m[i] = c;
#pragma unroll
    for (int d = 0; d < 3; ++d)
      for (int j = 0; j < ex[d]; ++j)
#pragma unroll
        for (int i = 0; i < NP; ++i) m[i] *= x[i][d];
#pragma unroll
    for (int i = 0; i < NP; ++i) fv[i] += m[i];
  }
#pragma unroll
  for (int i = 0; i < NP; ++i)
    if (q + i * G < q1) s += absdet * w[i] * fv[i];
  return s;
}

// A wave takes epw (a power of two, 64 / G <= epw <= INT_EPW) consecutive
// elements: lane = element for the gathers and the map (into LDS), then G lanes
// per element that has points.  A wave per element ran most of its lanes on
// nothing (27 points in 64 lanes, no points at all in the elements outside),
// and its one atomic add per wave queued up on the single address of the total:
// 262,144 adds took 3.16 ms at 64^3 cells, order 4.  Here a block adds its
// waves' sums in LDS and at most 1024 blocks run, so the adds are few.  Bound:
// the points (349 MB there, 73 us); the chain offsets, vertices, coordinates is
// taken once for many elements (with G lanes for every element of the list,
// empty or not, and the polynomial's terms point by point 147 us; now 116 us).
constexpr int INT_EPW = 32;

template <int D, int G>
__global__ __launch_bounds__(512) void k_integrate(int nel, const int32_t *__restrict__ elems,
                                                   const int32_t *__restrict__ el2v,
                                                   const double *__restrict__ coords, int epw,
                                                   const int32_t *__restrict__ offsets,
                                                   const double4 *__restrict__ pts, Poly f,
                                                   double *__restrict__ per_elem, double *total) {
  constexpr int NGEO = D + D * D + 1;
  __shared__ double s_sum[8];
  __shared__ double s_geo[8][INT_EPW][NGEO];  // last vertex, F, |det F|
  __shared__ int4 s_el[8][INT_EPW];           // first and last point, element of the list
  const int lane = threadIdx.x & 63, wv = threadIdx.x >> 6;
  const int sub = lane & (G - 1), grp = lane / G;
  const long long wid = (long long)blockIdx.x * 8 + wv, nwaves = (long long)gridDim.x * 8;
  double acc_all = 0.0;
  for (long long i0 = wid * epw; i0 < nel; i0 += nwaves * epw) {
    int q0 = 0, q1 = 0;
    const bool valid = lane < epw && i0 + lane < nel;
    if (valid) {
      q0 = offsets[i0 + lane];
      q1 = offsets[i0 + lane + 1];
    }
    const unsigned long long mp = __ballot(q1 > q0);
    if (per_elem && valid && q1 <= q0) per_elem[i0 + lane] = 0.0;
    if (!mp) continue;
    if (q1 > q0) {
      const int e = elems ? elems[i0 + lane] : (int)i0 + lane;
      double V[D + 1][3];
#pragma unroll
      for (int k = 0; k <= D; ++k) {
        const int v = el2v[(size_t)e * (D + 1) + k];
#pragma unroll
        for (int d = 0; d < 3; ++d) V[k][d] = d < D ? coords[(size_t)v * D + d] : 0.0;
      }
      double F[D * D], Finv[D * D], absdet;
      jacobian<D>(V, F, Finv, absdet);
      const int slot = __popcll(mp & ((1ull << lane) - 1ull));
      double *geo = s_geo[wv][slot];
#pragma unroll
      for (int r = 0; r < D; ++r) geo[r] = V[D][r];
#pragma unroll
      for (int k = 0; k < D * D; ++k) geo[D + k] = F[k];
      geo[D + D * D] = absdet;
      s_el[wv][slot] = make_int4(q0, q1, lane, 0);
    }
    ecore::wave_sync();
    const int n = __popcll(mp);
    for (int k = grp; k < n; k += 64 / G) {
      const int4 el = s_el[wv][k];
      double V[D], F[D * D];
#pragma unroll
      for (int r = 0; r < D; ++r) V[r] = s_geo[wv][k][r];
#pragma unroll
      for (int r = 0; r < D * D; ++r) F[r] = s_geo[wv][k][D + r];
      const double absdet = s_geo[wv][k][D + D * D];
      double s = 0.0;
      int q = el.x + sub;
      while (q < el.y) {
        if (__ballot(q + G < el.y) != 0ull) {
          s = integrate_points<D, G, 4>(q, el.y, V, F, absdet, pts, f, s);
          q += 4 * G;
        } else {
          s = integrate_points<D, G, 1>(q, el.y, V, F, absdet, pts, f, s);
          q += G;
        }
      }
#pragma unroll
      for (int o = G / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
      if (sub == 0) {
        if (per_elem) per_elem[i0 + el.z] = s;
        acc_all += s;
      }
    }
    ecore::wave_sync();
  }
  if (!total) return;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) acc_all += __shfl_xor(acc_all, o, 64);
  if (lane == 0) s_sum[wv] = acc_all;
  __syncthreads();
  if (threadIdx.x == 0) {
#pragma unroll
    for (int w = 1; w < 8; ++w) acc_all += s_sum[w];
    atomicAdd(total, acc_all);
  }
}

__global__ void k_zero_f64(double *p) { *p = 0.0; }

// integrals on fixed-node rules: W (nel x N) weights at the N nodes of the
// degree-Q Lagrange lattice of the reference tetrahedron (xg_subdiv_weights);
// one thread per element
template <int Q>
__global__ __launch_bounds__(256) void k_integrate_nodes(int nel, const int32_t *__restrict__ elems,
                                                         const int32_t *__restrict__ el2v,
                                                         const double *__restrict__ coords,
                                                         const double *__restrict__ W, Poly f,
                                                         double *__restrict__ per_elem, double *total) {
  constexpr Lattice<3, Q> LAT{};
  constexpr int N = Lattice<3, Q>::N;
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  double s = 0.0;
  if (i < nel) {
    const int e = elems ? elems[i] : i;
    double V[4][3];
#pragma unroll
    for (int k = 0; k <= 3; ++k) {
      const int v = el2v[(size_t)e * 4 + k];
#pragma unroll
      for (int d = 0; d < 3; ++d) V[k][d] = coords[(size_t)v * 3 + d];
    }
    double F[9], Finv[9], absdet;
    jacobian<3>(V, F, Finv, absdet);
    for (int k = 0; k < N; ++k) {
      double x[3];
#pragma unroll
      for (int r = 0; r < 3; ++r) {
        double a = V[3][r];
#pragma unroll
        for (int c = 0; c < 3; ++c) a += F[r * 3 + c] * ((double)LAT.a[k][c] / Q);
        x[r] = a;
      }
      double fv = 0.0;
      for (int t = 0; t < f.n; ++t) {
        double m = f.c[t];
        for (int d = 0; d < 3; ++d)
          for (int j = 0; j < f.ex[t][d]; ++j) m *= x[d];
        fv += m;
      }
      s += absdet * W[(size_t)i * N + k] * fv;
    }
    if (per_elem) per_elem[i] = s;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
  if ((threadIdx.x & 63) == 0 && total) atomicAdd(total, s);
}

// elements per wave of k_rule_fill: one while the waves would not fill the
// device (8192 wave slots), then doubling up to a lane each
int fill_epw(int nel) {
  int epw = 1;
  while (epw < 64 && nel / epw > 16384) epw *= 2;
  return epw;
}

template <int D, int G>
void launch_integrate(xg_ctx *ctx, int nel, const int32_t *elems, const int32_t *el2v, const double *coords,
                      const int32_t *offsets, const double4 *pts, const Poly &f, double *per_elem, double *total) {
  // elements per wave: one for each group of lanes while the waves fit on the
  // device at once, then more
  int epw = 64 / G;
  while (epw < INT_EPW && nel / epw > 16384) epw *= 2;
  const long long want = ((long long)nel + 8LL * epw - 1) / (8LL * epw);
  const int grid = (int)(want < 1024 ? want : 1024);
  k_integrate<D, G><<<grid, 512, 0, ctx->stream>>>(nel, elems, el2v, coords, epw, offsets, pts, f, per_elem, total);
}

}  // namespace

extern "C" int xg_rule_npts(int D, int order) {
  if (D < 0 || D > 3 || order < 0 || order / 2 + 1 > XG_RULE_NMAX) return XG_ERR_ARG;
  return xg_rule_cnt[D][order / 2 + 1];
}

extern "C" int xg_cut_rule_count(xg_ctx *ctx, int D, int nel, const int32_t *elems, const int32_t *el2v,
                                 const double *lset_v, int dt, int order, int32_t *offsets, uint8_t *nsub) {
  if (!ctx || D < 1 || D > 3 || nel < 0 || !offsets || dt < 0 || dt > 2 || order < 0 ||
      order / 2 + 1 > XG_RULE_NMAX)
    return set_error(XG_ERR_ARG, "xg_cut_rule_count: bad argument");
  if (nel > 0 && (!el2v || !lset_v)) return set_error(XG_ERR_ARG, "xg_cut_rule_count: null mesh");
  if (nel == 0) {
    XG_CHECK(hipMemsetAsync(offsets, 0, sizeof(int32_t), ctx->stream));
    return XG_OK;
  }
  const int grid = (nel + 255) / 256;
  switch (D) {
    case 1: k_rule_count<1><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, lset_v, dt, order, offsets, nsub, ctx->d_err); break;
    case 2: k_rule_count<2><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, lset_v, dt, order, offsets, nsub, ctx->d_err); break;
    default: k_rule_count<3><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, lset_v, dt, order, offsets, nsub, ctx->d_err); break;
  }
  XG_LAUNCH_CHECK();
  return scan_exclusive_i32(ctx, offsets, nel, true);
}

extern "C" int xg_cut_rule_fill(xg_ctx *ctx, int D, int nel, const int32_t *elems, const int32_t *el2v,
                                const double *coords, const double *lset_v, int dt, int order,
                                const int32_t *offsets, double *pts) {
  if (!ctx || D < 1 || D > 3 || nel < 0 || !offsets || dt < 0 || dt > 2 || order < 0 ||
      order / 2 + 1 > XG_RULE_NMAX)
    return set_error(XG_ERR_ARG, "xg_cut_rule_fill: bad argument");
  if (nel == 0) return XG_OK;
  if (!el2v || !lset_v || !coords || !pts) return set_error(XG_ERR_ARG, "xg_cut_rule_fill: null pointer");
  const int epw = fill_epw(nel);
  const long long want = ((long long)nel + 4LL * epw - 1) / (4LL * epw);
  const int grid = (int)(want < 65536 ? want : 65536);
  double4 *o = reinterpret_cast<double4 *>(pts);
  switch (D) {
    case 1: k_rule_fill<1><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, coords, lset_v, dt, order, epw, offsets, o); break;
    case 2: k_rule_fill<2><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, coords, lset_v, dt, order, epw, offsets, o); break;
    default: k_rule_fill<3><<<grid, 256, 0, ctx->stream>>>(nel, elems, el2v, coords, lset_v, dt, order, epw, offsets, o); break;
  }
  XG_LAUNCH_CHECK();
  return XG_OK;
}

extern "C" int xg_integrate(xg_ctx *ctx, int D, int nel, const int32_t *elems, const int32_t *el2v,
                            const double *coords, const int32_t *offsets, const double *pts, int nterms,
                            const double *coef, const int32_t *expo, double *per_elem, double *total) {
  if (!ctx || D < 1 || D > 3 || nel < 0 || nterms < 0 || nterms > 32 || (nterms > 0 && (!coef || !expo)))
    return set_error(XG_ERR_ARG, "xg_integrate: bad argument");
  if (total) k_zero_f64<<<1, 1, 0, ctx->stream>>>(total);
  XG_LAUNCH_CHECK();
  if (nel == 0) return XG_OK;
  if (!el2v || !coords || !offsets || !pts) return set_error(XG_ERR_ARG, "xg_integrate: null pointer");
  Poly f;
  f.n = nterms;
  for (int t = 0; t < nterms; ++t) {
    f.c[t] = coef[t];
    for (int d = 0; d < 3; ++d) {
      if (expo[3 * t + d] < 0 || expo[3 * t + d] > 64) return set_error(XG_ERR_ARG, "xg_integrate: bad exponent");
      f.ex[t][d] = expo[3 * t + d];
    }
  }
  // lanes per element: the fewest points that a rule of use has (order 2: 8 on
  // a tetrahedron, 4 on a triangle); a wave for each of few elements, whatever
  // their rules, since the others would be idle.  us, a wave per element and its
  // atomic / these lanes / a wave, tetrahedra: 64 of order 8 10.6 / 18.5 / 10.6, of
  // order 15 19.4 / 55.5 / 12.2, there with 20 terms 80.6 / 207 / 30.8; 2000 of
  // order 4 29.1 / 10.6 / 10.3, of order 15 40.5 / 64.4 / 17.7
  const bool few = nel <= 4096;
  const double4 *p = reinterpret_cast<const double4 *>(pts);
  switch (D) {
    case 1: launch_integrate<1, 2>(ctx, nel, elems, el2v, coords, offsets, p, f, per_elem, total); break;
    case 2:
      if (few) launch_integrate<2, 64>(ctx, nel, elems, el2v, coords, offsets, p, f, per_elem, total);
      else launch_integrate<2, 4>(ctx, nel, elems, el2v, coords, offsets, p, f, per_elem, total);
      break;
    default:
      if (few) launch_integrate<3, 64>(ctx, nel, elems, el2v, coords, offsets, p, f, per_elem, total);
      else launch_integrate<3, 8>(ctx, nel, elems, el2v, coords, offsets, p, f, per_elem, total);
      break;
  }
  XG_LAUNCH_CHECK();
  return XG_OK;
}

extern "C" int xg_integrate_nodes(xg_ctx *ctx, int nel, const int32_t *elems, const int32_t *el2v,
                                  const double *coords, int q, const double *weights, int nterms,
                                  const double *coef, const int32_t *expo, double *per_elem, double *total) {
  if (!ctx || nel < 0 || q != 4 || nterms < 0 || nterms > 32 || (nterms > 0 && (!coef || !expo)))
    return set_error(XG_ERR_ARG, "xg_integrate_nodes: bad argument (q == 4)");
  if (total) XG_CHECK(hipMemsetAsync(total, 0, sizeof(double), ctx->stream));
  if (nel == 0) return XG_OK;
  if (!el2v || !coords || !weights) return set_error(XG_ERR_ARG, "xg_integrate_nodes: null pointer");
  Poly f;
  f.n = nterms;
  for (int t = 0; t < nterms; ++t) {
    f.c[t] = coef[t];
    for (int d = 0; d < 3; ++d) {
      if (expo[3 * t + d] < 0 || expo[3 * t + d] > 64)
        return set_error(XG_ERR_ARG, "xg_integrate_nodes: bad exponent");
      f.ex[t][d] = expo[3 * t + d];
    }
  }
  k_integrate_nodes<4><<<(nel + 255) / 256, 256, 0, ctx->stream>>>(nel, elems, el2v, coords, weights, f, per_elem,
                                                                   total);
  XG_LAUNCH_CHECK();
  return XG_OK;
}
