// xg_pattern.hip -- sparsity pattern of the global matrix on the device.
//
// NGSolve's BilinearForm::Assemble (the caller of CalcElementMatrix,
// xfem/symboliccutbfi.cpp:37-46) builds the matrix graph from the element
// dof tables before the element matrices are added.  Here the graph is
// built on the GPU, row by row: the elements of every dof are listed (a count
// per dof, a scan, a fill), a wave sorts the columns of a row's elements in
// registers and drops the repeated ones, and a scan of the row lengths places
// the rows.  Bound: the rows' sorts (a P2 edge row of a tetrahedral mesh has
// about 60 candidates for 27 columns).  32^3 cells of 6 tetrahedra, P2 (19.7 M
// couplings, 275,000 rows): graph, matrices and values 2067 -> 368 us against
// the radix sort of all couplings as 64-bit keys (eight passes over 16 B each,
// unique, an atomic count per row), which rows that are long on average
// (rows_path) still take.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "xg_internal.hpp"

using namespace xg;

namespace {

__global__ void k_fill_i32(int32_t *p, long long n, int32_t v) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
}

// ---- row by row
// elements per dof, and the place of every table entry among its dof's (in no
// fixed order), so that the fill below needs no atomics of its own
__global__ __launch_bounds__(256) void k_dof_count(long long m, const int32_t *__restrict__ dofs, int n,
                                                   int32_t *__restrict__ cnt, int32_t *__restrict__ pos, int32_t *err) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= m) return;
  const int r = dofs[q];
  if (r >= n) atomicOr(err, 8);
  else if (r >= 0) pos[q] = atomicAdd(&cnt[r], 1);
}

// adj[off[r] ..] = the elements of dof r
__global__ __launch_bounds__(256) void k_dof_elements(long long m, int ndof, const int32_t *__restrict__ dofs, int n,
                                                      const int32_t *__restrict__ off,
                                                      const int32_t *__restrict__ pos, int32_t *__restrict__ adj) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= m) return;
  const int r = dofs[q];
  if (r >= 0 && r < n) adj[off[r] + pos[q]] = (int32_t)(q / ndof);
}

// the value of lane ^ S: cross-lane moves of the vector unit (a shuffle goes
// through the LDS crossbar, about ten times the latency; a row's sort is a
// chain of 21 of them and more)
template <int S>
__device__ __forceinline__ int32_t lane_xor(int32_t v) {
  if constexpr (S == 1) return __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xf, 0xf, true);        // quad_perm 1 0 3 2
  else if constexpr (S == 2) return __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xf, 0xf, true);   // quad_perm 2 3 0 1
  else if constexpr (S == 4) {                                                                 // ^7 then ^3
    const int32_t t = __builtin_amdgcn_update_dpp(0, v, 0x141, 0xf, 0xf, true);
    return __builtin_amdgcn_update_dpp(0, t, 0x1B, 0xf, 0xf, true);
  } else if constexpr (S == 8) return __builtin_amdgcn_update_dpp(0, v, 0x128, 0xf, 0xf, true);  // row_ror 8
  else return __shfl_xor(v, S, 64);
}
template <int S, int K>
__device__ __forceinline__ void lane_stage(int32_t *v, int size, int lane) {
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int32_t o = lane_xor<S>(v[k]);
    const bool up = ((k * 64 + lane) & size) == 0, first = (lane & S) == 0;
    const int32_t lo = min(v[k], o), hi = max(v[k], o);
    v[k] = up == first ? lo : hi;
  }
}

constexpr int32_t NO_COL = 0x7fffffff;  // a skipped column (sorts to the end; n <= 2^31 - 1, so never a dof)

// the candidates of a row, 64 K of them at most, number k * 64 + lane in v[k]:
// bitonic sort (strides of 64 and more between registers, below that between
// lanes), then the first of every run of equal columns to cols[0 ..]; returns
// their number
template <int K>
__device__ __forceinline__ int row_unique(int c, int ndof, const int32_t *__restrict__ adj,
                                          const int32_t *__restrict__ dofs, int n, int32_t *__restrict__ cols) {
  const int lane = threadIdx.x & 63;
  const float rnd = 1.0f / (float)ndof;
  int32_t v[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const int q = k * 64 + lane;
    v[k] = NO_COL;
    if (q < c) {
      int d = (int)((float)q * rnd), t = q - d * ndof;
      if (t >= ndof) ++d, t -= ndof;
      if (t < 0) --d, t += ndof;
      const int32_t x = dofs[(size_t)adj[d] * ndof + t];
      v[k] = (x >= 0 && x < n) ? x : NO_COL;
    }
  }
#pragma unroll
  for (int size = 2; size <= 64 * K; size <<= 1) {
#pragma unroll
    for (int stride = size >> 1; stride >= 64; stride >>= 1) {
      const int sk = stride >> 6;
#pragma unroll
      for (int k = 0; k < K; ++k)
        if ((k & sk) == 0) {
          const bool up = ((k * 64) & size) == 0;
          const int32_t lo = min(v[k], v[k + sk]), hi = max(v[k], v[k + sk]);
          v[k] = up ? lo : hi;
          v[k + sk] = up ? hi : lo;
        }
    }
    if (size > 32) lane_stage<32, K>(v, size, lane);
    if (size > 16) lane_stage<16, K>(v, size, lane);
    if (size > 8) lane_stage<8, K>(v, size, lane);
    if (size > 4) lane_stage<4, K>(v, size, lane);
    if (size > 2) lane_stage<2, K>(v, size, lane);
    lane_stage<1, K>(v, size, lane);
  }
  int m = 0;
  int32_t last = -1;
#pragma unroll
  for (int k = 0; k < K; ++k) {
    int32_t prev = __shfl_up(v[k], 1, 64);
    if (lane == 0) prev = last;
    last = __shfl(v[k], 63, 64);
    const bool first = v[k] != NO_COL && v[k] != prev;
    const unsigned long long b = __ballot(first);
    if (first) cols[m + __popcll(b & ((1ull << lane) - 1ull))] = v[k];
    m += __popcll(b);
  }
  return m;
}

// the sorted distinct columns of every row at cols[off[r] * ndof ..], their
// number in len[r]; a wave per row.  Rows of up to ROW_SHORT candidates here, the
// longer ones in k_long_rows, whose registers would cost these their waves.
constexpr int ROW_SHORT = 256;
__global__ __launch_bounds__(256) void k_row_columns(int n, int ndof, const int32_t *__restrict__ off,
                                                     const int32_t *__restrict__ adj,
                                                     const int32_t *__restrict__ dofs, int32_t *__restrict__ cols,
                                                     int32_t *__restrict__ len) {
  const int lane = threadIdx.x & 63;
  const long long nw = (long long)gridDim.x * 4;
  for (long long r = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); r < n; r += nw) {
    const int o = off[r], deg = off[r + 1] - o;
    const long long c = (long long)deg * ndof;
    if (c > ROW_SHORT) continue;
    const int32_t *a = adj + o;
    int32_t *out = cols + (size_t)o * ndof;
    int m = 0;
    if (c == 0) m = 0;
    else if (c <= 64) m = row_unique<1>((int)c, ndof, a, dofs, n, out);
    else if (c <= 128) m = row_unique<2>((int)c, ndof, a, dofs, n, out);
    else m = row_unique<4>((int)c, ndof, a, dofs, n, out);
    if (lane == 0) len[r] = m;
  }
}

// a wave looks through 64 rows and takes the long ones in turn
__global__ __launch_bounds__(256) void k_long_rows(int n, int ndof, const int32_t *__restrict__ off,
                                                   const int32_t *__restrict__ adj, const int32_t *__restrict__ dofs,
                                                   int32_t *__restrict__ cols, int32_t *__restrict__ len) {
  const int lane = threadIdx.x & 63;
  const long long nw = (long long)gridDim.x * 4;
  for (long long r0 = 64LL * __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); r0 < n;
       r0 += 64 * nw) {
    const long long rl = r0 + lane;
    const bool lng = rl < n && (long long)(off[rl + 1] - off[rl]) * ndof > ROW_SHORT;
    for (unsigned long long mk = __ballot(lng); mk; mk &= mk - 1) {
      const long long r = r0 + __builtin_ctzll(mk);
      const int o = off[r], deg = off[r + 1] - o;
      const long long c = (long long)deg * ndof;
      const int32_t *a = adj + o;
      int32_t *out = cols + (size_t)o * ndof;
      int m = 0;
      if (c <= 512) m = row_unique<8>((int)c, ndof, a, dofs, n, out);
      else if (c <= 1024) m = row_unique<16>((int)c, ndof, a, dofs, n, out);
      else {
        // a few very long rows: the next larger column, one at a time
        for (int32_t last = -1;;) {
          int32_t best = NO_COL;
          for (long long q = lane; q < c; q += 64) {
            const int32_t x = dofs[(size_t)a[q / ndof] * ndof + (int)(q % ndof)];
            if (x > last && x < n && x < best) best = x;
          }
#pragma unroll
          for (int s = 32; s > 0; s >>= 1) best = min(best, __shfl_xor(best, s, 64));
          if (best == NO_COL) break;
          if (lane == 0) out[m] = best;
          ++m;
          last = best;
        }
      }
      if (lane == 0) len[r] = m;
    }
  }
}

// rows to their places; 16 lanes per row
__global__ __launch_bounds__(256) void k_place_rows(int n, int ndof, const int32_t *__restrict__ off,
                                                    const int32_t *__restrict__ cols,
                                                    const int32_t *__restrict__ row_ptr, int32_t *__restrict__ col_idx,
                                                    long long cap, int32_t *__restrict__ nnz, int32_t *err) {
  const long long g = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (g == 0) {
    *nnz = row_ptr[n];
    if ((long long)row_ptr[n] > cap) atomicOr(err, 4);
  }
  const long long r = g >> 4;
  if (r >= n) return;
  const int32_t *src = cols + (size_t)off[r] * ndof;
  const int p0 = row_ptr[r], p1 = row_ptr[r + 1];
  for (int j = p0 + (int)(g & 15); j < p1; j += 16)
    if (j < cap) col_idx[j] = src[j - p0];
}

// Which path: with up to 256 candidates per row on average a wave sorts most
// rows in 4 registers or fewer; a longer row takes more stages for every
// candidate, while the radix sort's cost per coupling stays.
bool rows_path(long long nent, int n) { return nent <= 256LL * n; }

// ---- all couplings sorted as keys row << cb | column, cb the bits of a dof
__global__ __launch_bounds__(256) void k_pair_keys(long long nent, int ndof, const int32_t *__restrict__ dofs, int n,
                                                   int cb, uint64_t *__restrict__ keys, int32_t *err) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (q >= nent) return;
  const int nn = ndof * ndof;
  const long long e = q / nn;
  const int ab = (int)(q - e * nn), a = ab / ndof, b = ab - a * ndof;
  const int r = dofs[e * ndof + a], c = dofs[e * ndof + b];
  if (r >= n || c >= n) atomicOr(err, 8);
  // skipped dofs (< 0) and out-of-range ones sort to the end as all-ones keys
  // (of 2 cb bits; n < 2^cb, so no row has them)
  keys[q] = (r < 0 || c < 0 || r >= n || c >= n) ? (1ull << (2 * cb)) - 1ull
                                                  : ((uint64_t)(uint32_t)r << cb) | (uint32_t)c;
}

// unique keys -> column indices and a count per row; the trailing all-ones
// key (skipped couplings) is not an entry
__global__ __launch_bounds__(256) void k_unpack_keys(const uint64_t *__restrict__ ukeys, const int32_t *__restrict__ nu,
                                                     int cb, int32_t *__restrict__ col_idx, long long cap,
                                                     int32_t *__restrict__ row_cnt, int32_t *__restrict__ nnz,
                                                     int32_t *err) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int cnt = *nu;
  const uint64_t last = cnt > 0 ? ukeys[cnt - 1] : 0ull;
  const int n_ent = (cnt > 0 && last == (1ull << (2 * cb)) - 1ull) ? cnt - 1 : cnt;
  if (i == 0) {
    *nnz = n_ent;
    if ((long long)n_ent > cap) atomicOr(err, 4);
  }
  if (i >= n_ent || i >= cap) return;
  const uint64_t k = ukeys[i];
  col_idx[i] = (int32_t)(k & ((1ull << cb) - 1ull));
  atomicAdd(&row_cnt[(int)(k >> cb)], 1);
}

size_t align256(size_t x) { return (x + 255) & ~size_t(255); }

}  // namespace

extern "C" int xg_csr_pattern(xg_ctx *ctx, int nel, int ndof, const int32_t *dofs, int n, int32_t *row_ptr,
                              int32_t *col_idx, long long cap, int32_t *nnz) {
  if (!ctx || nel < 0 || ndof < 1 || n < 0 || cap < 0) return set_error(XG_ERR_ARG, "xg_csr_pattern: bad argument");
  if (!row_ptr || !nnz || (nel > 0 && (!dofs || (cap > 0 && !col_idx))))
    return set_error(XG_ERR_ARG, "xg_csr_pattern: null pointer");
  const long long nent = (long long)nel * ndof * ndof;
  if (nent > 0x7fffffffLL) return set_error(XG_ERR_ARG, "xg_csr_pattern: more than 2^31 couplings");
  hipStream_t st = ctx->stream;
  if (nent == 0) {
    k_fill_i32<<<(unsigned)(((long long)n + 1 + 255) / 256), 256, 0, st>>>(row_ptr, (long long)n + 1, 0);
    XG_LAUNCH_CHECK();
    k_fill_i32<<<1, 1, 0, st>>>(nnz, 1, 0);
    XG_LAUNCH_CHECK();
    return XG_OK;
  }
  if (rows_path(nent, n) && n < 0x7fffffff) {
    const long long m = (long long)nel * ndof;
    const long long n1 = (long long)n + 1;
    size_t t_scan = 0;
    XG_CHECK(hipcub::DeviceScan::ExclusiveSum(nullptr, t_scan, (int32_t *)nullptr, (int32_t *)nullptr, (int)n1, st));
    // counts (then row lengths), offsets, elements, places, columns
    const size_t b_n = align256(sizeof(int32_t) * (size_t)n1), b_m = align256(sizeof(int32_t) * (size_t)m);
    const size_t o_off = b_n, o_adj = 2 * b_n, o_pos = o_adj + b_m, o_col = o_pos + b_m;
    const size_t o_tmp = o_col + align256(sizeof(int32_t) * (size_t)nent);
    const int rc = ensure_ws(ctx, o_tmp + t_scan);
    if (rc != XG_OK) return rc;
    char *ws = (char *)ctx->ws;
    int32_t *cnt = (int32_t *)ws, *off = (int32_t *)(ws + o_off), *pos = (int32_t *)(ws + o_pos);
    int32_t *adj = (int32_t *)(ws + o_adj), *cols = (int32_t *)(ws + o_col);
    const unsigned g_n = (unsigned)((n1 + 255) / 256), g_m = (unsigned)((m + 255) / 256);
    k_fill_i32<<<g_n, 256, 0, st>>>(cnt, n1, 0);
    k_dof_count<<<g_m, 256, 0, st>>>(m, dofs, n, cnt, pos, ctx->d_err);
    XG_LAUNCH_CHECK();
    XG_CHECK(hipcub::DeviceScan::ExclusiveSum(ws + o_tmp, t_scan, cnt, off, (int)n1, st));
    k_dof_elements<<<g_m, 256, 0, st>>>(m, ndof, dofs, n, off, pos, adj);
    XG_LAUNCH_CHECK();
    // (the counts' buffer takes the row lengths; its last entry stays 0)
    const long long want = ((long long)n + 3) / 4, wl = ((long long)n + 255) / 256;
    if (n > 0) {
      k_row_columns<<<(unsigned)(want < 65536 ? want : 65536), 256, 0, st>>>(n, ndof, off, adj, dofs, cols, cnt);
      k_long_rows<<<(unsigned)(wl < 65536 ? wl : 65536), 256, 0, st>>>(n, ndof, off, adj, dofs, cols, cnt);
    }
    XG_LAUNCH_CHECK();
    XG_CHECK(hipcub::DeviceScan::ExclusiveSum(ws + o_tmp, t_scan, cnt, row_ptr, (int)n1, st));
    const long long thr = (long long)(n > 0 ? n : 1) * 16;
    k_place_rows<<<(unsigned)((thr + 255) / 256), 256, 0, st>>>(n, ndof, off, cols, row_ptr, col_idx, cap, nnz,
                                                                ctx->d_err);
    XG_LAUNCH_CHECK();
    return XG_OK;
  }
  // row counts in row_ptr[1..n] (then scanned in place), row_ptr[0] = 0
  k_fill_i32<<<(unsigned)(((long long)n + 1 + 255) / 256), 256, 0, st>>>(row_ptr, (long long)n + 1, 0);
  XG_LAUNCH_CHECK();
  int cb = 1;
  while (cb < 31 && (n >> cb) != 0) ++cb;  // n < 2^cb
  const int N = (int)nent;
  // workspace: keys, sorted keys, unique count, temp storage of the three
  // hipCUB passes (sort, unique, scan), sized by their dry runs
  size_t t_sort = 0, t_uniq = 0, t_scan = 0;
  XG_CHECK(hipcub::DeviceRadixSort::SortKeys(nullptr, t_sort, (uint64_t *)nullptr, (uint64_t *)nullptr, N, 0, 2 * cb, st));
  XG_CHECK(hipcub::DeviceSelect::Unique(nullptr, t_uniq, (uint64_t *)nullptr, (uint64_t *)nullptr, (int32_t *)nullptr,
                                        N, st));
  XG_CHECK(hipcub::DeviceScan::InclusiveSum(nullptr, t_scan, (int32_t *)nullptr, (int32_t *)nullptr, n, st));
  const size_t tmp = std::max(t_sort, std::max(t_uniq, t_scan));
  const size_t o_a = 0, o_b = align256(sizeof(uint64_t) * (size_t)N), o_n = o_b + align256(sizeof(uint64_t) * (size_t)N);
  const size_t o_t = o_n + 256;
  int rc = ensure_ws(ctx, o_t + tmp);
  if (rc != XG_OK) return rc;
  char *ws = (char *)ctx->ws;
  uint64_t *ka = (uint64_t *)(ws + o_a), *kb = (uint64_t *)(ws + o_b);
  int32_t *nu = (int32_t *)(ws + o_n);
  void *tp = ws + o_t;
  size_t tsz = tmp;
  k_pair_keys<<<(unsigned)((nent + 255) / 256), 256, 0, st>>>(nent, ndof, dofs, n, cb, ka, ctx->d_err);
  XG_LAUNCH_CHECK();
  XG_CHECK(hipcub::DeviceRadixSort::SortKeys(tp, tsz, ka, kb, N, 0, 2 * cb, st));
  tsz = tmp;
  XG_CHECK(hipcub::DeviceSelect::Unique(tp, tsz, kb, ka, nu, N, st));
  k_unpack_keys<<<(unsigned)((nent + 255) / 256), 256, 0, st>>>(ka, nu, cb, col_idx, cap, row_ptr + 1, nnz, ctx->d_err);
  XG_LAUNCH_CHECK();
  // row_ptr[r + 1] = number of entries in rows 0..r (inclusive scan of the
  // counts in place), row_ptr[0] = 0
  tsz = tmp;
  if (n > 0) XG_CHECK(hipcub::DeviceScan::InclusiveSum(tp, tsz, row_ptr + 1, row_ptr + 1, n, st));
  return XG_OK;
}
