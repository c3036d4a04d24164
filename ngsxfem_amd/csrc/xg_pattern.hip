// xg_pattern.hip -- sparsity pattern of the global matrix on the device.
//
// NGSolve's BilinearForm::Assemble (the caller of CalcElementMatrix,
// xfem/symboliccutbfi.cpp:37-46) builds the matrix graph from the element
// dof tables before the element matrices are added.  Here the graph is
// built on the GPU, row by row: the elements of every dof are listed (a count
// per dof, a scan, a fill), a wave sorts the columns of a row's elements in
// registers and drops the repeated ones (rows of over 1024 candidates: a block,
// in LDS), and a scan of the row lengths places the rows.  Bound: the rows'
// sorts (a P2 edge row of a tetrahedral mesh has about 60 candidates for 27
// columns).  32^3 cells of 6 tetrahedra, P2 (19.7 M
// couplings, 275,000 rows): graph, matrices and values 2067 -> 368 us against
// the radix sort of all couplings as 64-bit keys (eight passes over 16 B each,
// unique, an atomic count per row), which rows that are long on average
// (rows_path) still take.
#include <algorithm>

#include <hipcub/hipcub.hpp>

#include "xg_internal.hpp"

using namespace xg;

namespace {

// (zero3, nullable: three more words to clear)
__global__ void k_fill_i32(int32_t *p, long long n, int32_t v, int32_t *zero3 = nullptr) {
  const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) p[i] = v;
  if (zero3 && threadIdx.x < 3 && blockIdx.x == 0) zero3[threadIdx.x] = 0;
}

// ---- row by row
// elements per dof, and the place of every table entry among its dof's (in no
// fixed order), so that the fill below needs no atomics of its own.  An atomic
// on a word that others wait for takes 11 ns, 2240 us for one dof that all
// elements of 32^3 cells share: where the wave's elements all have the same dof
// in a column of the table, one lane counts for them.  (step: the bits ndof, 2
// ndof, .. below 64, so step << column are the column's lanes after the first.
// All runs of equal dofs by one atomic each, lane = element: 4.8 -> 8.2 us on a
// discontinuous P2 table of 20^3 cells, whose neighbours in memory were no longer
// counters in one line.)
__global__ __launch_bounds__(256) void k_dof_count(long long m, int ndof, unsigned long long step,
                                                   const int32_t *__restrict__ dofs, int n,
                                                   int32_t *__restrict__ cnt, int32_t *__restrict__ pos, int32_t *err) {
  const long long q = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  const int lane = threadIdx.x & 63;
  const int r = q < m ? dofs[q] : -1;
  // lane = rank ndof + first (half a lane more keeps the quotient off the integers)
  const int rank = (int)(((float)lane + 0.5f) * __builtin_amdgcn_rcpf((float)ndof)), first = lane - rank * ndof;
  const unsigned long long after = step << first;
  const unsigned long long same = __ballot(__shfl_up(r, ndof < 64 ? ndof : 0, 64) == r && rank > 0);
  const bool whole = after != 0ull && (same & after) == after;
  if (r >= n) atomicOr(err, 8);
  const bool valid = r >= 0 && r < n;
  int p = 0;
  if (valid && (!whole || rank == 0)) p = atomicAdd(&cnt[r], whole ? 1 + __popcll(after) : 1);
  const int base = __shfl(p, first, 64);
  if (valid) pos[q] = whole ? base + rank : p;
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

// Rows by the number of their candidates (deg x ndof): up to ROW_SHORT in
// k_row_columns, a wave each with 4 registers or fewer; up to ROW_WAVE in
// k_long_rows, whose registers would cost the short rows their waves; up to
// ROW_SORT, a block each that sorts them in LDS; more (a dof of nearly every
// element: a global multiplier, the hub of a fan), a block for every window of
// ROW_WIN columns that marks the window's columns in a bitmap in LDS.  So every
// row costs about as much per candidate, whatever its length (log^2 in the
// sorts): 32^3 cells of 6 tetrahedra, P2 and one dof more in every element
// (2.2 M candidates in its row): 1446 us, 5340 by the radix sort.
constexpr int ROW_SHORT = 256, ROW_WAVE = 1024;
constexpr int ROW_SORT = 4096;      // (8^3 cells, P1 and one dof in every element: 157 us with the row of 15,360
                                    // candidates sorted, 37 us by a window)
constexpr int ROW_WIN = 1 << 20;    // 128 KB of bits
constexpr int ROW_BLK = 1024;       // threads of a block
constexpr int ROW_BLOCKS = 256;     // blocks of k_long_rows (one in a CU)

// The rows of more than ROW_WAVE candidates: those up to ROW_SORT from the
// front of `rows`, the others from its back; cnt their numbers, cnt[2]: there
// are rows of more than ROW_SHORT.
struct RowList {
  int32_t *rows, *cnt;
  int cap;
};

// the sorted distinct columns of every row at cols[off[r] * ndof ..], their
// number in len[r]; a wave per row
__global__ __launch_bounds__(256) void k_row_columns(int n, int ndof, const int32_t *__restrict__ off,
                                                     const int32_t *__restrict__ adj,
                                                     const int32_t *__restrict__ dofs, int32_t *__restrict__ cols,
                                                     int32_t *__restrict__ len, RowList L) {
  const int lane = threadIdx.x & 63;
  const long long nw = (long long)gridDim.x * 4;
  for (long long r = __builtin_amdgcn_readfirstlane(blockIdx.x * 4 + (threadIdx.x >> 6)); r < n; r += nw) {
    const int o = off[r], deg = off[r + 1] - o;
    const long long c = (long long)deg * ndof;
    if (c > ROW_SHORT) {
      if (lane == 0) L.cnt[2] = 1;
      if (c > ROW_WAVE && lane == 0) {
        const int k = atomicAdd(&L.cnt[c > ROW_SORT], 1);
        L.rows[c > ROW_SORT ? L.cap - 1 - k : k] = (int32_t)r;
      }
      continue;
    }
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

// sum over the ROW_BLK threads of v below this one; total: of all (part: 16 words)
__device__ __forceinline__ int block_prefix(int v, int32_t *part, int &total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int s = 1; s < 64; s <<= 1) {
    const int y = __shfl_up(incl, s, 64);
    if (lane >= s) incl += y;
  }
  __syncthreads();
  if (lane == 63) part[w] = incl;
  __syncthreads();
  int before = 0;
  total = 0;
#pragma unroll
  for (int k = 0; k < ROW_BLK / 64; ++k) {
    const int p = part[k];
    before += k < w ? p : 0;
    total += p;
  }
  return before + incl - v;
}

// a block's row: its candidates sorted in LDS, equal ones dropped
__device__ __forceinline__ void row_sorted(int c, int ndof, const int32_t *__restrict__ adj,
                                           const int32_t *__restrict__ dofs, int n, int32_t *__restrict__ cols,
                                           int32_t *len, int32_t *v, int32_t *part) {
  int m = 2 * ROW_WAVE;
  while (m < c) m <<= 1;
  __syncthreads();  // (the row before)
  for (int q = threadIdx.x; q < m; q += ROW_BLK) {
    int32_t x = NO_COL;
    if (q < c) {
      const unsigned d = (unsigned)q / (unsigned)ndof;
      x = dofs[(size_t)adj[d] * ndof + (q - (int)d * ndof)];
      if (x < 0 || x >= n) x = NO_COL;
    }
    v[q] = x;
  }
  for (int size = 2; size <= m; size <<= 1)
    for (int stride = size >> 1; stride > 0; stride >>= 1) {
      __syncthreads();
      for (int i = threadIdx.x; i < m / 2; i += ROW_BLK) {
        const int a = 2 * i - (i & (stride - 1)), b = a + stride;
        const int32_t x = v[a], y = v[b];
        if ((x > y) == ((a & size) == 0)) {
          v[a] = y;
          v[b] = x;
        }
      }
    }
  __syncthreads();
  int done = 0;
  for (int q0 = 0; q0 < m; q0 += ROW_BLK) {
    const int q = q0 + (int)threadIdx.x;
    const int32_t x = v[q];
    const bool first = x != NO_COL && (q == 0 || v[q - 1] != x);
    int total;
    const int at = block_prefix(first ? 1 : 0, part, total);
    if (first) cols[done + at] = x;
    done += total;
  }
  if (threadIdx.x == 0) *len = done;
}

// a block's window w of a row: marks the columns w ROW_WIN .. in a bitmap in
// LDS and writes them (cols != nullptr) in order; returns their number
__device__ __forceinline__ int row_window(unsigned c, int ndof, const int32_t *__restrict__ adj,
                                          const int32_t *__restrict__ dofs, int n, int w, int32_t *__restrict__ cols,
                                          uint32_t *bits, int32_t *part) {
  const int base = w * ROW_WIN;
  const int words = (min(n - base, ROW_WIN) + 31) / 32;
  __syncthreads();  // (the window before)
  for (int k = threadIdx.x; k < words; k += ROW_BLK) bits[k] = 0u;
  __syncthreads();
  constexpr int U = 8;  // candidates in flight per thread
  for (unsigned q0 = 0; q0 < c; q0 += U * ROW_BLK) {
    int32_t x[U];
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const unsigned q = min(q0 + u * ROW_BLK + threadIdx.x, c - 1);  // (past the end: the last one again)
      const unsigned d = q / (unsigned)ndof;
      x[u] = dofs[(size_t)adj[d] * ndof + (q - d * ndof)];
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
      if (x[u] >= base && x[u] < n && x[u] - base < ROW_WIN)
        atomicOr(&bits[(x[u] - base) >> 5], 1u << (x[u] & 31));
  }
  __syncthreads();
  int done = 0;
  for (int k0 = 0; k0 < words; k0 += ROW_BLK) {
    const int k = k0 + (int)threadIdx.x;
    uint32_t b = k < words ? bits[k] : 0u;
    int total;
    int at = done + block_prefix(__popc(b), part, total);
    if (cols)
      for (; b; b &= b - 1) cols[at++] = base + 32 * k + __builtin_ctz(b);
    done += total;
  }
  return done;
}

// The blocks take the list's rows; then a wave looks through `span` rows and takes
// those of up to ROW_WAVE candidates in turn.  With nwin > 1 windows (of columns) the
// list's longest rows are only counted here, in wcnt, and written by
// k_window_rows.
__global__ __launch_bounds__(ROW_BLK) void k_long_rows(int n, int ndof, const int32_t *__restrict__ off,
                                                       const int32_t *__restrict__ adj,
                                                       const int32_t *__restrict__ dofs, int32_t *__restrict__ cols,
                                                       int32_t *__restrict__ len, RowList L, int span, int nwin,
                                                       int32_t *__restrict__ wcnt) {
  __shared__ int32_t row_lds[ROW_WIN / 32], part[ROW_BLK / 64];
  if (!L.cnt[2]) return;
  const int ns = L.cnt[0];
  for (int k = blockIdx.x; k < ns; k += gridDim.x) {
    const int r = L.rows[k], o = off[r];
    row_sorted((off[r + 1] - o) * ndof, ndof, adj + o, dofs, n, cols + (size_t)o * ndof, len + r, row_lds, part);
  }
  const long long nt = (long long)L.cnt[1] * nwin;
  for (long long t = blockIdx.x; t < nt; t += gridDim.x) {
    const int k = (int)(t / nwin), w = (int)(t - (long long)k * nwin);
    const int r = L.rows[L.cap - 1 - k], o = off[r];
    const int m = row_window((unsigned)(off[r + 1] - o) * ndof, ndof, adj + o, dofs, n, w,
                             nwin == 1 ? cols + (size_t)o * ndof : nullptr, (uint32_t *)row_lds, part);
    if (threadIdx.x == 0) {
      if (nwin == 1) len[r] = m;
      else wcnt[t] = m;
    }
  }
  const int lane = threadIdx.x & 63;
  const long long nw = (long long)gridDim.x * (ROW_BLK / 64);
  for (long long r0 =
           (long long)span * __builtin_amdgcn_readfirstlane(blockIdx.x * (ROW_BLK / 64) + (threadIdx.x >> 6));
       r0 < n; r0 += span * nw) {
    const long long rl = r0 + lane;
    const long long cl = lane < span && rl < n ? (long long)(off[rl + 1] - off[rl]) * ndof : 0;
    for (unsigned long long mk = __ballot(cl > ROW_SHORT && cl <= ROW_WAVE); mk; mk &= mk - 1) {
      const long long r = r0 + __builtin_ctzll(mk);
      const int o = off[r], c = (off[r + 1] - o) * ndof;
      const int32_t *a = adj + o;
      int32_t *out = cols + (size_t)o * ndof;
      const int m = c <= 512 ? row_unique<8>(c, ndof, a, dofs, n, out) : row_unique<16>(c, ndof, a, dofs, n, out);
      if (lane == 0) len[r] = m;
    }
  }
}

// the windows of the list's longest rows, each behind the windows before it
__global__ __launch_bounds__(ROW_BLK) void k_window_rows(int n, int ndof, const int32_t *__restrict__ off,
                                                         const int32_t *__restrict__ adj,
                                                         const int32_t *__restrict__ dofs, int32_t *__restrict__ cols,
                                                         int32_t *__restrict__ len, RowList L, int nwin,
                                                         const int32_t *__restrict__ wcnt) {
  __shared__ int32_t row_lds[ROW_WIN / 32], part[ROW_BLK / 64];
  const long long nt = (long long)L.cnt[1] * nwin;
  for (long long t = blockIdx.x; t < nt; t += gridDim.x) {
    const int k = (int)(t / nwin), w = (int)(t - (long long)k * nwin);
    const int r = L.rows[L.cap - 1 - k], o = off[r];
    int v = 0, before;
    for (int j = threadIdx.x; j < w; j += ROW_BLK) v += wcnt[(long long)k * nwin + j];
    block_prefix(v, part, before);
    const int m = row_window((unsigned)(off[r + 1] - o) * ndof, ndof, adj + o, dofs, n, w,
                             cols + (size_t)o * ndof + before, (uint32_t *)row_lds, part);
    if (w == nwin - 1 && threadIdx.x == 0) len[r] = before + m;
  }
}

// rows to their places; 16 lanes per row, and PLACE_BLOCKS blocks for the rows
// of the list (one each, the longest ones all together)
constexpr int PLACE_BLOCKS = 256;
__global__ __launch_bounds__(256) void k_place_rows(int n, int ndof, const int32_t *__restrict__ off,
                                                    const int32_t *__restrict__ cols,
                                                    const int32_t *__restrict__ row_ptr, int32_t *__restrict__ col_idx,
                                                    long long cap, RowList L, int32_t *__restrict__ nnz,
                                                    int32_t *err) {
  if (blockIdx.x < PLACE_BLOCKS) {
    auto place = [&](int r, int first, int step) {
      const int32_t *src = cols + (size_t)off[r] * ndof;
      const int p0 = row_ptr[r], p1 = row_ptr[r + 1];
      for (long long j = (long long)p0 + first; j < p1; j += step)
        if (j < cap) col_idx[j] = src[j - p0];
    };
    const int ns = L.cnt[0], nh = L.cnt[1];
    for (int k = blockIdx.x; k < ns; k += PLACE_BLOCKS) place(L.rows[k], threadIdx.x, 256);
    for (int k = 0; k < nh; ++k)
      place(L.rows[L.cap - 1 - k], blockIdx.x * 256 + threadIdx.x, PLACE_BLOCKS * 256);
    return;
  }
  const long long g = (long long)(blockIdx.x - PLACE_BLOCKS) * blockDim.x + threadIdx.x;
  if (g == 0) {
    *nnz = row_ptr[n];
    if ((long long)row_ptr[n] > cap) atomicOr(err, 4);
  }
  const long long r = g >> 4;
  if (r >= n) return;
  const int o = off[r];
  if ((long long)(off[r + 1] - o) * ndof > ROW_WAVE) return;
  const int32_t *src = cols + (size_t)o * ndof;
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
    // the list of long rows (the candidates of all rows are at most the
    // couplings), its two counters, the window counts of the longest
    RowList list{nullptr, nullptr, (int)(nent / (ROW_WAVE + 1)) + 1};
    const int nwin = (int)(((long long)n + ROW_WIN - 1) / ROW_WIN);
    const size_t o_list = o_tmp + align256(t_scan), o_lcnt = o_list + align256(sizeof(int32_t) * (size_t)list.cap);
    const size_t o_wcnt = o_lcnt + 256;
    const size_t b_wcnt = nwin > 1 ? sizeof(int32_t) * (size_t)(nent / (ROW_SORT + 1) + 1) * nwin : 0;
    const int rc = ensure_ws(ctx, o_wcnt + b_wcnt);
    if (rc != XG_OK) return rc;
    char *ws = (char *)ctx->ws;
    int32_t *cnt = (int32_t *)ws, *off = (int32_t *)(ws + o_off), *pos = (int32_t *)(ws + o_pos);
    int32_t *adj = (int32_t *)(ws + o_adj), *cols = (int32_t *)(ws + o_col), *wcnt = (int32_t *)(ws + o_wcnt);
    list.rows = (int32_t *)(ws + o_list);
    list.cnt = (int32_t *)(ws + o_lcnt);
    const unsigned g_n = (unsigned)((n1 + 255) / 256), g_m = (unsigned)((m + 255) / 256);
    k_fill_i32<<<g_n, 256, 0, st>>>(cnt, n1, 0, list.cnt);
    unsigned long long step = 0;
    for (int k = ndof; k < 64; k += ndof) step |= 1ull << k;
    k_dof_count<<<g_m, 256, 0, st>>>(m, ndof, step, dofs, n, cnt, pos, ctx->d_err);
    XG_LAUNCH_CHECK();
    XG_CHECK(hipcub::DeviceScan::ExclusiveSum(ws + o_tmp, t_scan, cnt, off, (int)n1, st));
    k_dof_elements<<<g_m, 256, 0, st>>>(m, ndof, dofs, n, off, pos, adj);
    XG_LAUNCH_CHECK();
    // (the counts' buffer takes the row lengths; its last entry stays 0)
    // a wave for each row that may be long, up to ROW_BLOCKS x 16; as many rows
    // for each to look through
    const long long most = nent / (ROW_SHORT + 1) / (ROW_BLK / 64) + 1;
    const unsigned g_long = (unsigned)(most < ROW_BLOCKS ? most : ROW_BLOCKS);
    int span = 1;
    while (span < 64 && (long long)g_long * (ROW_BLK / 64) * span < n) span *= 2;
    const long long want = ((long long)n + 3) / 4;
    k_row_columns<<<(unsigned)(want < 65536 ? want : 65536), 256, 0, st>>>(n, ndof, off, adj, dofs, cols, cnt, list);
    XG_LAUNCH_CHECK();
    k_long_rows<<<g_long, ROW_BLK, 0, st>>>(n, ndof, off, adj, dofs, cols, cnt, list, span, nwin, wcnt);
    XG_LAUNCH_CHECK();
    if (nwin > 1) {
      k_window_rows<<<ROW_BLOCKS, ROW_BLK, 0, st>>>(n, ndof, off, adj, dofs, cols, cnt, list, nwin, wcnt);
      XG_LAUNCH_CHECK();
    }
    XG_CHECK(hipcub::DeviceScan::ExclusiveSum(ws + o_tmp, t_scan, cnt, row_ptr, (int)n1, st));
    const long long thr = (long long)n * 16;
    k_place_rows<<<(unsigned)(PLACE_BLOCKS + (thr + 255) / 256), 256, 0, st>>>(n, ndof, off, cols, row_ptr, col_idx,
                                                                               cap, list, nnz, ctx->d_err);
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
