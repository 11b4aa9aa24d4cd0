// ILU(k) / IC(k) numeric factorisation on the device.
//
// The symbolic phase stays on the host (iluk_symbolic / icc_symbolic, bit-
// exact with the reference); the numeric phase runs on gfx950 with the
// reference's arithmetic in the reference's order, so the factor is bitwise
// the host's:
//  * ILU (mkl_wrapper/incomplete_lu.cpp:277-325, row IKJ): for each row i,
//    for each k < i in the row's pattern in ascending order,
//    l_ik = a_ik / u_kk, then a_ij -= l_ik * u_kj for every j > k of row k's
//    upper part that is in row i's pattern.
//  * IC (sparse_mat_op/precond.hpp:615-693, up-looking on the upper
//    pattern): the diagonal is scaled by (1 + omega); for each row k with an
//    entry in column j, in the reference's linked-list order (recorded on
//    the host once per pattern), u_j* -= u_kj * u_k* over the merged
//    columns; then u_jj = sqrt(pivot) and the row is divided by it; a
//    pivot < 0 fails.
//  * IC with the additive shift (mkl_wrapper/incomplete_cholesky.cpp:
//    195-274, incomplete_cholesky_k): the same updates with the shift added
//    to the diagonal, the rows k of each column taken first-in first-out
//    (that class's column vectors), and a pivot <= 0 failing.
// Products and differences are rounded separately (no fused multiply-add),
// as in the reference's x86-64 build.
//
// Rows of at most 64 entries (and eliminations): one launch, sync-free
// (k_factor_rows). Longer rows, and few levels of very many rows (see
// factor_one_launch): level by level (one launch per level of the factorisation's dependency DAG, which is the lower triangular solve's), one
// 64-lane workgroup per row with the row's columns and values in LDS; for
// each eliminating row k the lanes take k's entries, find their column in the
// row by binary search and update it. A row longer than kRowCap is done by
// one lane in global memory, in the host's loop order.
#include <algorithm>
#include <climits>
#include <cmath>

#include "dev_util.hpp"
#include "device.hpp"
#include "host_algos.hpp"

// every product and difference in this file rounds on its own (the
// library's rounding intrinsics do not stop the fusion once inlined; the
// pragma on plain operators does)
#pragma clang fp contract(off)

namespace laamd {
using namespace dev;

struct NumericPlan {
  bool ic = false;
  int n = 0;
  int64_t nnzA = 0, nnzF = 0;
  double omega = 0.0;
  bool additive = false;   // IC: incomplete_cholesky_k's arithmetic, omega = the shift
  DevBuf fai, faj, fu;     // pattern (0-based); ILU: first upper position per row
  DevBuf a2f;              // per entry of A: its position in the factor, or -1
  DevBuf fav, diag;        // factor values; ILU: u_ii per row
  DevBuf rows;             // rows in dependency-level order
  std::vector<int> level_ptr;
  DevBuf pptr, pk, pq;     // IC: per row j the (k, q) eliminations, host order
  DevBuf err;              // row + 1 of a failed pivot, else 0; a wait that ran out
  // the sync-free form: lanes per row (0: not used), chunks of rows that
  // never span a level, per factor entry its entry of A or -1, per row the
  // diagonal's position (ILU), the ticket counter
  int lanes = 0, nchunks = 0;
  DevBuf chunk_start, f2a, dpos, ticket;
  std::vector<int> h_fai, h_faj;
};
void NumericPlanDeleter::operator()(NumericPlan *p) const { delete p; }

namespace {
constexpr int kRowCap = 512;

__global__ void k_scatter(int64_t m, const int64_t *__restrict__ a2f,
                          const double *__restrict__ av, double *fav) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  if (t < m) {
    const int64_t p = a2f[t];
    if (p >= 0) fav[p] = av[t];
  }
}

__global__ void k_scale_first(int n, const int *__restrict__ fai, double *fav, double f) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n && fai[j + 1] > fai[j]) fav[fai[j]] = fav[fai[j]] * f;
}
__global__ void k_shift_first(int n, const int *__restrict__ fai, double *fav, double a) {
  const int j = blockIdx.x * blockDim.x + threadIdx.x;
  if (j < n && fai[j + 1] > fai[j]) fav[fai[j]] = fav[fai[j]] + a;
}

__global__ void k_fill_zero(int64_t m, double *v) {
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < m;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    v[t] = 0.0;
}

__device__ __forceinline__ int find_col(const int *cols, int lo, int hi, int c) {
  while (lo < hi) {
    const int mid = (lo + hi) >> 1;
    if (cols[mid] < c) lo = mid + 1;
    else hi = mid;
  }
  return lo;
}

__device__ __forceinline__ void flag_row(int *err, int row) {
  atomicCAS(err, 0, row + 1);
}

// one row of ILU by one lane, in global memory (rows longer than kRowCap)
__device__ void ilu_row_serial(int i, const int *fai, const int *faj, const int *fu, double *fav,
                               double *diag, int *err) {
  const int fb = fai[i], fe = fai[i + 1];
  int t = fb;
  for (; t < fe && faj[t] != i; ++t) {
    const int k = faj[t];
    fav[t] = fav[t] / diag[k];
    const double lik = fav[t];
    int p = t, q = fu[k];
    const int qe = fai[k + 1];
    while (q != qe && p != fe) {
      if (faj[p] == faj[q]) {
        fav[p] = fav[p] - lik * fav[q];
        ++p;
        ++q;
      } else if (faj[p] < faj[q]) {
        ++p;
      } else {
        ++q;
      }
    }
  }
  if (t == fe) flag_row(err, i);
  else diag[i] = fav[t];
}

__global__ __launch_bounds__(64) void k_ilu_rows(int k0, const int *__restrict__ rows,
                                                 const int *__restrict__ fai,
                                                 const int *__restrict__ faj,
                                                 const int *__restrict__ fu, double *fav,
                                                 double *diag, int *err) {
  __shared__ int cols[kRowCap];
  __shared__ double vals[kRowCap];
  const int i = rows[k0 + blockIdx.x];
  const int lane = threadIdx.x;
  const int fb = fai[i], len = fai[i + 1] - fb;
  if (len > kRowCap) {
    if (lane == 0) ilu_row_serial(i, fai, faj, fu, fav, diag, err);
    return;
  }
  for (int t = lane; t < len; t += 64) {
    cols[t] = faj[fb + t];
    vals[t] = fav[fb + t];
  }
  __syncthreads();
  int t = 0;
  for (; t < len && cols[t] != i; ++t) {
    const int k = cols[t];
    if (lane == 0) vals[t] = vals[t] / diag[k];
    __syncthreads();
    const double lik = vals[t];
    const int qe = fai[k + 1];
    for (int q = fu[k] + lane; q < qe; q += 64) {
      const int c = faj[q];
      const int p = find_col(cols, t + 1, len, c);
      if (p < len && cols[p] == c) vals[p] = vals[p] - lik * fav[q];
    }
    __syncthreads();
  }
  if (lane == 0) {
    if (t == len) flag_row(err, i);
    else diag[i] = vals[t];
  }
  for (int u = lane; u < len; u += 64) fav[fb + u] = vals[u];
}

// one row of IC by one lane, in global memory
// (strict: a zero pivot fails too)
__device__ void ic_row_serial(int j, const int *fai, const int *faj, const int *pptr,
                              const int *pk, const int *pq, double *fav, int *err, int strict) {
  const int ps = fai[j], pe = fai[j + 1];
  for (int e = pptr[j]; e < pptr[j + 1]; ++e) {
    const int k = pk[e];
    int q = pq[e];
    const int qe = fai[k + 1];
    const double ukj = fav[q];
    int t = ps;
    while (q < qe && t < pe) {
      if (faj[q] == faj[t]) {
        fav[t] = fav[t] - ukj * fav[q];
        ++t;
        ++q;
      } else if (faj[q] < faj[t]) {
        ++q;
      } else {
        ++t;
      }
    }
  }
  if (strict ? fav[ps] <= 0 : fav[ps] < 0) {
    flag_row(err, j);
    return;
  }
  const double d = sqrt(fav[ps]);
  fav[ps] = d;
  for (int t = ps + 1; t < pe; ++t) fav[t] = fav[t] / d;
}

__global__ __launch_bounds__(64) void k_ic_rows(int k0, const int *__restrict__ rows,
                                                const int *__restrict__ fai,
                                                const int *__restrict__ faj,
                                                const int *__restrict__ pptr,
                                                const int *__restrict__ pk,
                                                const int *__restrict__ pq, double *fav,
                                                int *err, int strict) {
  __shared__ int cols[kRowCap];
  __shared__ double vals[kRowCap];
  const int j = rows[k0 + blockIdx.x];
  const int lane = threadIdx.x;
  const int ps = fai[j], len = fai[j + 1] - ps;
  if (len > kRowCap) {
    if (lane == 0) ic_row_serial(j, fai, faj, pptr, pk, pq, fav, err, strict);
    return;
  }
  for (int t = lane; t < len; t += 64) {
    cols[t] = faj[ps + t];
    vals[t] = fav[ps + t];
  }
  __syncthreads();
  for (int e = pptr[j]; e < pptr[j + 1]; ++e) {
    const int k = pk[e], q0 = pq[e], qe = fai[k + 1];
    const double ukj = fav[q0];
    for (int q = q0 + lane; q < qe; q += 64) {
      const int c = faj[q];
      const int t = find_col(cols, 0, len, c);
      if (t < len && cols[t] == c) vals[t] = vals[t] - ukj * fav[q];
    }
    __syncthreads();
  }
  const double piv = vals[0];
  if (strict ? piv <= 0 : piv < 0) {
    if (lane == 0) flag_row(err, j);
    return;
  }
  const double d = sqrt(piv);
  for (int u = lane; u < len; u += 64) fav[ps + u] = u == 0 ? d : vals[u] / d;
}

// ---------------------------------------------------------------- sync-free
// One launch for the whole factorisation: a wavefront takes 64 / G rows, G
// lanes each, one entry per lane, and keeps them in registers. Everything
// that depends on the pattern alone is done first (the row's columns, where
// each eliminating row's entries fall in it, by binary search in LDS); then
// the values of the eliminating rows are polled as they appear (a value that
// is no longer the sentinel is final: agent-scope relaxed loads and stores,
// as in the sync-free solves) and applied in the host's order. Workgroups
// claim chunks of rows in level order, so every wait is on a row of an
// earlier ticket or a smaller level, which a running wavefront holds.
// What bounds it is the chain of rows: per level one store-to-poll hop and
// the divisions of the row's last eliminations. One launch per level with a
// row's three dependent loads per elimination in the loop, against this
// form: 27-point ILU(1) on 48^3 (612 levels, rows of up to 61 entries)
// 20.8 -> 2.2 ms, ILU(0) 5.45 -> 1.15 ms; 72^3 IC(0) 1.55 -> 0.48 ms; 128^2
// IC(0) (255 levels) 1.18 -> 0.36 ms (with the refreshed solve plans).
constexpr int kFacWaves = 4;
constexpr int kFacMaxLanes = 64;
constexpr uint64_t kFacWaitTicks = 20000000;  // 0.2 s of the 100 MHz clock

template <int G>
__device__ __forceinline__ int row_bcast(int v, int l) {
  if constexpr (G == 64) return __builtin_amdgcn_readlane(v, l);
  else return __shfl(v, l, G);
}
template <int G>
__device__ __forceinline__ double row_bcast(double v, int l) {
  const long long b = __double_as_longlong(v);
  const int lo = row_bcast<G>(static_cast<int>(b), l);
  const int hi = row_bcast<G>(static_cast<int>(b >> 32), l);
  return __longlong_as_double((static_cast<long long>(hi) << 32) | static_cast<unsigned int>(lo));
}

// src: ILU the diagonals' positions, IC the rows' elimination lists (pptr,
// with pk and pq)
template <int G, bool IC>
__global__ __launch_bounds__(64 * kFacWaves) void k_factor_rows(
    int nchunks, const int *__restrict__ chunk_start, const int *__restrict__ rows,
    const int *__restrict__ fai, const int *__restrict__ faj, const int *__restrict__ src,
    const int *__restrict__ pk, const int *__restrict__ pq, const int *__restrict__ f2a,
    const double *__restrict__ av, double *fav, double diag_mul, double diag_add, int strict,
    unsigned *ticket, int *err) {
  constexpr int B = G < 8 ? G : 8;  // eliminations whose loads are in flight together
  __shared__ int s_cols[kFacWaves][64];
  __shared__ uint8_t s_map[kFacWaves][G * 64];
  __shared__ int s_c[2];
  const int wave = static_cast<int>(threadIdx.x) >> 6, lane = threadIdx.x & 63;
  const int sub = lane & (G - 1), row0 = lane - sub;  // lane in the row, the row's first lane
  int *const cols = s_cols[wave];
  uint8_t *const map = s_map[wave];
  if (threadIdx.x == 0) s_c[0] = static_cast<int>(atomicAdd(ticket, 1u));
  __syncthreads();
  for (int it = 0;; ++it) {
    const int c = __builtin_amdgcn_readfirstlane(s_c[it & 1]);
    if (c >= nchunks) break;
    if (threadIdx.x == 0) s_c[(it + 1) & 1] = static_cast<int>(atomicAdd(ticket, 1u));
    const int k = chunk_start[c] + (wave * 64 + lane) / G;
    const bool on = k < chunk_start[c + 1];
    if (__ballot(on)) {
      const int i = on ? rows[k] : 0;
      const int fb = on ? fai[i] : 0, len = on ? fai[i + 1] - fb : 0;
      const bool mine = sub < len;
      const int col = mine ? faj[fb + sub] : INT_MAX;
      const int a = mine ? f2a[fb + sub] : -1;
      double val = a >= 0 ? av[a] : 0.0;
      cols[lane] = col;
      // eliminations e: entries start .. start + cnt of the factor, the first
      // of them the pivot (ILU) or this row's multiplier (IC)
      int ne, start = 0, cnt = 0;
      if constexpr (IC) {
        if (sub == 0) val = diag_add != 0.0 ? val + diag_add : val * diag_mul;
        const int e0 = on ? src[i] : 0;
        ne = on ? src[i + 1] - e0 : 0;
        if (sub < ne) {
          start = pq[e0 + sub];
          cnt = fai[pk[e0 + sub] + 1] - start;
        }
      } else {
        const uint64_t low = __ballot(mine && col < i);
        ne = G == 64 ? __popcll(low)
                     : __popcll((low >> row0) & ((1ull << (G & 63)) - 1ull));
        if (sub < ne) {
          start = src[col];
          cnt = fai[col + 1] - start;
        }
      }
      int nmax = ne;  // over the wavefront's rows
      if constexpr (G < 64) {
#pragma unroll
        for (int d = G; d < 64; d <<= 1) nmax = max(nmax, __shfl_xor(nmax, d, 64));
      }
      nmax = __builtin_amdgcn_readfirstlane(nmax);
      // where the eliminating rows' entries fall: map[e][lane] = the entry
      // that updates this lane's, 0xFF for none
      for (int e = 0; e < nmax; ++e) map[e * 64 + lane] = 0xFF;
      for (int e0 = 0; e0 < nmax; e0 += B) {
        int cc[B], pos[B];
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const int es = e0 + u < nmax ? e0 + u : nmax - 1;
          const int st = row_bcast<G>(start, es), m = row_bcast<G>(cnt, es);
          const bool in = e0 + u < ne && sub < m && (IC || sub > 0);
          cc[u] = in ? faj[st + sub] : -1;
          pos[u] = row0;
        }
#pragma unroll
        for (int d = G / 2; d >= 1; d >>= 1)
#pragma unroll
          for (int u = 0; u < B; ++u)
            if (cols[pos[u] + d - 1] < cc[u]) pos[u] += d;
#pragma unroll
        for (int u = 0; u < B; ++u)
          if (cc[u] >= 0 && cols[pos[u]] == cc[u])
            map[(e0 + u) * 64 + pos[u]] = static_cast<uint8_t>(sub);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "workgroup", "local");
      double v[B], vn[B];
      int at[B], an[B];  // -1: no such elimination in this lane's row
      bool hit[B], hn[B];
      auto fetch = [&](int e0, double(&w)[B], int(&p)[B], bool(&h)[B]) {
#pragma unroll
        for (int u = 0; u < B; ++u) {
          p[u] = -1;
          h[u] = false;
          w[u] = 0.0;
          if (e0 + u < nmax) {
            const int st = row_bcast<G>(start, e0 + u);
            const int q = map[(e0 + u) * 64 + lane];
            h[u] = q != 0xFF && e0 + u < ne;
            if (e0 + u < ne) {
              p[u] = st + (h[u] ? q : 0);
              w[u] = load_ready(fav + p[u]);
            }
          }
        }
      };
      if (nmax > 0) fetch(0, v, at, hit);
      for (int e0 = 0; e0 < nmax; e0 += B) {
        fetch(e0 + B, vn, an, hn);
        const uint64_t t0 = __builtin_amdgcn_s_memrealtime();
        for (unsigned polls = 1;; ++polls) {
          bool wait = false;
#pragma unroll
          for (int u = 0; u < B; ++u) wait |= at[u] >= 0 && is_sentinel(v[u]);
          if (!__ballot(wait)) break;
          __builtin_amdgcn_s_sleep(1);
          if ((polls & 255u) == 0 &&
              (__hip_atomic_load(err + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0 ||
               __builtin_amdgcn_s_memrealtime() - t0 > kFacWaitTicks)) {
            __hip_atomic_fetch_or(err + 1, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            break;
          }
#pragma unroll
          for (int u = 0; u < B; ++u)
            if (at[u] >= 0 && is_sentinel(v[u])) v[u] = load_ready(fav + at[u]);
#pragma unroll
          for (int u = 0; u < B; ++u)
            if (an[u] >= 0 && is_sentinel(vn[u])) vn[u] = load_ready(fav + an[u]);
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
          const int e = e0 + u;
          if (e >= nmax) break;
          if constexpr (IC) {
            const double ukj = row_bcast<G>(v[u], 0);
            if (hit[u]) val = val - ukj * v[u];
          } else {
            // (the lane of column k holds the pivot: nothing updates it)
            const double l = row_bcast<G>(val, e) / row_bcast<G>(v[u], e);
            if (hit[u]) val = val - l * v[u];
            if (sub == e && e < ne) val = l;
          }
        }
#pragma unroll
        for (int u = 0; u < B; ++u) {
          v[u] = vn[u];
          at[u] = an[u];
          hit[u] = hn[u];
        }
      }
      if constexpr (IC) {
        const double piv = row_bcast<G>(val, 0);
        if (sub == 0 && on && (strict ? piv <= 0 : piv < 0)) flag_row(err, i);
        const double d = sqrt(piv);
        val = sub == 0 ? d : val / d;
      }
      if (mine) {
        unsigned long long o = to_bits<double>(val);
        if (o == Sentinel<double>::bits) o = Sentinel<double>::qnan;
        store_ready(fav + fb + sub, from_bits<double>(o));
      }
    }
    __syncthreads();
  }
}

// every factor value <- sentinel
__global__ void k_factor_mark(int64_t m, double *v) {
  for (int64_t t = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x; t < m;
       t += static_cast<int64_t>(gridDim.x) * blockDim.x)
    v[t] = from_bits<double>(Sentinel<double>::bits);
}

template <typename T>
void upload_vec(DevBuf &b, const std::vector<T> &v, hipStream_t s) {
  b.alloc(sizeof(T) * std::max<size_t>(v.size(), 1));
  if (!v.empty()) b.upload(v.data(), sizeof(T) * v.size(), s);
}

// strict lower (cols < row) or upper (cols > row) part of a 0-based pattern,
// with each entry's position in the pattern
void strict_part(int n, const std::vector<int> &pi, const std::vector<int> &pj, bool upper,
                 std::vector<int> &ti, std::vector<int> &tj, std::vector<int64_t> &src) {
  ti.assign(static_cast<size_t>(n) + 1, 0);
  tj.clear();
  src.clear();
  for (int i = 0; i < n; ++i) {
    for (int p = pi[i]; p < pi[i + 1]; ++p) {
      const int c = pj[p];
      if (upper ? c > i : c < i) {
        tj.push_back(c);
        src.push_back(p);
      }
    }
    ti[i + 1] = static_cast<int>(tj.size());
  }
}

// per entry of A (0-based CSR): position of its column in the factor row,
// or -1 when the entry is not part of the factor (IC: below the diagonal)
std::vector<int64_t> map_a_to_f(int n, const int *ai, const int *aj, int base,
                                const std::vector<int> &fi, const std::vector<int> &fj,
                                bool upper_only) {
  const int64_t nnz = static_cast<int64_t>(ai[n]) - base;
  std::vector<int64_t> m(static_cast<size_t>(nnz), -1);
  for (int i = 0; i < n; ++i) {
    int p = fi[i];
    for (int64_t a = ai[i] - base; a < ai[i + 1] - base; ++a) {
      const int c = aj[a] - base;
      if (upper_only && c < i) continue;
      while (p < fi[i + 1] && fj[p] < c) ++p;
      LA_CHECK_ARG(p < fi[i + 1] && fj[p] == c, "matrix entry outside the factor's pattern");
      m[a] = p;
    }
  }
  return m;
}

void finish_plans(Prec &P, NumericPlan &N, const std::vector<int> &Li, const std::vector<int> &Lj,
                  const std::vector<int64_t> &Ls, const std::vector<int64_t> *Ld,
                  const std::vector<int> &Ui, const std::vector<int> &Uj,
                  const std::vector<int64_t> &Us, const std::vector<int64_t> &Ud, hipStream_t s) {
  const int n = N.n;
  std::vector<double> zl(std::max<size_t>(Lj.size(), 1), 0.0), zu(std::max<size_t>(Uj.size(), 1), 0.0),
      ones(static_cast<size_t>(std::max(n, 1)), 1.0);
  P.lower = make_trsv(n, 0, Li.data(), Lj.data(), zl.data(), Ld ? ones.data() : nullptr, false, s);
  P.upper = make_trsv(n, 0, Ui.data(), Uj.data(), zu.data(), ones.data(), true, s);
  trsv_set_sources(*P.lower, Ls.data(), Ld ? Ld->data() : nullptr, s);
  trsv_set_sources(*P.upper, Us.data(), Ud.data(), s);
  // the factorisation's dependency levels are the lower solve's
  upload_vec(N.rows, P.lower->h_perm, s);
  N.level_ptr = P.lower->level_ptr;
  N.fav.alloc(sizeof(double) * static_cast<size_t>(std::max<int64_t>(N.nnzF, 1)));
  N.err.alloc(sizeof(int) * 4);
  P.tmp[0].alloc(sizeof(double) * std::max(n, 1));
  P.tmp[1].alloc(sizeof(float) * std::max(n, 1));
  LA_HIP(hipStreamSynchronize(s));
}
// The sync-free form applies when a row and its eliminations fit a wavefront
// and it is the faster one: the fewest lanes per row that hold both (at least
// 4).
void plan_sync_free(NumericPlan &N, const std::vector<int> &fai, const std::vector<int64_t> &a2f,
                    int max_elim, int64_t eliminations, const std::vector<int> &dpos,
                    hipStream_t s) {
  int longest = max_elim;
  for (int i = 0; i < N.n; ++i) longest = std::max(longest, fai[i + 1] - fai[i]);
  if (longest > kFacMaxLanes || N.nnzA >= INT32_MAX) return;
  int lanes = 4;
  while (lanes < longest) lanes *= 2;
  const int levels = std::max<int>(1, static_cast<int>(N.level_ptr.size()) - 1);
  if (!factor_one_launch(N.n, levels, lanes, eliminations)) return;
  N.lanes = lanes;
  std::vector<int> f2a(static_cast<size_t>(N.nnzF), -1), chunks;
  for (size_t a = 0; a < a2f.size(); ++a)
    if (a2f[a] >= 0) f2a[a2f[a]] = static_cast<int>(a);
  const int per = kFacWaves * 64 / N.lanes;
  for (size_t l = 0; l + 1 < N.level_ptr.size(); ++l)
    for (int k = N.level_ptr[l]; k < N.level_ptr[l + 1]; k += per) {
      chunks.push_back(k);
    }
  N.nchunks = static_cast<int>(chunks.size());
  // a chunk ends where the next one starts: the last one of a level at the
  // level's end, which is the next level's start
  chunks.push_back(N.n);
  upload_vec(N.chunk_start, chunks, s);
  upload_vec(N.f2a, f2a, s);
  upload_vec(N.dpos, dpos, s);
  N.ticket.alloc(sizeof(unsigned) * 4);
  LA_HIP(hipStreamSynchronize(s));
}
}  // namespace

std::unique_ptr<Prec> make_prec_ilu_gpu(int n, int base, const int *ai, const int *aj, int level,
                                        hipStream_t s) {
  LA_CHECK_ARG(n >= 0 && level >= 0, "bad size or level");
  auto P = std::make_unique<Prec>();
  P->n = n;
  P->stream = s;
  P->num.reset(new NumericPlan());
  NumericPlan &N = *P->num;
  N.n = n;
  std::vector<int> fai, faj, fu;
  iluk_symbolic(n, base, ai, aj, level, fai, faj, fu);
  for (auto &v : fai) v -= base;
  for (auto &v : faj) v -= base;
  N.nnzF = fai[n];
  N.nnzA = static_cast<int64_t>(ai[n]) - base;
  // diagonal positions; ILU needs every one
  std::vector<int64_t> dpos(static_cast<size_t>(n));
  for (int i = 0; i < n; ++i) {
    int p = fai[i];
    while (p < fai[i + 1] && faj[p] != i) ++p;
    if (p == fai[i + 1]) throw la_error(LA_ERR_NUMERIC, "ILU pattern has a row without a diagonal");
    dpos[i] = p;
  }
  std::vector<int64_t> a2f = map_a_to_f(n, ai, aj, base, fai, faj, false);
  std::vector<int> Li, Lj, Ui, Uj;
  std::vector<int64_t> Ls, Us;
  strict_part(n, fai, faj, false, Li, Lj, Ls);
  strict_part(n, fai, faj, true, Ui, Uj, Us);
  upload_vec(N.fai, fai, s);
  upload_vec(N.faj, faj, s);
  upload_vec(N.fu, fu, s);
  upload_vec(N.a2f, a2f, s);
  N.diag.alloc(sizeof(double) * std::max(n, 1));
  finish_plans(*P, N, Li, Lj, Ls, nullptr, Ui, Uj, Us, dpos, s);
  plan_sync_free(N, fai, a2f, 0, static_cast<int64_t>(Lj.size()),
                 std::vector<int>(dpos.begin(), dpos.end()), s);
  N.h_fai = std::move(fai);
  N.h_faj = std::move(faj);
  return P;
}

std::unique_ptr<Prec> make_prec_ic_gpu(int n, int base, const int *ai, const int *aj, int level,
                                       double omega, hipStream_t s, bool additive) {
  LA_CHECK_ARG(n >= 0 && level >= 0, "bad size or level");
  auto P = std::make_unique<Prec>();
  P->ic = true;
  P->n = n;
  P->stream = s;
  P->num.reset(new NumericPlan());
  NumericPlan &N = *P->num;
  N.ic = true;
  N.n = n;
  N.omega = omega;
  N.additive = additive;
  N.nnzA = static_cast<int64_t>(ai[n]) - base;
  // upper part of A with the diagonal first in each row
  std::vector<int> ui(static_cast<size_t>(n) + 1, 0), uj, dpos(static_cast<size_t>(n));
  for (int i = 0; i < n; ++i) {
    bool has_diag = false;
    for (int64_t a = ai[i] - base; a < ai[i + 1] - base; ++a) {
      const int c = aj[a] - base;
      if (c < i) continue;
      if (c == i) {
        has_diag = true;
        dpos[i] = static_cast<int>(uj.size());
      }
      uj.push_back(c);
    }
    if (!has_diag || uj[dpos[i]] != i || dpos[i] != ui[i])
      throw la_error(LA_ERR_NUMERIC, "IC needs every diagonal entry (sorted rows)");
    ui[i + 1] = static_cast<int>(uj.size());
  }
  std::vector<int> fai, faj;
  icc_symbolic(n, 0, ui.data(), uj.data(), dpos.data(), level, fai, faj);
  N.nnzF = fai[n];
  std::vector<int64_t> a2f = map_a_to_f(n, ai, aj, base, fai, faj, true);
  // the reference's elimination order per row: icc_numeric's list walk
  // (last-in first-out) or ick_numeric's column queues (first-in first-out)
  std::vector<int> pptr(static_cast<size_t>(n) + 1, 0), pk, pq;
  if (!additive) {
    const int NONE = INT_MAX;
    std::vector<int> llist(static_cast<size_t>(n), NONE);
    std::vector<int64_t> jk(static_cast<size_t>(n), 0);
    for (int j = 0; j < n; ++j) {
      const int64_t ps = fai[j], pe = fai[j + 1];
      for (int k = llist[j]; k < j;) {
        const int64_t q = jk[k]++;
        const int64_t qe = fai[k + 1];
        const int knext = llist[k];
        if (q + 1 < qe) {
          const int c = faj[q + 1];
          llist[k] = llist[c];
          llist[c] = k;
        }
        pk.push_back(k);
        pq.push_back(static_cast<int>(q));
        k = knext;
      }
      if (pe - ps > 1) {
        const int c = faj[ps + 1];
        llist[j] = llist[c];
        llist[c] = j;
        jk[j] = ps + 1;
      }
      pptr[j + 1] = static_cast<int>(pk.size());
    }
  } else {
    const int NONE = -1;
    std::vector<int> head(static_cast<size_t>(n), NONE), tail(static_cast<size_t>(n), NONE),
        next(static_cast<size_t>(n), NONE);
    std::vector<int64_t> pos(static_cast<size_t>(n), 0);
    auto enqueue = [&](int k, int c) {
      next[k] = NONE;
      if (head[c] == NONE) head[c] = k;
      else next[tail[c]] = k;
      tail[c] = k;
    };
    for (int j = 0; j < n; ++j) {
      const int64_t ps = fai[j], pe = fai[j + 1];
      for (int k = head[j]; k != NONE;) {
        const int knext = next[k];
        const int64_t q = pos[k];
        if (q + 1 < fai[k + 1]) {
          pos[k] = q + 1;
          enqueue(k, faj[q + 1]);
        }
        pk.push_back(k);
        pq.push_back(static_cast<int>(q));
        k = knext;
      }
      head[j] = NONE;
      if (pe - ps > 1) {
        pos[j] = ps + 1;
        enqueue(j, faj[ps + 1]);
      }
      pptr[j + 1] = static_cast<int>(pk.size());
    }
  }
  // solves: upper = strict upper of R with its diagonal, lower = its transpose
  std::vector<int> Ui, Uj;
  std::vector<int64_t> Us, dsrc(static_cast<size_t>(n));
  strict_part(n, fai, faj, true, Ui, Uj, Us);
  for (int j = 0; j < n; ++j) dsrc[j] = fai[j];
  std::vector<int> Li(static_cast<size_t>(n) + 1), Lj(Uj.size());
  std::vector<double> uv(Us.begin(), Us.end()), lv(Uj.size());
  transpose(n, n, 0, Ui.data(), Uj.data(), uv.data(), Li.data(), Lj.data(), lv.data());
  std::vector<int64_t> Ls(lv.begin(), lv.end());
  upload_vec(N.fai, fai, s);
  upload_vec(N.faj, faj, s);
  upload_vec(N.a2f, a2f, s);
  upload_vec(N.pptr, pptr, s);
  upload_vec(N.pk, pk, s);
  upload_vec(N.pq, pq, s);
  finish_plans(*P, N, Li, Lj, Ls, &dsrc, Ui, Uj, Us, dsrc, s);
  int max_elim = 0;
  for (int j = 0; j < n; ++j) max_elim = std::max(max_elim, pptr[j + 1] - pptr[j]);
  plan_sync_free(N, fai, a2f, max_elim, static_cast<int64_t>(pk.size()), {}, s);
  N.h_fai = std::move(fai);
  N.h_faj = std::move(faj);
  return P;
}

namespace {
void factor_rows(NumericPlan &N, const double *a_vals, hipStream_t s) {
  double *fav = N.fav.as<double>();
  LA_HIP(hipMemsetAsync(N.ticket.p, 0, sizeof(unsigned) * 4, s));
  hipLaunchKernelGGL(k_factor_mark, dim3(2048), dim3(256), 0, s, N.nnzF, fav);
  LA_HIP(hipGetLastError());
  const int levels = std::max<int>(1, static_cast<int>(N.level_ptr.size()) - 1);
  const unsigned grid = static_cast<unsigned>(factor_workgroups(N.nchunks, levels));
  const bool add = N.ic && N.additive;
#define LA_FAC(G, IC)                                                                          \
  hipLaunchKernelGGL((k_factor_rows<G, IC>), dim3(grid), dim3(64 * kFacWaves), 0, s, N.nchunks, \
                     N.chunk_start.as<int>(), N.rows.as<int>(), N.fai.as<int>(),                \
                     N.faj.as<int>(), IC ? N.pptr.as<int>() : N.dpos.as<int>(), N.pk.as<int>(), \
                     N.pq.as<int>(), N.f2a.as<int>(), a_vals, fav, 1.0 + N.omega,               \
                     add ? N.omega : 0.0, add ? 1 : 0, N.ticket.as<unsigned>(), N.err.as<int>())
#define LA_FACG(IC)                                                                            \
  switch (N.lanes) {                                                                           \
    case 4: LA_FAC(4, IC); break;                                                              \
    case 8: LA_FAC(8, IC); break;                                                              \
    case 16: LA_FAC(16, IC); break;                                                            \
    case 32: LA_FAC(32, IC); break;                                                            \
    default: LA_FAC(64, IC); break;                                                            \
  }
  if (N.ic) LA_FACG(true) else LA_FACG(false)
#undef LA_FACG
#undef LA_FAC
  LA_HIP(hipGetLastError());
}

void factor_levels(NumericPlan &N, const double *a_vals, hipStream_t s) {
  double *fav = N.fav.as<double>();
  hipLaunchKernelGGL(k_fill_zero, dim3(2048), dim3(256), 0, s, N.nnzF, fav);
  if (N.nnzA)
    hipLaunchKernelGGL(k_scatter, dim3(static_cast<unsigned>((N.nnzA + 255) / 256)), dim3(256),
                       0, s, N.nnzA, N.a2f.as<int64_t>(), a_vals, fav);
  if (N.ic && N.additive)
    hipLaunchKernelGGL(k_shift_first, dim3((N.n + 255) / 256), dim3(256), 0, s, N.n,
                       N.fai.as<int>(), fav, N.omega);
  else if (N.ic)
    hipLaunchKernelGGL(k_scale_first, dim3((N.n + 255) / 256), dim3(256), 0, s, N.n,
                       N.fai.as<int>(), fav, 1.0 + N.omega);
  LA_HIP(hipGetLastError());
  const int L = static_cast<int>(N.level_ptr.size()) - 1;
  for (int l = 0; l < L; ++l) {
    const int k0 = N.level_ptr[l], cnt = N.level_ptr[l + 1] - k0;
    if (cnt <= 0) continue;
    if (N.ic)
      hipLaunchKernelGGL(k_ic_rows, dim3(cnt), dim3(64), 0, s, k0, N.rows.as<int>(),
                         N.fai.as<int>(), N.faj.as<int>(), N.pptr.as<int>(), N.pk.as<int>(),
                         N.pq.as<int>(), fav, N.err.as<int>(), N.additive ? 1 : 0);
    else
      hipLaunchKernelGGL(k_ilu_rows, dim3(cnt), dim3(64), 0, s, k0, N.rows.as<int>(),
                         N.fai.as<int>(), N.faj.as<int>(), N.fu.as<int>(), fav,
                         N.diag.as<double>(), N.err.as<int>());
  }
  LA_HIP(hipGetLastError());
}
}  // namespace

void prec_refactor(Prec &P, const double *a_vals, hipStream_t s) {
  if (!P.num) throw la_error(LA_ERR_STATE, "preconditioner was built from a host factor");
  NumericPlan &N = *P.num;
  LA_CHECK_ARG(a_vals || N.nnzA == 0, "null values");
  if (N.n == 0) return;
  LA_HIP(hipMemsetAsync(N.err.p, 0, sizeof(int) * 4, s));
  if (N.lanes) factor_rows(N, a_vals, s);
  else factor_levels(N, a_vals, s);
  double *fav = N.fav.as<double>();
  int bad[2] = {0, 0};
  LA_HIP(hipMemcpyAsync(bad, N.err.p, sizeof(bad), hipMemcpyDeviceToHost, s));
  LA_HIP(hipStreamSynchronize(s));
  if (bad[1]) throw la_error(LA_ERR_TIMEOUT, "sync-free factorisation exceeded its spin bound");
  if (bad[0])
    throw la_error(LA_ERR_NUMERIC, !N.ic        ? "ILU factorisation met a row without a diagonal"
                                   : N.additive ? "IC factorisation hit a non-positive pivot"
                                                : "IC factorisation hit a negative pivot");
  trsv_refresh(*P.lower, fav, s);
  trsv_refresh(*P.upper, fav, s);
  LA_HIP(hipStreamSynchronize(s));
}

void prec_factor(Prec &P, std::vector<int> *fai, std::vector<int> *faj, std::vector<double> *fav,
                 hipStream_t s) {
  if (!P.num) throw la_error(LA_ERR_STATE, "preconditioner was built from a host factor");
  NumericPlan &N = *P.num;
  if (fai) *fai = N.h_fai;
  if (faj) *faj = N.h_faj;
  if (fav) {
    fav->resize(static_cast<size_t>(N.nnzF));
    if (N.nnzF)
      LA_HIP(hipMemcpyAsync(fav->data(), N.fav.p, sizeof(double) * N.nnzF, hipMemcpyDeviceToHost,
                            s));
    LA_HIP(hipStreamSynchronize(s));
  }
}

}  // namespace laamd
