// k_prox.hip -- sp / spcol / splin / splincol / supp / normcol / normlin projectors (FP64).
//
// The selected support must equal the reference's std::partial_sort result
// bit for bit, ties included.  A workgroup radix select finds the k-th largest
// magnitude T of each line (row or column, staged in LDS) or of the whole
// matrix.  When the entries equal to T are all needed to reach k, the support
// is {|x| >= T} whatever the order of the scan; only when ties at T straddle
// the k boundary does the exact heap selection of heap_select.hpp run, on one
// lane, to pick the tied entries partial_sort keeps.  Zero magnitudes never
// need it: selecting a zero leaves a zero.  The selection is followed by a
// canonical Frobenius normalisation (faust_prox.hpp:72-200;
// MatDense::normalize, faust_MatDense.hpp:1226-1250).
#include <algorithm>
#include <climits>

#include "fh_internal.hpp"
#include "heap_select.hpp"

namespace fh {

// Magnitude key: the bits of |x| order non-negative doubles like their values.
__device__ inline unsigned long long mag_key(double x) {
  return (unsigned long long)__double_as_longlong(fabs(x));
}

// Workgroup radix select (8-bit digits, most significant first) of the k-th
// largest of len keys, 1 <= k <= len.  On return *T is a threshold such that
// the keys >= *T are exactly the k largest, unless the function returns true:
// then *T is the k-th largest key itself and the keys equal to it straddle
// the k boundary, so which of them partial_sort keeps depends on positions
// (the caller runs the exact heap selection); a zero T is never reported as
// ambiguous, since keeping a zero or not gives the same output.  hist: 256 LDS counters; sh: 3
// LDS ints.  Each lane caches two (digit, count) pairs before its LDS atomics,
// which keeps the passes where most keys share a digit (the exponent bits)
// free of atomic contention.
template <class KeyAt>
__device__ bool wg_select_threshold(KeyAt key_at, int len, int k, unsigned* hist, int* sh,
                                    unsigned long long* T) {
  const int tid = threadIdx.x, nt = blockDim.x;
  unsigned long long prefix = 0, mask = 0;
  int kk = k;  // rank of the target among the candidates, from the top
  for (int shift = 56; shift >= 0; shift -= 8) {
    for (int b = tid; b < 256; b += nt) hist[b] = 0u;
    __syncthreads();
    unsigned d0 = 256, c0 = 0, d1 = 256, c1 = 0;
    for (int i = tid; i < len; i += nt) {
      const unsigned long long x = key_at(i);
      if ((x & mask) != prefix) continue;
      const unsigned d = (unsigned)(x >> shift) & 255u;
      if (d == d0) {
        ++c0;
      } else if (d == d1) {
        ++c1;
      } else {
        if (c1) atomicAdd(&hist[d1], c1);
        d1 = d0;
        c1 = c0;
        d0 = d;
        c0 = 1;
      }
    }
    if (c0) atomicAdd(&hist[d0], c0);
    if (c1) atomicAdd(&hist[d1], c1);
    __syncthreads();
    if (tid < 64) {
      // lane l owns bins 255-4l .. 252-4l; inclusive scan of their sums from the top
      const int hi = 255 - 4 * tid;
      const int s = (int)(hist[hi] + hist[hi - 1] + hist[hi - 2] + hist[hi - 3]);
      int incl = s;
      for (int d = 1; d < 64; d <<= 1) {
        const int o = __shfl_up(incl, d, 64);
        if (tid >= d) incl += o;
      }
      const unsigned long long bal = __ballot(incl >= kk);
      const int L = __ffsll((unsigned long long)bal) - 1;
      if (tid == L) {
        int acc = incl - s, b = hi, c = 0;
        for (int j = 0; j < 4; ++j, --b) {
          c = (int)hist[b];
          if (acc + c >= kk) break;
          acc += c;
        }
        sh[0] = b;
        sh[1] = kk - acc;
        sh[2] = c;
      }
    }
    __syncthreads();
    const int b = sh[0], cnt = sh[2];
    kk = sh[1];
    prefix |= (unsigned long long)b << shift;
    mask |= 255ull << shift;
    if (cnt == kk) {  // every candidate left in the bin is taken
      *T = prefix;
      return false;
    }
  }
  *T = prefix;
  return prefix != 0;  // tied zeros: every choice gives the same output
}

// One 64-lane workgroup per line: the first ncol_lines are columns (spcol), the
// rest rows (splin), written to outc and outr; a line is staged before it is
// written, so an output may be M itself (when only one kind is selected).
// Dynamic LDS holds the line values and
// the heap when they fit (lds_ok), else per-line global scratch is used.  The
// radix threshold decides the support unless ties straddle the k boundary;
// only those lines run the heap selection on one lane.
__global__ __launch_bounds__(64) void k_prox_lines(const double* M, int m, int n, int ncol_lines, int k, double* outc,
                                                   double* outr, int lds_ok, double* __restrict__ gvals,
                                                   int* __restrict__ gidx, double* __restrict__ gabs) {
  extern __shared__ double smem[];
  __shared__ unsigned hist[256];
  __shared__ int sh[3];
  const bool along_rows = (int)blockIdx.x >= ncol_lines;
  const int line = along_rows ? blockIdx.x - ncol_lines : blockIdx.x;
  const int len = along_rows ? n : m;
  double* out = along_rows ? outr : outc;
  double* vals;
  double* habs;
  int* hidx;
  if (lds_ok) {
    vals = smem;
    habs = smem + len;
    hidx = reinterpret_cast<int*>(smem + len + k);
  } else {
    vals = gvals + (size_t)blockIdx.x * max(m, n);
    habs = gabs + (size_t)blockIdx.x * k;
    hidx = gidx + (size_t)blockIdx.x * k;
  }
  const int lane = threadIdx.x;
  for (int t = lane; t < len; t += 64) vals[t] = along_rows ? M[(size_t)t * m + line] : M[(size_t)line * m + t];
  __syncthreads();
  unsigned long long T;
  const bool ambiguous = wg_select_threshold([vals](int i) { return mag_key(vals[i]); }, len, k, hist, sh, &T);
  for (int t = lane; t < len; t += 64) {
    const double x = (!ambiguous && mag_key(vals[t]) >= T) ? vals[t] : 0.0;
    if (along_rows)
      out[(size_t)t * m + line] = x;
    else
      out[(size_t)line * m + t] = x;
  }
  if (!ambiguous) return;
  __syncthreads();
  if (lane == 0) heap_select<double>(len, k, [vals](int i) { return fabs(vals[i]); }, hidx, habs);
  __syncthreads();
  for (int q = lane; q < k; q += 64) {
    int t = hidx[q];
    if (along_rows)
      out[(size_t)t * m + line] = vals[t];
    else
      out[(size_t)line * m + t] = vals[t];
  }
}

// Global top-k over all m*n entries in column-major order (prox_sp).
struct SpSel {
  unsigned long long T;
  int ambiguous;
};

// The k-th largest magnitude of N entries in one workgroup: a radix select with
// 11-bit digits (the exponent first) over the entries in global memory, 16
// loads in flight per thread, until at most SP_LIST candidates share the
// digits found; those are then gathered in LDS and ranked against each other.
// Ties that straddle k (see wg_select_threshold) are settled by the exact heap
// selection on one lane, and the k entries it keeps are saved before the
// caller overwrites M.  8-bit digits over all of M until the bin was exact
// took 45 us for 256 x 256 entries.
constexpr int SP_BITS = 11, SP_BINS = 1 << SP_BITS, SP_LIST = 512, SP_LOADS = 16;
__global__ __launch_bounds__(1024) void k_sp_threshold(const double* __restrict__ M, int N, int k,
                                                       SpSel* __restrict__ sel, int* __restrict__ hidx,
                                                       double* __restrict__ habs, double* __restrict__ hval) {
  __shared__ unsigned hist[SP_BINS];
  __shared__ unsigned wtot[16];
  __shared__ int sh[3], nlist, amb;
  __shared__ unsigned long long list[SP_LIST];
  __shared__ unsigned long long thr;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  unsigned long long prefix = 0, mask = 1ull << 63;  // magnitudes have no sign bit
  int kk = k;
  // runs f(key) for every entry
  auto each = [&](auto&& f) {
    for (int64_t i0 = t; i0 < N; i0 += 1024 * SP_LOADS) {
      unsigned long long x[SP_LOADS];
#pragma unroll
      for (int u = 0; u < SP_LOADS; ++u) x[u] = mag_key(M[min(i0 + 1024 * u, (int64_t)N - 1)]);
#pragma unroll
      for (int u = 0; u < SP_LOADS; ++u)
        if (i0 + 1024 * u < N) f(x[u]);
    }
  };
  bool done = false;
  for (int shift = 63 - SP_BITS; !done; shift = max(shift - SP_BITS, 0)) {
    const int bits = mask == 1ull << 63 ? SP_BITS : min(SP_BITS, __builtin_ctzll(mask));
    for (int b = t; b < SP_BINS; b += 1024) hist[b] = 0u;
    if (t == 0) nlist = 0;
    __syncthreads();
    // two (digit, count) pairs per thread ahead of the LDS atomics
    unsigned d0 = SP_BINS, c0 = 0, d1 = SP_BINS, c1 = 0;
    const unsigned dmask = (1u << bits) - 1;
    each([&](unsigned long long x) {
      if ((x & mask) != prefix) return;
      const unsigned d = (unsigned)(x >> shift) & dmask;
      if (d == d0) {
        ++c0;
      } else if (d == d1) {
        ++c1;
      } else {
        if (c1) atomicAdd(&hist[d1], c1);
        d1 = d0;
        c1 = c0;
        d0 = d;
        c0 = 1;
      }
    });
    if (c0) atomicAdd(&hist[d0], c0);
    if (c1) atomicAdd(&hist[d1], c1);
    __syncthreads();
    // thread t owns the bins SP_BINS - 1 - 2t and the one below; inclusive scan from the top
    const int hi = SP_BINS - 1 - 2 * t;
    const unsigned h0 = hist[hi], h1 = hist[hi - 1];
    unsigned incl = h0 + h1;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const unsigned o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) wtot[w] = incl;
    __syncthreads();
    for (int q = 0; q < w; ++q) incl += wtot[q];
    const int before = (int)(incl - h0 - h1);
    if (before < kk && kk <= (int)incl) {
      const bool first = before + (int)h0 >= kk;
      sh[0] = first ? hi : hi - 1;
      sh[1] = kk - before - (first ? 0 : (int)h0);
      sh[2] = first ? (int)h0 : (int)h1;
    }
    __syncthreads();
    const int cnt = sh[2];
    kk = sh[1];
    prefix |= (unsigned long long)sh[0] << shift;
    mask |= (unsigned long long)dmask << shift;
    if (cnt == kk || shift == 0) {  // every candidate is taken, or all are equal
      if (t == 0) {
        thr = prefix;
        amb = cnt != kk && prefix != 0;
      }
      done = true;
    } else if (cnt <= SP_LIST) {
      each([&](unsigned long long x) {
        if ((x & mask) == prefix) list[atomicAdd(&nlist, 1)] = x;
      });
      __syncthreads();
      if (t < cnt) {  // x is the threshold when fewer than kk are larger and at least kk are as large
        const unsigned long long x = list[t];
        int gt = 0, ge = 0;
        for (int q = 0; q < cnt; ++q) {
          gt += list[q] > x;
          ge += list[q] >= x;
        }
        if (gt < kk && kk <= ge) {  // the same values from every thread that gets here
          thr = x;
          amb = ge != kk && x != 0;
        }
      }
      done = true;
    }
    __syncthreads();
  }
  if (t == 0) {
    sel->T = thr;
    sel->ambiguous = amb;
    if (amb) heap_select<double>(N, k, [M](int i) { return fabs(M[i]); }, hidx, habs);
  }
  if (!amb) return;
  __threadfence_block();
  __syncthreads();
  for (int q = t; q < k; q += 1024) hval[q] = M[hidx[q]];
}

// in place; the ambiguous case clears everything and k_scatter_sel puts the saved entries back
__global__ void k_sp_apply(double* __restrict__ M, int64_t N, const SpSel* __restrict__ sel) {
  const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= N) return;
  const double x = M[i];
  M[i] = (!sel->ambiguous && mag_key(x) >= sel->T) ? x : 0.0;
}

__global__ void k_scatter_sel(double* __restrict__ M, const int* __restrict__ idx, const double* __restrict__ val,
                              int k, const SpSel* __restrict__ sel) {
  if (!sel->ambiguous) return;
  int q = blockIdx.x * blockDim.x + threadIdx.x;
  if (q < k) M[idx[q]] = val[q];
}

__global__ void k_pos(double* __restrict__ M, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n && (float)M[i] < 0.0f) M[i] = 0.0;
}

// Mc and Ml may be out
__global__ void k_union(const double* Mc, const double* Ml, double* out, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    double c = Mc[i];
    double l = (c != 0.0) ? 0.0 : Ml[i];
    out[i] = c + l;
  }
}

__global__ void k_fill_zero(double* __restrict__ M, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) M[i] = 0.0;
}

__global__ void k_hadamard(double* __restrict__ M, const double* __restrict__ S, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) M[i] = M[i] * S[i];
}

// normcol / normlin (faust_prox.hpp:205-255): one 256-lane workgroup per
// line scales it to 2-norm s.  The line's squared norm is the canonical dot
// (4096-element chunks, lane t takes t, t+256, ..., a halving tree per chunk,
// chunk partials added in order), so the scale s/||line|| has the oracle's bits.
__global__ __launch_bounds__(256) void k_line_norm_scale(double* __restrict__ M, int m, int n, int along_rows,
                                                         double s) {
  __shared__ double p[256];
  const int line = blockIdx.x, t = threadIdx.x;
  const int len = along_rows ? n : m;
  const int64_t stride = along_rows ? m : 1;
  double* x = along_rows ? M + line : M + (int64_t)line * m;
  double tot = 0.0;
  for (int c0 = 0; c0 < len; c0 += RED_CHUNK) {
    double acc = 0.0;
    for (int j = 0; j < RED_CHUNK / RED_LANES; ++j) {
      const int i = c0 + j * RED_LANES + t;
      if (i < len) {
        const double v = x[i * stride];
        acc = fma(v, v, acc);
      }
    }
    p[t] = acc;
    __syncthreads();
    for (int h = RED_LANES / 2; h >= 1; h >>= 1) {
      if (t < h) p[t] = p[t] + p[t + h];
      __syncthreads();
    }
    tot = tot + p[0];
    __syncthreads();
  }
  double scale = sqrt(tot);
  if (scale != 0.0) scale = s / scale;
  for (int i = t; i < len; i += RED_LANES) x[i * stride] = x[i * stride] * scale;
}

static inline dim3 g1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }

// top-k per column into outc and per row into outr (dense, same shape as M;
// null: not selected; M itself when the other is null)
static void prox_lines(const double* M, int m, int n, int k, double* outc, double* outr, hipStream_t st) {
  const int ncl = outc ? n : 0, nlines = ncl + (outr ? m : 0);
  const int len = outc && outr ? std::max(m, n) : outc ? m : n;
  if (nlines == 0) return;
  size_t lds = sizeof(double) * ((size_t)len + k) + sizeof(int) * (size_t)k;
  const size_t LDS_MAX = 60 * 1024;
  if (lds <= LDS_MAX) {
    hipLaunchKernelGGL(k_prox_lines, dim3(nlines), dim3(64), lds, st, M, m, n, ncl, k, outc, outr, 1,
                       (double*)nullptr, (int*)nullptr, (double*)nullptr);
  } else {
    DBuf gv(sizeof(double) * (size_t)nlines * std::max(m, n)), gi(sizeof(int) * (size_t)nlines * k),
        ga(sizeof(double) * (size_t)nlines * k);
    hipLaunchKernelGGL(k_prox_lines, dim3(nlines), dim3(64), 0, st, M, m, n, ncl, k, outc, outr, 0, gv.as<double>(),
                       gi.as<int>(), ga.as<double>());
    FH_LAUNCH_CHECK();
    return;
  }
  FH_LAUNCH_CHECK();
}

void check_norm() {
  if (mail()[MAIL_NORM] == 0.0) throw Error(FH_ERR_NUMERIC, "the norm is zero, can't normalize.");
}

static void normalize_inplace(double* M, int64_t N, hipStream_t st, bool defer_norm) {
  double* sq = mail() + MAIL_NORM;
  DBuf s(sizeof(double));
  reduce_dot_f64(M, M, N, s.as<double>(), st, sq);
  if (!defer_norm) {
    FH_HIP(hipStreamSynchronize(st));
    check_norm();
  }
  scale_f64(M, N, s.as<double>(), 0.0, 1, st);
}

void prox_f64(int name, double* M, int m, int n, int64_t k, bool normalized, bool pos, const double* supp,
              hipStream_t st, bool defer_norm) {
  const int64_t N = (int64_t)m * n;
  if (defer_norm) mail()[MAIL_NORM] = 1.0;  // nothing to check unless a norm is taken
  if (N == 0) return;
  auto zero_all = [&]() { FH_HIP(hipMemsetAsync(M, 0, sizeof(double) * N, st)); };
  switch (name) {
    case FH_PROX_SP: {
      if (pos) hipLaunchKernelGGL(k_pos, g1(N), dim3(256), 0, st, M, N);
      if (k <= 0)
        zero_all();
      else if (k < N) {
        FH_CHECK(N < (int64_t)1 << 31, "prox_sp: matrix too large");
        DBuf hi(sizeof(int) * k), ha(sizeof(double) * k), hv(sizeof(double) * k), sel(sizeof(SpSel));
        hipLaunchKernelGGL(k_sp_threshold, dim3(1), dim3(1024), 0, st, M, (int)N, (int)k, sel.as<SpSel>(),
                           hi.as<int>(), ha.as<double>(), hv.as<double>());
        FH_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_sp_apply, g1(N), dim3(256), 0, st, M, N, sel.as<SpSel>());
        FH_LAUNCH_CHECK();
        hipLaunchKernelGGL(k_scatter_sel, g1(k), dim3(256), 0, st, M, hi.as<int>(), hv.as<double>(), (int)k,
                           sel.as<SpSel>());
        FH_LAUNCH_CHECK();
      }
      break;
    }
    case FH_PROX_SPCOL:
    case FH_PROX_SPLIN: {
      const bool rows = (name == FH_PROX_SPLIN);
      if (pos) hipLaunchKernelGGL(k_pos, g1(N), dim3(256), 0, st, M, N);
      if (k <= 0)
        zero_all();
      else if (k < (rows ? n : m))
        prox_lines(M, m, n, (int)k, rows ? nullptr : M, rows ? M : nullptr, st);
      break;
    }
    case FH_PROX_SPLINCOL: {
      // faust_prox.hpp:180-200: both selections run on the input (pos only
      // affects the matrix that is then overwritten)
      if (k <= 0) {
        zero_all();
        break;
      }
      // a selection that keeps whole lines is M itself
      DBuf mc(k < m ? sizeof(double) * N : 0), ml(k < n ? sizeof(double) * N : 0);
      prox_lines(M, m, n, (int)std::min<int64_t>(k, INT_MAX), mc.as<double>(), ml.as<double>(), st);
      const double* pc = k < m ? mc.as<double>() : M;
      const double* pl = k < n ? ml.as<double>() : M;
      hipLaunchKernelGGL(k_union, g1(N), dim3(256), 0, st, pc, pl, M, N);
      FH_LAUNCH_CHECK();
      break;
    }
    case FH_PROX_SUPP: {
      FH_CHECK(supp != nullptr, "prox_supp: missing support matrix");
      if (pos) hipLaunchKernelGGL(k_pos, g1(N), dim3(256), 0, st, M, N);
      hipLaunchKernelGGL(k_hadamard, g1(N), dim3(256), 0, st, M, supp, N);
      FH_LAUNCH_CHECK();
      break;
    }
    default:
      throw Error(FH_ERR_ARG, "prox: unknown constraint");
  }
  if (normalized) normalize_inplace(M, N, st, defer_norm);
}

void prox_real_f64(int name, double* M, int m, int n, double s, bool normalized, bool pos, hipStream_t st,
                   bool defer_norm) {
  const int64_t N = (int64_t)m * n;
  if (defer_norm) mail()[MAIL_NORM] = 1.0;
  FH_CHECK(name == FH_PROX_NORMCOL || name == FH_PROX_NORMLIN, "prox: unknown real-parameter constraint");
  if (N == 0) return;
  if (pos) {
    hipLaunchKernelGGL(k_pos, g1(N), dim3(256), 0, st, M, N);
    FH_LAUNCH_CHECK();
  }
  if (s < 0) throw Error(FH_ERR_ARG, "Faust::prox_normcol : s < 0 ");
  if (s == 0) {
    hipLaunchKernelGGL(k_fill_zero, g1(N), dim3(256), 0, st, M, N);
  } else {
    const bool rows = name == FH_PROX_NORMLIN;
    hipLaunchKernelGGL(k_line_norm_scale, dim3(rows ? m : n), dim3(256), 0, st, M, m, n, rows ? 1 : 0, s);
  }
  FH_LAUNCH_CHECK();
  if (normalized) normalize_inplace(M, N, st, defer_norm);
}

}  // namespace fh
