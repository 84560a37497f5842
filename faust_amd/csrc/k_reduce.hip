// k_reduce.hip -- canonical FP64 reductions, elementwise kernels and
// dense <-> CSR/CSC conversions.
#include <algorithm>
#include <numeric>

#include "fh_internal.hpp"

namespace fh {

// ---------------------------------------------------------------- reductions
// One workgroup of 256 lanes per 4096-element chunk; lane t accumulates
// elements c*4096 + t + 256*m (m = 0..15), then a halving tree.
template <int MODE>  // 0: sum x, 1: dot x.y
__global__ __launch_bounds__(256) void k_reduce_chunks(const double* __restrict__ x, const double* __restrict__ y,
                                                       int64_t n, double* __restrict__ part) {
  __shared__ double p[RED_LANES];
  const int t = threadIdx.x;
  const int64_t base = (int64_t)blockIdx.x * RED_CHUNK;
  double acc = 0.0;
#pragma unroll
  for (int m = 0; m < RED_CHUNK / RED_LANES; ++m) {
    int64_t i = base + (int64_t)m * RED_LANES + t;
    if (i < n) acc = MODE ? fma(x[i], y[i], acc) : acc + x[i];
  }
  p[t] = acc;
  __syncthreads();
  for (int s = RED_LANES / 2; s >= 1; s >>= 1) {
    if (t < s) p[t] = p[t] + p[t + s];
    __syncthreads();
  }
  if (t == 0) part[blockIdx.x] = p[0];
}

// chunk partials in order: staged in LDS so that their loads are in flight
// together (one at a time they took 3 us for 16 chunks)
__global__ __launch_bounds__(256) void k_reduce_final(const double* __restrict__ part, int64_t nchunks,
                                                      double* __restrict__ out, double* __restrict__ out2) {
  __shared__ double p[256];
  double tot = 0.0;
  for (int64_t c0 = 0; c0 < nchunks; c0 += 256) {
    const int nc = (int)min((int64_t)256, nchunks - c0);
    if ((int)threadIdx.x < nc) p[threadIdx.x] = part[c0 + threadIdx.x];
    __syncthreads();
    if (threadIdx.x == 0)
      for (int c = 0; c < nc; ++c) tot = tot + p[c];
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    *out = tot;
    if (out2) *out2 = tot;
  }
}

static void reduce_launch(int mode, const double* x, const double* y, int64_t n, double* out, double* out2,
                          hipStream_t st) {
  const int64_t nch = n <= 0 ? 0 : (n + RED_CHUNK - 1) / RED_CHUNK;
  DBuf part(sizeof(double) * std::max<int64_t>(nch, 1));
  if (nch > 0) {
    if (mode)
      hipLaunchKernelGGL(k_reduce_chunks<1>, dim3((unsigned)nch), dim3(RED_LANES), 0, st, x, y, n, part.as<double>());
    else
      hipLaunchKernelGGL(k_reduce_chunks<0>, dim3((unsigned)nch), dim3(RED_LANES), 0, st, x, y, n, part.as<double>());
    FH_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_reduce_final, dim3(1), dim3(256), 0, st, part.as<double>(), nch, out, out2);
  FH_LAUNCH_CHECK();
}

void reduce_dot_f64(const double* x, const double* y, int64_t n, double* out, hipStream_t st, double* out2) {
  reduce_launch(1, x, y, n, out, out2, st);
}
void reduce_sum_f64(const double* x, int64_t n, double* out, hipStream_t st, double* out2) {
  reduce_launch(0, x, nullptr, n, out, out2, st);
}

__global__ __launch_bounds__(256) void k_any_nan(const double* __restrict__ x, int64_t n, double* __restrict__ out) {
  bool nan = false;
  for (int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x; i < n; i += (int64_t)gridDim.x * 256) nan |= x[i] != x[i];
  if (__any(nan) && (threadIdx.x & 63) == 0) *out = 1.0;  // the same value from every wave that gets here
}

void any_nan_f64(const double* x, int64_t n, double* out, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_any_nan, dim3((unsigned)std::min<int64_t>(1024, (n + 255) / 256)), dim3(256), 0, st, x, n, out);
  FH_LAUNCH_CHECK();
}

// diag[i] = sum_k A[k,i]*S[k,i] in ascending k (the diagonal of A^T S): one
// fma chain per column.  A workgroup stages 16 columns of both matrices in LDS,
// 128 rows at a time and coalesced (the next 128 in flight meanwhile), and 16
// lanes run the chains.  With a thread reading its own column from memory, 256
// columns of 256 took 63 us.
constexpr int DD_COLS = 16, DD_K = 128, DD_PT = DD_COLS * DD_K / 256;
__global__ __launch_bounds__(256) void k_diag_dot(const double* __restrict__ A, const double* __restrict__ S, int m,
                                                  int n, double* __restrict__ diag) {
  __shared__ double la[DD_COLS][DD_K + 1], ls[DD_COLS][DD_K + 1];
  const int t = threadIdx.x, i0 = blockIdx.x * DD_COLS;
  double ra[DD_PT], rs[DD_PT];
  auto fetch = [&](int k0) {
#pragma unroll
    for (int q = 0; q < DD_PT; ++q) {
      const int e = t + 256 * q, k = min(k0 + e % DD_K, m - 1), i = min(i0 + e / DD_K, n - 1);
      ra[q] = A[(size_t)i * m + k];
      rs[q] = S[(size_t)i * m + k];
    }
  };
  double acc = 0.0;
  fetch(0);
  for (int k0 = 0; k0 < m; k0 += DD_K) {
    __syncthreads();  // the previous rows have been used
#pragma unroll
    for (int q = 0; q < DD_PT; ++q) {
      const int e = t + 256 * q;
      la[e / DD_K][e % DD_K] = ra[q];
      ls[e / DD_K][e % DD_K] = rs[q];
    }
    __syncthreads();
    if (k0 + DD_K < m) fetch(k0 + DD_K);
    if (t < DD_COLS) {
      const int nk = min(DD_K, m - k0);
      int k = 0;
      for (; k + 16 <= nk; k += 16) {
        double x[16], y[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
          x[u] = la[t][k + u];
          y[u] = ls[t][k + u];
        }
#pragma unroll
        for (int u = 0; u < 16; ++u) acc = fma(x[u], y[u], acc);
      }
      for (; k < nk; ++k) acc = fma(la[t][k], ls[t][k], acc);
    }
  }
  if (t < DD_COLS && i0 + t < n) diag[i0 + t] = acc;
}

void diag_dot_f64(const double* A, const double* S, int m, int n, double* diag, hipStream_t st) {
  if (n <= 0) return;
  if (m <= 0) {
    fill_f64(diag, n, 0.0, st);
    return;
  }
  hipLaunchKernelGGL(k_diag_dot, dim3((n + DD_COLS - 1) / DD_COLS), dim3(256), 0, st, A, S, m, n, diag);
  FH_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- elementwise
__global__ void k_axpby(double* __restrict__ y, const double* __restrict__ x, int64_t n, double a, double b) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) {
    double t = a * x[i];
    y[i] = (b == 0.0) ? t : fma(b, y[i], t);
  }
}
void axpby_f64(double* y, const double* x, int64_t n, double a, double b, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_axpby, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, x, n, a, b);
  FH_LAUNCH_CHECK();
}

// mode 0: x *= hscale; mode 1: x *= 1/sqrt(*dscale) (Frobenius normalisation
// from a device sum of squares: nrm = sqrt(s), inv = 1.0/nrm, x *= inv)
__global__ void k_scale(double* __restrict__ x, int64_t n, const double* __restrict__ ds, double hs, int mode) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= n) return;
  double s = hs;
  if (mode == 1) {
    double nrm = sqrt(*ds);
    s = 1.0 / nrm;
  }
  x[i] = x[i] * s;
}
void scale_f64(double* x, int64_t n, const double* dscale, double hscale, int mode, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_scale, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, n, dscale, hscale, mode);
  FH_LAUNCH_CHECK();
}

__global__ void k_sub(double* __restrict__ y, const double* __restrict__ x, int64_t n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) y[i] = y[i] - x[i];
}
void sub_f64(double* y, const double* x, int64_t n, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_sub, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, y, x, n);
  FH_LAUNCH_CHECK();
}

__global__ void k_fill(double* __restrict__ x, int64_t n, double v) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < n) x[i] = v;
}
void fill_f64(double* x, int64_t n, double v, hipStream_t st) {
  if (n <= 0) return;
  hipLaunchKernelGGL(k_fill, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, x, n, v);
  FH_LAUNCH_CHECK();
}

__global__ void k_eye(double* __restrict__ x, int m, int n) {
  int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  if (i < (int64_t)m * n) {
    int r = (int)(i % m), c = (int)(i / m);
    x[i] = (r == c) ? 1.0 : 0.0;
  }
}
void eye_f64(double* x, int m, int n, hipStream_t st) {
  int64_t N = (int64_t)m * n;
  if (N <= 0) return;
  hipLaunchKernelGGL(k_eye, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st, x, m, n);
  FH_LAUNCH_CHECK();
}

// ---------------------------------------------------------------- conversions
// Dense -> CSR and CSC, by tiles of 64 rows x 64 columns (a lane per row, a
// wave per 16 columns, so the loads are coalesced and 16 deep): a count of
// every tile's rows and columns, a scan of the counts into line pointers and
// per-tile offsets (one workgroup for the rows, one for the columns), and a
// second pass over the tiles that writes each entry at its offset, columns
// ascending inside a row and rows ascending inside a column.  The only wait
// is for the entry count that sizes the arrays, which the scan writes to
// mail(); with the scan on the host, between two copies each way, a 256 x 256
// conversion took 4 kernels of 7 us, 6 copies and 2 waits.
constexpr int CV_T = 64;

// the 16 values of row r0 + lane, columns c0 .. c0 + 15 (0 outside the matrix)
__device__ __forceinline__ void cv_load(const double* __restrict__ D, int m, int n, int r, int c0, double (&x)[16]) {
  const int rr = min(r, m - 1);
#pragma unroll
  for (int j = 0; j < 16; ++j) x[j] = D[(size_t)min(c0 + j, n - 1) * m + rr];
#pragma unroll
  for (int j = 0; j < 16; ++j) x[j] = (r < m && c0 + j < n) ? x[j] : 0.0;
}

__global__ __launch_bounds__(256) void k_cv_count(const double* __restrict__ D, int m, int n, int* __restrict__ cntR,
                                                  int* __restrict__ cntC) {
  __shared__ int rc[4][CV_T];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = blockIdx.x * CV_T + lane, c0 = blockIdx.y * CV_T + 16 * w;
  double x[16];
  cv_load(D, m, n, r, c0, x);
  int rows = 0, cols = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const bool nz = x[j] != 0.0;
    rows += nz;
    const int k = __popcll(__ballot(nz));
    cols = lane == j ? k : cols;
  }
  if (lane < 16 && c0 + lane < n) cntC[(size_t)blockIdx.x * n + c0 + lane] = cols;
  rc[w][lane] = rows;
  __syncthreads();
  if (w == 0 && r < m) cntR[(size_t)blockIdx.y * m + r] = rc[0][lane] + rc[1][lane] + rc[2][lane] + rc[3][lane];
}

// cnt[ntiles][len] -> write offsets in place, ptr[len + 1], and the largest
// line; block 0: rows, block 1: columns
struct CvScan {
  int* cnt;
  int* ptr;
  int ntiles, len;
};
__global__ __launch_bounds__(1024) void k_cv_scan(CvScan rows, CvScan cols, double* __restrict__ mail3) {
  __shared__ int wsum[16], wmax[16];
  const CvScan s = blockIdx.x ? cols : rows;
  const int t = threadIdx.x, lane = t & 63, w = t >> 6;
  int carry = 0, widest = 0;
  for (int i0 = 0; i0 < s.len; i0 += 1024) {
    const int i = i0 + t;
    int tot = 0;
    if (i < s.len)
      for (int c = 0; c < s.ntiles; ++c) tot += s.cnt[(size_t)c * s.len + i];
    widest = max(widest, tot);
    int incl = tot;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int o = __shfl_up(incl, d, 64);
      if (lane >= d) incl += o;
    }
    if (lane == 63) wsum[w] = incl;
    __syncthreads();
    int before = 0, all = 0;
#pragma unroll
    for (int q = 0; q < 16; ++q) {
      before += q < w ? wsum[q] : 0;
      all += wsum[q];
    }
    int p = carry + before + incl - tot;
    if (i < s.len) {
      s.ptr[i] = p;
      for (int c = 0; c < s.ntiles; ++c) {
        const int k = s.cnt[(size_t)c * s.len + i];
        s.cnt[(size_t)c * s.len + i] = p;
        p += k;
      }
    }
    carry += all;
    __syncthreads();  // wsum read before the next 1024 lines write it
  }
#pragma unroll
  for (int d = 32; d >= 1; d >>= 1) widest = max(widest, __shfl_xor(widest, d, 64));
  if (lane == 0) wmax[w] = widest;
  __syncthreads();
  if (t == 0) {
    s.ptr[s.len] = carry;
    for (int q = 1; q < 16; ++q) widest = max(widest, wmax[q]);
    if (blockIdx.x == 0) mail3[0] = (double)carry;
    mail3[1 + blockIdx.x] = (double)widest;
  }
}

__global__ __launch_bounds__(256) void k_cv_fill(const double* __restrict__ D, int m, int n,
                                                 const int* __restrict__ offR, const int* __restrict__ offC,
                                                 int* __restrict__ ci, double* __restrict__ v, int* __restrict__ ri,
                                                 double* __restrict__ cv) {
  __shared__ int rc[4][CV_T];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int r = blockIdx.x * CV_T + lane, c0 = blockIdx.y * CV_T + 16 * w;
  double x[16];
  cv_load(D, m, n, r, c0, x);
  int rows = 0;
#pragma unroll
  for (int j = 0; j < 16; ++j) rows += x[j] != 0.0;
  rc[w][lane] = rows;
  __syncthreads();
  int p = r < m ? offR[(size_t)blockIdx.y * m + r] : 0;
  for (int q = 0; q < w; ++q) p += rc[q][lane];
  const unsigned long long below = ((unsigned long long)1 << lane) - 1;
#pragma unroll
  for (int j = 0; j < 16; ++j) {
    const bool nz = x[j] != 0.0;  // only inside the matrix
    const unsigned long long mask = __ballot(nz);
    if (nz) {
      ci[p] = c0 + j;
      v[p] = x[j];
      ++p;
      const int q = offC[(size_t)blockIdx.x * n + c0 + j] + __popcll(mask & below);
      ri[q] = r;
      cv[q] = x[j];
    }
  }
}

void dense_to_csr_f64(const double* D, int m, int n, DMat& out, hipStream_t st) {
  out.kind = K_CSR;
  out.dtype = FH_F64;
  out.m = m;
  out.n = n;
  out.has_csc = true;
  out.rp.alloc(sizeof(int) * ((size_t)m + 1));
  out.cp.alloc(sizeof(int) * ((size_t)n + 1));
  double* size = mail() + MAIL_CSR;
  const bool any = m > 0 && n > 0;
  const int tr = (m + CV_T - 1) / CV_T, tc = (n + CV_T - 1) / CV_T;
  DBuf cr(sizeof(int) * std::max<size_t>((size_t)tc * m, 1)), cc(sizeof(int) * std::max<size_t>((size_t)tr * n, 1));
  const dim3 grid(tr, tc);
  if (any) {
    hipLaunchKernelGGL(k_cv_count, grid, dim3(256), 0, st, D, m, n, cr.as<int>(), cc.as<int>());
    FH_LAUNCH_CHECK();
  }
  hipLaunchKernelGGL(k_cv_scan, dim3(2), dim3(1024), 0, st, CvScan{cr.as<int>(), out.rp.as<int>(), any ? tc : 0, m},
                     CvScan{cc.as<int>(), out.cp.as<int>(), any ? tr : 0, n}, size);
  FH_LAUNCH_CHECK();
  FH_HIP(hipStreamSynchronize(st));
  const int64_t nnz = (int64_t)size[0];
  out.nnz = nnz;
  out.max_row = (int)size[1];
  out.max_col = (int)size[2];
  out.ci.alloc(sizeof(int) * std::max<int64_t>(nnz, 1));
  out.v.alloc(sizeof(double) * std::max<int64_t>(nnz, 1));
  out.ri.alloc(sizeof(int) * std::max<int64_t>(nnz, 1));
  out.cv.alloc(sizeof(double) * std::max<int64_t>(nnz, 1));
  if (nnz > 0) {
    hipLaunchKernelGGL(k_cv_fill, grid, dim3(256), 0, st, D, m, n, cr.as<int>(), cc.as<int>(), out.ci.as<int>(),
                       out.v.as<double>(), out.ri.as<int>(), out.cv.as<double>());
    FH_LAUNCH_CHECK();
  }
}

// CSC -> dense: a wave per column composes 512 rows at a time in LDS (zeros,
// then the column's entries among them) and stores them coalesced; one launch
// in place of a fill and a scatter of one thread per row
constexpr int CD_ROWS = 512;
__global__ __launch_bounds__(256) void k_csc_dense(int m, int n, const int* __restrict__ cp,
                                                   const int* __restrict__ ri, const double* __restrict__ cv,
                                                   double* __restrict__ D) {
  __shared__ double buf[4][CD_ROWS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int j = blockIdx.x * 4 + w, r0 = blockIdx.y * CD_ROWS;
  if (j >= n) return;  // the whole wave; waves share nothing
  const int nr = min(CD_ROWS, m - r0), b = cp[j], e = cp[j + 1];
  double* col = buf[w];
#pragma unroll
  for (int q = 0; q < CD_ROWS / 64; ++q) col[lane + 64 * q] = 0.0;
  __builtin_amdgcn_wave_barrier();
  for (int p = b + lane; p < e; p += 64) {
    const int r = ri[p] - r0;
    if (r >= 0 && r < nr) col[r] = cv[p];
  }
  __builtin_amdgcn_wave_barrier();
#pragma unroll
  for (int q = 0; q < CD_ROWS / 64; ++q)
    if (lane + 64 * q < nr) D[(size_t)j * m + r0 + lane + 64 * q] = col[lane + 64 * q];
}

__global__ void k_csr_scatter(int m, const int* __restrict__ rp, const int* __restrict__ ci,
                              const double* __restrict__ v, double* __restrict__ D) {
  int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i >= m) return;
  for (int p = rp[i]; p < rp[i + 1]; ++p) D[(size_t)ci[p] * m + i] = v[p];
}

void csr_to_dense_f64(const DMat& S, double* D, hipStream_t st) {
  if (S.m == 0 || S.n == 0) return;
  const int chunks = (S.m + CD_ROWS - 1) / CD_ROWS;
  // every chunk of a column walks its entries: the scatter stays for tall matrices
  if (S.has_csc && chunks <= 16) {
    hipLaunchKernelGGL(k_csc_dense, dim3((S.n + 3) / 4, chunks), dim3(256), 0, st, S.m, S.n, S.cp.as<int>(),
                       S.ri.as<int>(), S.cv.as<double>(), D);
    FH_LAUNCH_CHECK();
    return;
  }
  FH_HIP(hipMemsetAsync(D, 0, sizeof(double) * (size_t)S.m * S.n, st));
  if (S.nnz > 0) {
    hipLaunchKernelGGL(k_csr_scatter, dim3((S.m + 255) / 256), dim3(256), 0, st, S.m, S.rp.as<int>(),
                       S.ci.as<int>(), S.v.as<double>(), D);
    FH_LAUNCH_CHECK();
  }
}

__device__ __forceinline__ bool nz_val(double x) { return x != 0.0; }
__device__ __forceinline__ bool nz_val(float x) { return x != 0.0f; }
__device__ __forceinline__ bool nz_val(uint16_t x) { return (x & 0x7fffu) != 0; }  // BF16 bits: +-0 are zero

// grid-stride count: per-thread counts, a block sum in LDS, one partial per
// workgroup; the partials are added by one more workgroup, which stores the
// count where the host can read it after the stream is synchronized
template <class T>
__global__ __launch_bounds__(256) void k_count_nnz(const T* __restrict__ D, int64_t n, unsigned* __restrict__ out) {
  __shared__ unsigned int part[256];
  unsigned int c = 0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    c += nz_val(D[i]) ? 1u : 0u;
  part[threadIdx.x] = c;
  __syncthreads();
  for (int s = 128; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) part[threadIdx.x] += part[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) out[blockIdx.x] = part[0];
}

__global__ __launch_bounds__(1024) void k_count_final(const unsigned* __restrict__ part, int n,
                                                      unsigned long long* __restrict__ out) {
  __shared__ unsigned long long p[1024];
  p[threadIdx.x] = (int)threadIdx.x < n ? part[threadIdx.x] : 0ull;
  __syncthreads();
  for (int s = 512; s > 0; s >>= 1) {
    if ((int)threadIdx.x < s) p[threadIdx.x] += p[threadIdx.x + s];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = p[0];
}

int64_t count_nnz_f64(const double* D, int64_t n, hipStream_t st) { return count_nnz(D, FH_F64, n, st); }

int64_t count_nnz(const void* D, int dtype, int64_t n, hipStream_t st) {
  if (n <= 0) return 0;
  const int blocks = (int)std::min<int64_t>(1024, (n + 255) / 256);
  DBuf c(sizeof(unsigned) * blocks);
  unsigned* part = c.as<unsigned>();
  const dim3 grid((unsigned)blocks);
  if (dtype == FH_F64)
    hipLaunchKernelGGL(k_count_nnz<double>, grid, dim3(256), 0, st, (const double*)D, n, part);
  else if (dtype == FH_F32)
    hipLaunchKernelGGL(k_count_nnz<float>, grid, dim3(256), 0, st, (const float*)D, n, part);
  else
    hipLaunchKernelGGL(k_count_nnz<uint16_t>, grid, dim3(256), 0, st, (const uint16_t*)D, n, part);
  FH_LAUNCH_CHECK();
  auto* out = reinterpret_cast<unsigned long long*>(mail() + MAIL_COUNT);
  hipLaunchKernelGGL(k_count_final, dim3(1), dim3(1024), 0, st, part, blocks, out);
  FH_LAUNCH_CHECK();
  FH_HIP(hipStreamSynchronize(st));
  return (int64_t)*out;
}

}  // namespace fh
