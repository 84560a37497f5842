// k_power.hip -- power iteration on a factor chain in one persistent launch.
//
// The reference (power_iteration, faust_linear_algebra.hpp:808-898) runs up
// to 100 dependent rounds of "normalise, apply the F F^H chain, Rayleigh
// quotient", each a string of tiny mat-vecs.  Here a single 1024-thread
// workgroup keeps both vectors in LDS and runs every round, every mat-vec and
// the stopping test on the device: no launch or host round trip per step.
// Mat-vecs are one fma chain per output row (k ascending); norms and dots use
// the canonical 256-lane chunk reduction, so the result matches the oracle
// bit for bit.
//
// The chains of PALM4MSA's Lipschitz constants are long strings of small
// sparse factors (a global update of a 10-factor Faust applies up to 18
// factors of 2 entries per row each round, for 100 rounds when the estimate
// does not settle), so a round is a string of dependent latencies, not of
// bytes.  The kernel therefore copies the chain's row pointers into LDS once
// per call, reads the operator descriptors through scalar loads, and loads the
// entries of a thread's rows for the operator after next while it computes the
// current one (rows of up to PW_PF entries; longer rows read theirs in the
// loop), with barriers that order only the LDS vectors, so those loads stay in
// flight across them.  Measured on the 1024 Hadamard hierarchy (100
// iterations per PALM4MSA): 0.71 us per operator and 3.3 us of norm,
// normalisation and Rayleigh quotient per round (11.5 s in this kernel); the
// whole hierarchy takes 24.1 s, against 26.8 s when each thread read its row
// pointers and entries from global memory as it needed them.  Chains whose
// operators are all sparse with rows of at most PW_PF entries run a second
// copy of the round loop without the loops over long rows and dense
// operators: with those in the loop, the compiler waited for every load in
// flight at the start of each operator, the prefetched set included
// (hierarchy 24.3 -> 23.6 s).
#include <algorithm>
#include <climits>
#include <cstdlib>
#include <map>
#include <mutex>

#include "fh_internal.hpp"

namespace fh {

constexpr int PW_THREADS = 1024;
constexpr int PW_VMAX = 2048;  // max vector length kept in LDS (3 vectors: 48 KiB)

struct PwOp {
  int kind;   // 0 dense, 1 row-compressed sparse
  int trans;  // dense only: op(A) = A^T
  int rows, cols;
  const int* rp;
  const int* ci;
  const double* v;  // sparse values or dense data (ld = rows of A)
  int lda;
  int rpo;      // sparse only: offset of the row pointers' copy in dynamic LDS, or -1
  int width;    // sparse only: the longest row, -1 when unknown
  int64_t nnz;  // sparse only
};

constexpr int PW_MAX_OPS = 48;        // longest chain of the persistent form
constexpr int PW_PF = 4;              // entries per row loaded ahead
constexpr int PW_RP_LDS = 96 * 1024;  // dynamic LDS for cached row pointers (bytes)

__device__ __forceinline__ int pw_sgpr(int x) { return __builtin_amdgcn_readfirstlane(x); }

// canonical reduction of dot(x, y) over n values held in LDS; every thread
// returns the same value.  red: 256 doubles of LDS scratch; tot: 1 double.
// Per 4096-value chunk: lane t (< 256) sums x[i] y[i] for i = t, t + 256, ...
// in order, then the halving tree red[t] += red[t + h], h = 128 ... 1; the
// last six levels run inside wave 0 through lane shuffles (the same pairs,
// in the same order).  Chunk sums are added in chunk order.
__device__ double pw_dot(const double* x, const double* y, int n, double* red, double* tot) {
  const int t = threadIdx.x;
  const int nch = (n + RED_CHUNK - 1) / RED_CHUNK;
  double acc_tot = 0.0;
  for (int c = 0; c < nch; ++c) {
    if (t < RED_LANES) {
      double acc = 0.0;
      for (int m = 0; m < RED_CHUNK / RED_LANES; ++m) {
        int i = c * RED_CHUNK + m * RED_LANES + t;
        if (i < n) acc = fma(x[i], y[i], acc);
      }
      red[t] = acc;
    }
    __syncthreads();
    if (t < 128) red[t] = red[t] + red[t + 128];
    __syncthreads();
    if (t < 64) {
      double v = red[t] + red[t + 64];
#pragma unroll
      for (int h = 32; h >= 1; h >>= 1) v = v + __shfl_down(v, h, 64);
      if (t == 0) acc_tot = acc_tot + v;
    }
  }
  if (t == 0) *tot = acc_tot;
  __syncthreads();
  double r = *tot;
  __syncthreads();
  // the same on every lane; said so to the compiler, which then keeps the
  // loop tests that depend on it (and everything inside) scalar
  const unsigned long long u = __builtin_bit_cast(unsigned long long, r);
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Entries of one row of a sparse operator, loaded ahead of their use.
struct PwPre {
  double v[PW_PF];
  int c[PW_PF];
  int p, n;  // first entry and count; n > PW_PF: read in the loop
};

typedef unsigned int pw_u4 __attribute__((ext_vector_type(4)));
typedef double pw_d2 __attribute__((ext_vector_type(2)));
constexpr int PW_RSRC_WORD3 = 0x00020000;

// Global-memory views of the operator arrays for the loops over long rows and
// dense operators (vector memory loads, counted on vmcnt only).
typedef const __attribute__((address_space(1))) double* pw_gd;
typedef const __attribute__((address_space(1))) int* pw_gi;
// Operator descriptors: read-only for the whole launch, read word by word
// through the constant address space (scalar loads).
typedef const __attribute__((address_space(4))) int* pw_cop;
struct PwOpWords {
  int w[sizeof(PwOp) / 4];
};
static_assert(sizeof(PwOp) % 4 == 0, "PwOp is read as words");
__device__ __forceinline__ PwOp pw_op(pw_cop ops, int s) {
  PwOpWords x;
#pragma unroll
  for (int i = 0; i < (int)(sizeof(PwOp) / 4); ++i) x.w[i] = ops[s * (int)(sizeof(PwOp) / 4) + i];
  return __builtin_bit_cast(PwOp, x);
}

// Barrier between operators: orders the LDS vectors only, without waiting
// for the entry loads of the next operators.
__device__ __forceinline__ void pw_lds_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// Loads the first PW_PF entries of row r: two 16-byte buffer loads of values
// and one of column indices, whatever the row and the operator.  The buffers
// cover exactly the operator's entries (none for a dense operator), so reads
// past them return zeros; rows past the operator and dense operators get
// n = 0.  Every thread thus issues the same three loads for every operator,
// and the wait before their use covers only the loads issued before them.
// RP_LDS: the row pointers are in LDS (a dense operator's rpo points at valid
// LDS), else they are read from global memory.
// The descriptor fields pw_fetch needs, read from LDS into scalar registers
// (the same for every lane), so the buffer resources are scalar.
struct PwU {
  const double* v;
  const int* ci;
  const int* rp;
  int kind, rows, rpo, nnz;
};
template <class T>
__device__ __forceinline__ T* pw_sptr(T* p) {
  const unsigned long long u = (unsigned long long)p;
  const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)u), hi = __builtin_amdgcn_readfirstlane((unsigned)(u >> 32));
  return (T*)(((unsigned long long)hi << 32) | lo);
}
__device__ __forceinline__ PwU pw_uniform(const PwOp o) {
  PwU u;
  u.v = pw_sptr(o.v);
  u.ci = pw_sptr(o.ci);
  u.rp = pw_sptr(o.rp);
  u.kind = pw_sgpr(o.kind);
  u.rows = pw_sgpr(o.rows);
  u.rpo = pw_sgpr(o.rpo);
  u.nnz = pw_sgpr((int)o.nnz);
  return u;
}

template <bool RP_LDS, bool SHORT = false>
__device__ __forceinline__ void pw_fetch(const PwOp od, const int* rpl, int r, PwPre& f) {
  const PwU o = pw_uniform(od);
  const bool sp = SHORT || o.kind == 1;
  const int rr = min(r, o.rows - 1);
  int p0, p1;
  if (RP_LDS) {
    p0 = rpl[o.rpo + rr];
    p1 = rpl[o.rpo + rr + 1];
  } else {
    const pw_gi rp = (pw_gi)o.rp;
    p0 = sp ? rp[rr] : 0;
    p1 = sp ? rp[rr + 1] : 0;
  }
  f.p = p0;
  f.n = (sp && r < o.rows) ? p1 - p0 : 0;
  const int vb = sp ? o.nnz * 8 : 0, cb = sp ? o.nnz * 4 : 0;
  const __amdgpu_buffer_rsrc_t rv = __builtin_amdgcn_make_buffer_rsrc((void*)o.v, 0, vb, PW_RSRC_WORD3);
  const __amdgpu_buffer_rsrc_t rc = __builtin_amdgcn_make_buffer_rsrc((void*)o.ci, 0, cb, PW_RSRC_WORD3);
  const pw_d2 v01 = __builtin_bit_cast(pw_d2, __builtin_amdgcn_raw_buffer_load_b128(rv, p0 * 8, 0, 0));
  const pw_d2 v23 = __builtin_bit_cast(pw_d2, __builtin_amdgcn_raw_buffer_load_b128(rv, p0 * 8 + 16, 0, 0));
  const pw_u4 c = __builtin_amdgcn_raw_buffer_load_b128(rc, p0 * 4, 0, 0);
  f.v[0] = v01.x;
  f.v[1] = v01.y;
  f.v[2] = v23.x;
  f.v[3] = v23.y;
  f.c[0] = (int)c.x;
  f.c[1] = (int)c.y;
  f.c[2] = (int)c.z;
  f.c[3] = (int)c.w;
}

// row r of op(o) applied to cur (LDS), entries from f when they were loaded.
// SHORT: every operator of the chain is sparse with rows of at most PW_PF
// entries, so the row is the prefetched slots alone, taken without branches:
// every slot's column is a valid column of the operator (an entry of this
// row or a later one, or 0 past the entries) and the terms past the row end
// are computed and not kept (the same fma chain, the same bits).
// K (SHORT only): the operator's longest row, the same on every lane, so that
// rows of at most two entries gather two slots, not four.
template <bool SHORT>
__device__ __forceinline__ double pw_row(const PwOp o, const PwPre& f, int r, const double* cur, int K = PW_PF) {
  double acc = 0.0;
  if (SHORT) {
    // two slots when no row has more than two entries, else all four; the
    // gathers of a case are issued before its fma chain
    if (K <= 2) {
      const double x0 = cur[f.c[0]], x1 = cur[f.c[1]];
      const double t0 = fma(f.v[0], x0, acc);
      acc = (0 < f.n) ? t0 : acc;
      const double t1 = fma(f.v[1], x1, acc);
      return (1 < f.n) ? t1 : acc;
    }
    double x[PW_PF];
#pragma unroll
    for (int k = 0; k < PW_PF; ++k) x[k] = cur[f.c[k]];
#pragma unroll
    for (int k = 0; k < PW_PF; ++k) {
      const double tk = fma(f.v[k], x[k], acc);
      acc = (k < f.n) ? tk : acc;
    }
    return acc;
  }
  if (o.kind == 1) {
    if (f.n <= PW_PF) {
#pragma unroll
      for (int k = 0; k < PW_PF; ++k)
        if (k < f.n) acc = fma(f.v[k], cur[f.c[k]], acc);
    } else {
      const pw_gd v = (pw_gd)o.v;
      const pw_gi ci = (pw_gi)o.ci;
      for (int p = f.p, pe = f.p + f.n; p < pe; ++p) acc = fma(v[p], cur[ci[p]], acc);
    }
  } else if (!o.trans) {
    const pw_gd a = (pw_gd)o.v + r;
    for (int kk = 0; kk < o.cols; ++kk) acc = fma(a[(size_t)kk * o.lda], cur[kk], acc);
  } else {
    const pw_gd a = (pw_gd)o.v + (size_t)r * o.lda;
    for (int kk = 0; kk < o.cols; ++kk) acc = fma(a[kk], cur[kk], acc);
  }
  return acc;
}

// One operator of the chain: row t (and t + PW_THREADS when TWO_ROWS) of
// operator s from cur into nxt with the entries in (f0, f1), which are then
// reloaded with those of operator s - 2; ends with the LDS barrier.
// Marks the prefetched registers as read on every path, so that the wait for
// their loads sits here (with the next operator's loads still in flight) and
// the registers can be reused afterwards without a wait for everything.
__device__ __forceinline__ void pw_settle(const PwPre& f) {
  asm volatile("" ::"v"(f.v[0]), "v"(f.v[1]), "v"(f.v[2]), "v"(f.v[3]), "v"(f.c[0]), "v"(f.c[1]), "v"(f.c[2]),
               "v"(f.c[3]));
}

template <bool RP_LDS, bool TWO_ROWS, bool SHORT>
__device__ __forceinline__ void pw_apply(pw_cop sops, const int* rpl, const int* opw, int s, const double* cur,
                                         double* nxt, PwPre& f0, PwPre& f1) {
  const int t = threadIdx.x;
  pw_settle(f0);
  if (TWO_ROWS) pw_settle(f1);
  s = pw_sgpr(s);  // the same on every lane: descriptors come through scalar loads
  const PwOp o = pw_op(sops, s);
  const int rows = o.rows;
  const int K = SHORT ? pw_sgpr(opw[s]) : PW_PF;
  double y0 = 0.0, y1 = 0.0;
  if (t < rows) y0 = pw_row<SHORT>(o, f0, t, cur, K);
  if (TWO_ROWS && t + PW_THREADS < rows) y1 = pw_row<SHORT>(o, f1, t + PW_THREADS, cur, K);
  // (operators 1 and 0 reload operator 0: unused, keeps the loads unconditional)
  const PwOp o2 = pw_op(sops, max(s - 2, 0));
  pw_fetch<RP_LDS, SHORT>(o2, rpl, t, f0);
  if (TWO_ROWS) pw_fetch<RP_LDS, SHORT>(o2, rpl, t + PW_THREADS, f1);
  if (t < rows) nxt[t] = y0;
  if (TWO_ROWS && t + PW_THREADS < rows) nxt[t + PW_THREADS] = y1;
  pw_lds_barrier();
}

// out[0] = lambda, out[1] = flag (iterations, or -1), out[2] = status
// (0 ok, 1 zero-norm vector, 2 A x == 0)
// One chain per workgroup: workgroup b runs jobs[b] (independent chains, e.g.
// the L and R norms of one PALM factor update, share a launch).  A chain has
// at most PW_MAX_OPS operators.
struct PwJob {
  const PwOp* ops;
  int nops;
  int n;
  const double* x0;
  double* out;
};

// The rounds of one chain (the reference's loop, faust_linear_algebra.hpp:
// 808-898): normalise xa into xn, apply the operators last to first, Rayleigh
// quotient.  Instantiated for SHORT chains (every operator sparse, rows of at
// most PW_PF entries: no loops over entries, so nothing but the prefetch is
// in flight across the operator barriers) and for the general case.
template <bool RP_LDS, bool TWO_ROWS, bool SHORT>
__device__ __forceinline__ void pw_rounds(pw_cop sops, const int* rpl, const int* opw, int nops, int n, int maxit,
                                          double thr,
                                          double* xa, double* xb, double* xn, double* red, double* tot,
                                          double& lambda, int& it, int& status) {
  const int t = threadIdx.x;
  double lambda_old = 1.0;
  const double athr = fabs(thr);
  // entries of rows t and t + PW_THREADS (rows <= PW_VMAX = 2 x PW_THREADS) of
  // the operators applied 1st, 3rd, ... (a) and 2nd, 4th, ... (b)
  PwPre a0, a1, b0, b1;
  while ((fabs(lambda_old - lambda) > athr || fabs(lambda) <= athr) && it < maxit) {
    it++;
    lambda_old = lambda;
    double nrm = sqrt(pw_dot(xa, xa, n, red, tot));
    if (nrm == 0.0) {
      status = 1;
      break;
    }
    pw_fetch<RP_LDS, SHORT>(pw_op(sops, nops - 1), rpl, t, a0);
    if (TWO_ROWS) pw_fetch<RP_LDS, SHORT>(pw_op(sops, nops - 1), rpl, t + PW_THREADS, a1);
    pw_fetch<RP_LDS, SHORT>(pw_op(sops, max(nops - 2, 0)), rpl, t, b0);
    if (TWO_ROWS) pw_fetch<RP_LDS, SHORT>(pw_op(sops, max(nops - 2, 0)), rpl, t + PW_THREADS, b1);
    const double inv = 1 / nrm;
    for (int i = t; i < n; i += PW_THREADS) xn[i] = xa[i] * inv;
    pw_lds_barrier();
    // apply ops last to first, ping-pong between xb and xa (xn stays the
    // normalised start vector)
    const double* cur = xn;
    double* nxt = xb;
    int len = n;
    for (int s = nops - 1; s >= 0; s -= 2) {
      pw_apply<RP_LDS, TWO_ROWS, SHORT>(sops, rpl, opw, s, cur, nxt, a0, a1);
      len = pw_op(sops, s).rows;
      cur = nxt;
      nxt = (nxt == xb) ? xa : xb;
      if (s == 0) break;
      pw_apply<RP_LDS, TWO_ROWS, SHORT>(sops, rpl, opw, s - 1, cur, nxt, b0, b1);
      len = pw_op(sops, s - 1).rows;
      cur = nxt;
      nxt = (nxt == xb) ? xa : xb;
    }
    // result vector is `cur`; move it into xa if needed
    if (cur != xa) {
      for (int i = t; i < len; i += PW_THREADS) xa[i] = cur[i];
      __syncthreads();
    }
    int nz = 0;
    for (int i = t; i < n; i += PW_THREADS) nz |= (xa[i] != 0.0);
    if (!__syncthreads_or(nz)) {
      status = 2;
      break;
    }
    lambda = pw_dot(xn, xa, n, red, tot);
  }
}

template <bool RP_LDS, bool TWO_ROWS>
__global__ __launch_bounds__(PW_THREADS) void k_power_iteration(const PwJob* __restrict__ jobs, int maxit,
                                                                 double thr) {
  extern __shared__ int rpl[];  // cached row pointers (PwOp::rpo)
  const PwJob job = jobs[blockIdx.x];
  const int nops = job.nops, n = job.n;
  const double* __restrict__ x0 = job.x0;
  double* __restrict__ out = job.out;
  __shared__ double xa[PW_VMAX], xb[PW_VMAX], xn[PW_VMAX];
  __shared__ double red[RED_LANES];
  __shared__ double tot;
  // operator descriptors: read-only and indexed by loop counters, so they
  // come through scalar loads
  const pw_cop sops = (pw_cop)job.ops;
  const int t = threadIdx.x;
  for (int i = t; i < n; i += PW_THREADS) xa[i] = x0[i];
  // copy the row pointers, find each operator's longest row (opw) and whether
  // every operator is sparse with rows of at most PW_PF entries
  __shared__ int opw[PW_MAX_OPS];
  for (int s = t; s < nops; s += PW_THREADS) opw[s] = 0;
  __syncthreads();
  int wide_row = 0;
  for (int s = 0; s < nops; ++s) {
    const PwOp o = pw_op(sops, s);
    if (o.kind != 1) {
      wide_row = 1;
      continue;
    }
    int w = 0;
    for (int i = t; i <= o.rows; i += PW_THREADS) {
      const int q = o.rp[i];
      if (RP_LDS) rpl[o.rpo + i] = q;
      if (i < o.rows) w = max(w, o.rp[i + 1] - q);
    }
    wide_row |= w > PW_PF;
    if (w > 0) atomicMax(&opw[s], w);
  }
  const bool short_chain = !__syncthreads_or(wide_row);
  double lambda = 0.0;
  int it = 0;
  int status = 0;
  if (short_chain)
    pw_rounds<RP_LDS, TWO_ROWS, true>(sops, rpl, opw, nops, n, maxit, thr, xa, xb, xn, red, &tot, lambda, it,
                                      status);
  else
    pw_rounds<RP_LDS, TWO_ROWS, false>(sops, rpl, opw, nops, n, maxit, thr, xa, xb, xn, red, &tot, lambda, it,
                                       status);
  if (t == 0) {
    out[0] = (status == 2) ? 0.0 : lambda;
    out[1] = (it < maxit) ? (double)it : -1.0;
    out[2] = (double)status;
  }
}

// ---------------------------------------------------------------------------
// LDS form: chains whose operators all fit one workgroup's LDS (at most 1024
// rows each), one workgroup per chain like the persistent form, and the same
// bits.  That form waits on global loads, on scalar loads of the operator
// descriptors and on barriers of 16 waves whatever the chain; here every
// entry is staged once, a workgroup has only as many waves as the longest
// vector needs (one for up to 64, where no barrier is left), and a round's
// two sums (the Rayleigh quotient and the next round's squared norm) share one
// reduction, whose last six levels are lane permutes in registers.
//
// Staged layout: a sparse operator's entry q of row r at [q][r] (values, then
// the columns of all operators behind them), so the 64 rows of a wave read
// consecutive words; rows shorter than the operator's width are padded with
// value -0 and the column of a slot that always holds +0, and adding -0
// changes no bit of an fma chain.  A dense operator's row r, column q is at
// [q][r] and needs no columns.  Rows of up to four entries are read into
// registers while the operator before is computed.
// Measured on the hierarchy of the Hadamard matrix of order 64 (10 iterations
// per PALM4MSA, 300 launches of one or two chains of 2 to 10 operators): mean
// 339 -> 104 us per launch (medians 52 with one chain, 18 with two: most of
// those converge early), 168 -> 99 ms in all by this form alone.  Norms of chains of random
// factors, us per call: 5 factors of 64^2 with 2 entries per row 374 -> 132,
// 2 of 64^2 with 32 entries 1920 -> 454, a dense 64^2 one 1037 -> 199.
constexpr int PL_MAX_OPS = 36;             // operators per chain (both chains' descriptors are kernel arguments)
constexpr int PL_ROWS = 1024;              // longest vector
constexpr int PL_LDS_BYTES = 152 * 1024;   // dynamic LDS (operators and the three vectors)

struct PlOp {
  const int* rp;    // sparse: row pointers, columns; dense: unused
  const int* ci;
  const double* v;  // sparse values or dense data
  int kind, trans;  // as PwOp
  int rows, cols;
  int width;        // staged entries per row (sparse: the widest row, rounded up to 2)
  int lda;
};
struct PlJob {
  PlOp ops[PL_MAX_OPS];
  int nops, n;
  int ld;    // vector slots: the longest vector + 1, the last one always +0
  int nval;  // staged values of all operators
};
struct PlArgs {
  PlJob job[2];
};

__device__ __forceinline__ double pl_bits(unsigned lo, unsigned hi) {
  return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}
// x of lane l + H in lane l (the lanes that the halving tree still uses)
template <int H>
__device__ __forceinline__ double pl_down(double x) {
  const unsigned long long u = __builtin_bit_cast(unsigned long long, x);
  const unsigned lo = (unsigned)u, hi = (unsigned)(u >> 32);
  if constexpr (H == 32) {
    return pl_bits(__builtin_amdgcn_permlane32_swap(lo, lo, false, false)[1],
                   __builtin_amdgcn_permlane32_swap(hi, hi, false, false)[1]);
  } else if constexpr (H == 16) {
    return pl_bits(__builtin_amdgcn_permlane16_swap(lo, lo, false, false)[1],
                   __builtin_amdgcn_permlane16_swap(hi, hi, false, false)[1]);
  } else {  // row_shl:H
    return pl_bits((unsigned)__builtin_amdgcn_update_dpp(0, (int)lo, 0x100 + H, 0xf, 0xf, true),
                   (unsigned)__builtin_amdgcn_update_dpp(0, (int)hi, 0x100 + H, 0xf, 0xf, true));
  }
}
// lane 0: the halving tree over the wave's 64 values; the same on every lane after
__device__ __forceinline__ double pl_tree(double v) {
  v = v + pl_down<32>(v);
  v = v + pl_down<16>(v);
  v = v + pl_down<8>(v);
  v = v + pl_down<4>(v);
  v = v + pl_down<2>(v);
  v = v + pl_down<1>(v);
  v = 0.0 + v;  // the chunk's sum added to the total
  const unsigned long long u = __builtin_bit_cast(unsigned long long, v);
  return pl_bits(__builtin_amdgcn_readfirstlane((unsigned)u), __builtin_amdgcn_readfirstlane((unsigned)(u >> 32)));
}

// canonical <x, y> and <y, y> over n <= 1024 values, and whether any y is not
// 0; xt, yt: this thread's values (0 past n), which are also in LDS (x, y).
template <int NT>
__device__ __forceinline__ void pl_sums(const double* x, const double* y, int n, double xt, double yt, double* red,
                                        int* flag, double& sxy, double& syy, int& any) {
  const int t = threadIdx.x, l = t & 63;
  double a = 0.0, b = 0.0;
  int nz = 0;
  if (NT <= 256) {  // one value per lane of the canonical 256
    a = fma(xt, yt, 0.0);
    b = fma(yt, yt, 0.0);
    nz = yt != 0.0;
  } else {
    __syncthreads();  // y complete
    if (t < RED_LANES)
#pragma unroll
      for (int m = 0; m < PL_ROWS / RED_LANES; ++m) {
        const int i = t + m * RED_LANES;
        if (i < n) {
          const double u = x[i], w = y[i];
          a = fma(u, w, a);
          b = fma(w, w, b);
          nz |= w != 0.0;
        }
      }
  }
  if (NT == 64) {
    any = __any(nz);
    sxy = pl_tree(a + 0.0);
    syy = pl_tree(b + 0.0);
    return;
  }
  constexpr int NW = NT < RED_LANES ? NT / 64 : RED_LANES / 64;
  const int wnz = __any(nz);
  if (t < 64 * NW) {
    red[t] = a;
    red[RED_LANES + t] = b;
    if (l == 0) flag[t >> 6] = wnz;
  }
  __syncthreads();
  // lane l of every wave: levels 128 and 64 of the tree (lanes past NT hold 0)
  if (NW == 2) {
    a = (red[l] + 0.0) + (red[l + 64] + 0.0);
    b = (red[RED_LANES + l] + 0.0) + (red[RED_LANES + l + 64] + 0.0);
    any = flag[0] | flag[1];
  } else {
    a = (red[l] + red[l + 128]) + (red[l + 64] + red[l + 192]);
    b = (red[RED_LANES + l] + red[RED_LANES + l + 128]) + (red[RED_LANES + l + 64] + red[RED_LANES + l + 192]);
    any = flag[0] | flag[1] | flag[2] | flag[3];
  }
  sxy = pl_tree(a);
  syy = pl_tree(b);
}

struct PlPre {
  double v[4];
  int c[4];
};

template <int NT>
__global__ __launch_bounds__(NT) void k_power_lds(PlArgs args, const double* __restrict__ x0, int maxit, double thr,
                                                  double* __restrict__ out) {
  extern __shared__ double lds[];  // values, three vectors, columns
  __shared__ double red[2 * RED_LANES];
  __shared__ int flag[4];
  __shared__ int4 desc[PL_MAX_OPS];  // per operator: rows, width (0: dense), first value, first column (dense: columns)
  const PlJob& job = args.job[blockIdx.x];
  const int t = threadIdx.x, nops = job.nops, n = job.n, ld = job.ld;
  double* const val = lds;
  double* vec = lds + job.nval;
  int* const col = reinterpret_cast<int*>(vec + 3 * ld);
  double *xn = vec, *b0 = vec + ld, *b1 = vec + 2 * ld;
  {
    int vo = 0, co = 0;
    for (int s = 0; s < nops; ++s) {
      const PlOp o = job.ops[s];
      const bool sp = o.kind == 1;
      if (t == 0) desc[s] = make_int4(o.rows, sp ? o.width : 0, vo, sp ? co : o.cols);
      if (t < o.rows) {
        if (sp) {
          const int p0 = o.rp[t], len = o.rp[t + 1] - p0;
          for (int q = 0; q < o.width; ++q) {
            const bool on = q < len;
            const int p = on ? p0 + q : 0;
            const double w = o.v[p];
            const int c = o.ci[p];
            val[vo + q * o.rows + t] = on ? w : -0.0;
            col[co + q * o.rows + t] = on ? c : ld - 1;
          }
        } else {
          const double* a = o.trans ? o.v + (size_t)t * o.lda : o.v + t;
          const size_t st = o.trans ? 1 : (size_t)o.lda;
#pragma unroll 8
          for (int q = 0; q < o.cols; ++q) val[vo + q * o.rows + t] = a[q * st];
        }
      }
      vo += o.rows * (sp ? o.width : o.cols);
      co += sp ? o.rows * o.width : 0;
    }
  }
  if (t < 3) vec[t * ld + ld - 1] = 0.0;
  double xt = t < n ? x0[t] : 0.0;
  if (t < n) b0[t] = xt;
  __syncthreads();
  // entries of row t of operator s, when its rows have at most four
  auto fetch = [&](const int4 d, PlPre& f) {
    const int r = min(t, d.x - 1), w = d.y;
    if (w == 0 || w > 4) return;
    const double* v = val + d.z + r;
    const int* c = col + d.w + r;
#pragma unroll
    for (int q = 0; q < 2; ++q) {
      f.v[q] = v[q * d.x];
      f.c[q] = c[q * d.x];
    }
    if (w > 2)
#pragma unroll
      for (int q = 2; q < 4; ++q) {
        f.v[q] = v[q * d.x];
        f.c[q] = c[q * d.x];
      }
  };
  auto row = [&](const int4 d, const PlPre& f, const double* cur) {
    const int w = d.y;
    double acc = 0.0;
    if (w == 0) {
      const double* v = val + d.z + t;
      const int cols = d.w;
      int q = 0;
      for (; q + 8 <= cols; q += 8) {
        double m[8], x[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
          m[u] = v[(q + u) * d.x];
          x[u] = cur[q + u];
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) acc = fma(m[u], x[u], acc);
      }
      for (; q < cols; ++q) acc = fma(v[q * d.x], cur[q], acc);
      return acc;
    }
    if (w <= 4) {
      const double y0 = cur[f.c[0]], y1 = cur[f.c[1]];
      if (w > 2) {
        const double y2 = cur[f.c[2]], y3 = cur[f.c[3]];
        acc = fma(f.v[1], y1, fma(f.v[0], y0, acc));
        return fma(f.v[3], y3, fma(f.v[2], y2, acc));
      }
      return fma(f.v[1], y1, fma(f.v[0], y0, acc));
    }
    const double* v = val + d.z + t;
    const int* c = col + d.w + t;
    int q = 0;
    for (; q + 8 <= w; q += 8) {
      int k[8];
      double m[8], x[8];
#pragma unroll
      for (int u = 0; u < 8; ++u) {
        k[u] = c[(q + u) * d.x];
        m[u] = v[(q + u) * d.x];
      }
#pragma unroll
      for (int u = 0; u < 8; ++u) x[u] = cur[k[u]];
#pragma unroll
      for (int u = 0; u < 8; ++u) acc = fma(m[u], x[u], acc);
    }
    for (; q < w; q += 2) {  // widths are even
      const int k0 = c[q * d.x], k1 = c[(q + 1) * d.x];
      const double m0 = v[q * d.x], m1 = v[(q + 1) * d.x];
      const double x0v = cur[k0], x1v = cur[k1];
      acc = fma(m1, x1v, fma(m0, x0v, acc));
    }
    return acc;
  };
  // lane s of every wave keeps operator s's descriptor
  const int4 dl = desc[min(t & 63, nops - 1)];
  auto get = [&](int s) {
    return make_int4(__builtin_amdgcn_readlane(dl.x, s), __builtin_amdgcn_readlane(dl.y, s),
                     __builtin_amdgcn_readlane(dl.z, s), __builtin_amdgcn_readlane(dl.w, s));
  };
  double lambda = 0.0, lambda_old = 1.0, sxy = 0.0, syy;
  int it = 0, status = 0, any = 1;
  pl_sums<NT>(b0, b0, n, xt, xt, red, flag, sxy, syy, any);
  double yt = xt;  // the current vector's value, unnormalised
  const double athr = fabs(thr);
  PlPre f0, f1;
  while ((fabs(lambda_old - lambda) > athr || fabs(lambda) <= athr) && it < maxit) {
    it++;
    lambda_old = lambda;
    const double nrm = sqrt(syy);
    if (nrm == 0.0) {
      status = 1;
      break;
    }
    int4 d = get(nops - 1);
    fetch(d, f0);
    const double inv = 1 / nrm;
    xt = yt * inv;  // yt is +0 past n, inv finite or not: the lanes past n are not stored
    if (t < n) xn[t] = xt;
    __syncthreads();
    const double* cur = xn;
    double* nxt = b0;
    for (int s = nops - 1; s >= 0; --s) {
      const int4 dn = get(max(s - 1, 0));
      if (s > 0) fetch(dn, f1);
      yt = 0.0;
      if (t < d.x) {
        yt = row(d, f0, cur);
        nxt[t] = yt;
      }
      if (s > 0) __syncthreads();
      cur = nxt;
      nxt = nxt == b0 ? b1 : b0;
      d = dn;
      f0 = f1;
    }
    if (t >= n) {
      yt = 0.0;
      xt = 0.0;
    }
    pl_sums<NT>(xn, cur, n, xt, yt, red, flag, sxy, syy, any);
    if (!any) {
      status = 2;
      break;
    }
    lambda = sxy;
  }
  if (t == 0) {
    double* o = out + 3 * blockIdx.x;
    o[0] = (status == 2) ? 0.0 : lambda;
    o[1] = (it < maxit) ? (double)it : -1.0;
    o[2] = (double)status;
  }
}

// ---------------------------------------------------------------------------
// Wide form: one launch per operator per round, for chains whose operators are
// too large for a single CU to stream every round.  Each row is still one fma
// chain on one lane (k ascending), so the result is bit-identical to the
// persistent kernel; the row data is staged through LDS by all 256 threads of
// the workgroup in contiguous chunks, and the first R lanes (one per row) run
// the chains.  A round's boundary (the zero test, the Rayleigh quotient, the
// loop test and the normalisation) runs at the start of its first operator's
// launch, in every workgroup alike and while that operator's first entries are
// on their way; workgroup 0 stores what the next round needs.  A device state
// carries lambda, the round count and a done flag (two copies: a round reads
// one and writes the other, so no workgroup reads what another one writes);
// the host enqueues rounds ahead and launches after convergence return at once.
struct PwState {
  double lambda, lambda_old;
  int it, status, done, pad;
};

constexpr int PW_WIDE_THREADS = 256;
constexpr int PW_CH = 2048;  // entries per LDS chunk of a sparse operator

// A round boundary: xa = the chain's output (first round: the start vector,
// mode 0), xn_in = the vector it was applied to, xn_out = its successor.
// Used when first; res (host memory) receives lambda, flag, status, done.
struct PwBound {
  int first, mode, n, maxit;
  double thr;
  const double* xa;
  const double* xn_in;
  double* xn_out;
  const PwState* in;
  PwState* out;
  double* res;
};

__device__ __forceinline__ void pw_post(const PwState& st, int maxit, double* res) {
  res[0] = st.status == 2 ? 0.0 : st.lambda;
  res[1] = st.it < maxit ? (double)st.it : -1.0;
  res[2] = (double)st.status;
  res[3] = 1.0;
}

// The boundary in a workgroup of 256 threads; lead: this one stores the
// results.  Writes the normalised vector to xs (LDS) and returns true, or
// returns false when the iteration is over.  red: 512 doubles, flag: 4 ints of LDS.
__device__ __forceinline__ bool pw_bound(const PwBound& b, bool lead, double* xs, double* red, int* flag) {
  const int t = threadIdx.x, l = t & 63;
  PwState st = *b.in;
  if (!st.done) {
    double sxy = 0.0, syy = 0.0;
    int nz = 0;
    for (int i = t; i < b.n; i += RED_LANES) {
      const double y = b.xa[i], x = b.mode ? b.xn_in[i] : 0.0;
      xs[i] = y;
      sxy = fma(x, y, sxy);
      syy = fma(y, y, syy);
      nz |= y != 0.0;
    }
    const int any_w = __any(nz);
    red[t] = sxy;
    red[RED_LANES + t] = syy;
    if (l == 0) flag[t >> 6] = any_w;
    __syncthreads();
    sxy = pl_tree((red[l] + red[l + 128]) + (red[l + 64] + red[l + 192]));
    syy = pl_tree((red[RED_LANES + l] + red[RED_LANES + l + 128]) + (red[RED_LANES + l + 64] + red[RED_LANES + l + 192]));
    const int any = flag[0] | flag[1] | flag[2] | flag[3];
    if (b.mode && !any) {
      st.status = 2;
      st.done = 1;
    } else {
      const double lambda = b.mode ? sxy : st.lambda;
      const double athr = fabs(b.thr);
      st.lambda = lambda;
      if (!((fabs(st.lambda_old - lambda) > athr || fabs(lambda) <= athr) && st.it < b.maxit)) {
        st.done = 1;
      } else {
        st.it++;
        st.lambda_old = lambda;
        const double nrm = sqrt(syy);
        if (nrm == 0.0) {
          st.status = 1;
          st.done = 1;
        } else {
          const double inv = 1 / nrm;
          for (int i = t; i < b.n; i += RED_LANES) {
            const double x = xs[i] * inv;
            xs[i] = x;
            if (lead) b.xn_out[i] = x;
          }
        }
      }
    }
    if (lead && t == 0 && st.done) pw_post(st, b.maxit, b.res);
  }
  if (lead && t == 0) *b.out = st;
  return !st.done;
}

// sparse rows (row pointers rp, indices ci, values v): rows r0..r0+R-1 per workgroup
__global__ __launch_bounds__(PW_WIDE_THREADS) void k_pw_csr(const int* __restrict__ rp, const int* __restrict__ ci,
                                                            const double* __restrict__ v, int rows, int cols, int R,
                                                            const double* __restrict__ cur, double* __restrict__ nxt,
                                                            const PwState* __restrict__ s, PwBound bound) {
  __shared__ double xs[PW_VMAX];
  __shared__ double sv[PW_CH];
  __shared__ int sci[PW_CH];
  __shared__ double red[2 * RED_LANES];
  __shared__ int flag[4];
  const int t = threadIdx.x;
  if (bound.first) {
    if (!pw_bound(bound, blockIdx.x == 0, xs, red, flag)) return;
  } else {
    if (s->done) return;
    for (int i = t; i < cols; i += PW_WIDE_THREADS) xs[i] = cur[i];
  }
  const int r0 = blockIdx.x * R, r1 = min(rows, r0 + R), nr = r1 - r0;
  const int p0 = rp[r0], p1 = rp[r1];
  int p = 0, pe = 0;
  if (t < nr) {
    p = rp[r0 + t];
    pe = rp[r0 + t + 1];
  }
  double acc = 0.0;
  for (int c0 = p0; c0 < p1; c0 += PW_CH) {
    const int c1 = min(p1, c0 + PW_CH);
    __syncthreads();  // previous chunk consumed; xs staged before the first
    for (int q = c0 + t; q < c1; q += PW_WIDE_THREADS) {
      sv[q - c0] = v[q];
      sci[q - c0] = ci[q];
    }
    __syncthreads();
    if (t < nr) {
      const int e = min(pe, c1);
      for (; p < e; ++p) acc = fma(sv[p - c0], xs[sci[p - c0]], acc);
    }
  }
  if (t < nr) nxt[r0 + t] = acc;
}

// dense op(A) rows (A column-major, leading dimension lda); TRANS: op(A) = A^T.
// A workgroup computes four rows.  Its entries come in chunks of 1024 columns,
// 16 loads per thread issued together; they go to LDS in four parts of 256
// columns, each followed by a barrier, and the first wave runs the four chains
// over one part while the others store the next as it arrives.  Workgroups
// are dealt to the XCDs in turn, so each XCD takes a contiguous run of rows:
// the four workgroups that share the 128-byte lines of a column find them in
// one L2.  The floor is the chain: 1024 dependent fma, 2.7 us; its lanes read
// pairs of columns 16 ahead, since waiting for each 16 took as long again.
// Measured per launch in chains of 20 operators of order 1024 (8 MiB each):
// 23 us with loads of one entry at a time, 14.2 with the parts above, 10.2
// with the lanes reading ahead; order 256 (PALM4MSA's step sizes): 5.4 us and
// a boundary launch of 3.8 us per round -> 4.9 us and none.
constexpr int PD_ROWS = 4, PD_PARTS = 4, PD_PCOLS = 256, PD_COLS = PD_PARTS * PD_PCOLS, PD_LD = PD_PCOLS + 2;
constexpr int PD_LOADS = PD_ROWS * PD_PCOLS / PW_WIDE_THREADS;  // per thread and part
template <bool TRANS>
__global__ __launch_bounds__(PW_WIDE_THREADS) void k_pw_dense(const double* __restrict__ A, int lda, int rows,
                                                              int cols, const double* __restrict__ cur,
                                                              double* __restrict__ nxt,
                                                              const PwState* __restrict__ s, PwBound bound) {
  __shared__ __align__(16) double xs[PW_VMAX];
  __shared__ __align__(16) double tile[PD_PARTS][PD_ROWS * PD_LD];  // [row][column]
  __shared__ double red[2 * RED_LANES];
  __shared__ int flag[4];
  const int t = threadIdx.x;
  const int rb = (blockIdx.x & 7) * (int)(gridDim.x >> 3) + (blockIdx.x >> 3);
  const int r0 = rb * PD_ROWS, nr = min(rows - r0, PD_ROWS);
  if (nr <= 0) return;  // the grid is a multiple of 8
  double x[PD_PARTS][PD_LOADS];
  // entry u of this thread in a part: its row and column there
  auto at = [&](int u, int& i, int& c) {
    const int e = t + PW_WIDE_THREADS * u;
    i = TRANS ? e / PD_PCOLS : e % PD_ROWS;
    c = TRANS ? e % PD_PCOLS : e / PD_ROWS;
  };
  auto fetch = [&](int c0, double (&v)[PD_LOADS]) {
#pragma unroll
    for (int u = 0; u < PD_LOADS; ++u) {
      int i, c;
      at(u, i, c);
      const int r = min(r0 + i, rows - 1), k = min(c0 + c, cols - 1);  // entries past the end are not used
      v[u] = TRANS ? A[(size_t)r * lda + k] : A[(size_t)k * lda + r];
    }
  };
#pragma unroll
  for (int j = 0; j < PD_PARTS; ++j) fetch(j * PD_PCOLS, x[j]);
  if (bound.first) {
    if (!pw_bound(bound, rb == 0, xs, red, flag)) return;
  } else {
    if (s->done) return;
    for (int i = t; i < cols; i += PW_WIDE_THREADS) xs[i] = cur[i];
  }
  double acc = 0.0;
  for (int c0 = 0; c0 < cols; c0 += PD_COLS) {
#pragma unroll
    for (int j = 0; j < PD_PARTS; ++j) {
      const int p0 = c0 + j * PD_PCOLS;
      if (p0 < cols) {  // the same for the whole workgroup
        // this part of the tile was last read before the previous part's barrier
#pragma unroll
        for (int u = 0; u < PD_LOADS; ++u) {
          int i, c;
          at(u, i, c);
          tile[j][i * PD_LD + c] = x[j][u];
        }
        if (p0 + PD_COLS < cols) fetch(p0 + PD_COLS, x[j]);
        __syncthreads();
        if (t < PD_ROWS) {
          const int nc = min(PD_PCOLS, cols - p0);
          const pw_d2* m = reinterpret_cast<const pw_d2*>(tile[j] + t * PD_LD);
          const pw_d2* xc = reinterpret_cast<const pw_d2*>(xs + p0);
          // 16 columns at a time, the next 16 on their way from LDS meanwhile
          // (reads past the part stay inside the arrays and are not used)
          pw_d2 a[2][8], y[2][8];
          auto load = [&](int c, pw_d2 (&la)[8], pw_d2 (&ly)[8]) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              la[u] = m[min(c, PD_PCOLS - 16) / 2 + u];
              ly[u] = xc[min(c, PD_PCOLS - 16) / 2 + u];
            }
          };
          auto mac = [&](const pw_d2 (&la)[8], const pw_d2 (&ly)[8]) {
#pragma unroll
            for (int u = 0; u < 8; ++u) {
              acc = fma(la[u].x, ly[u].x, acc);
              acc = fma(la[u].y, ly[u].y, acc);
            }
          };
          load(0, a[0], y[0]);
          int c = 0;
          for (; c + 32 <= nc; c += 32) {
            load(c + 16, a[1], y[1]);
            __builtin_amdgcn_sched_barrier(0);
            mac(a[0], y[0]);
            __builtin_amdgcn_sched_barrier(0);
            load(c + 32, a[0], y[0]);
            __builtin_amdgcn_sched_barrier(0);
            mac(a[1], y[1]);
            __builtin_amdgcn_sched_barrier(0);
          }
          const double* ms = tile[j] + t * PD_LD;
          for (; c < nc; ++c) acc = fma(ms[c], xs[p0 + c], acc);
        }
      }
    }
  }
  if (t < nr) nxt[r0 + t] = acc;
}

// Operators with more than PW_VMAX columns: x read from global memory (the
// L2 holds it), one row per thread, the same fma chain per row.
__global__ __launch_bounds__(PW_WIDE_THREADS) void k_pw_csr_g(const int* __restrict__ rp, const int* __restrict__ ci,
                                                              const double* __restrict__ v, int rows,
                                                              const double* __restrict__ cur,
                                                              double* __restrict__ nxt,
                                                              const PwState* __restrict__ s) {
  if (s->done) return;
  const int r = blockIdx.x * PW_WIDE_THREADS + threadIdx.x;
  if (r >= rows) return;
  double acc = 0.0;
  for (int p = rp[r], pe = rp[r + 1]; p < pe; ++p) acc = fma(v[p], cur[ci[p]], acc);
  nxt[r] = acc;
}

__global__ __launch_bounds__(PW_WIDE_THREADS) void k_pw_dense_g(const double* __restrict__ A, int lda, int trans,
                                                                int rows, int cols, const double* __restrict__ cur,
                                                                double* __restrict__ nxt,
                                                                const PwState* __restrict__ s) {
  if (s->done) return;
  const int r = blockIdx.x * PW_WIDE_THREADS + threadIdx.x;
  if (r >= rows) return;
  double acc = 0.0;
  if (trans) {  // row r of A^T = column r of A
    const double* col = A + (size_t)r * lda;
    for (int c = 0; c < cols; ++c) acc = fma(col[c], cur[c], acc);
  } else {
    for (int c = 0; c < cols; ++c) acc = fma(A[(size_t)c * lda + r], cur[c], acc);
  }
  nxt[r] = acc;
}

// A boundary of its own: in front of an operator that reads x from global
// memory, and after the last round (which only evaluates the loop test).
__global__ __launch_bounds__(PW_THREADS) void k_pw_step(PwBound b) {
  __shared__ double red[RED_LANES];
  __shared__ double tot;
  const int t = threadIdx.x;
  PwState st = *b.in;
  if (st.done) {
    if (t == 0) *b.out = st;
    return;
  }
  if (b.mode == 1) {
    int nz = 0;
    for (int i = t; i < b.n; i += PW_THREADS) nz |= (b.xa[i] != 0.0);
    if (!__syncthreads_or(nz)) {
      st.status = 2;
      st.done = 1;
    } else {
      st.lambda = pw_dot(b.xn_in, b.xa, b.n, red, &tot);
    }
  }
  if (!st.done) {
    const double athr = fabs(b.thr);
    if (!((fabs(st.lambda_old - st.lambda) > athr || fabs(st.lambda) <= athr) && st.it < b.maxit)) {
      st.done = 1;
    } else {
      st.it++;
      st.lambda_old = st.lambda;
      const double nrm = sqrt(pw_dot(b.xa, b.xa, b.n, red, &tot));
      if (nrm == 0.0) {
        st.status = 1;
        st.done = 1;
      } else {
        const double inv = 1 / nrm;
        for (int i = t; i < b.n; i += PW_THREADS) b.xn_out[i] = b.xa[i] * inv;
      }
    }
  }
  if (t == 0) {
    if (st.done) pw_post(st, b.maxit, b.res);
    *b.out = st;
  }
}

__global__ void k_pw_init(PwState* __restrict__ s) {
  if (threadIdx.x == 0) {
    s->lambda = 0.0;
    s->lambda_old = 1.0;
    s->it = 0;
    s->status = 0;
    s->done = 0;
    s->pad = 0;
  }
}

const std::vector<double>& power_x0(int n) {
  static std::mutex mu;
  static std::map<int, std::vector<double>> cache;
  std::lock_guard<std::mutex> lk(mu);
  auto it = cache.find(n);
  if (it != cache.end()) return it->second;
  // srand(0xF4+'u'+57); Eigen::Matrix::Random: x + (y-x)*Scalar(std::rand())/Scalar(RAND_MAX) on [-1, 1]
  srand(0xF4 + 'u' + 57);
  std::vector<double> x(n);
  for (int i = 0; i < n; ++i) x[i] = -1.0 + (2.0 * (double)std::rand()) / (double)RAND_MAX;
  return cache.emplace(n, std::move(x)).first->second;
}

// start vector on the device: power_x0(PL_ROWS), whose first n values are
// power_x0(n) for every n (one random sequence), uploaded once per device
static const double* pl_x0() {
  constexpr int kMaxDevices = 64;
  static std::mutex mu;
  static double* dx[kMaxDevices] = {};
  int dev = 0;
  FH_HIP(hipGetDevice(&dev));
  FH_CHECK(dev >= 0 && dev < kMaxDevices, "power_iteration: device index out of range");
  const std::vector<double>& x = power_x0(PL_ROWS);
  std::lock_guard<std::mutex> lk(mu);
  if (!dx[dev]) {
    // held to process end, and not a block of the pool: work queued on the
    // caller's stream may still use one, and this copy does not wait for it
    void* p = nullptr;
    FH_HIP(hipMalloc(&p, sizeof(double) * PL_ROWS));
    const hipError_t e = hipMemcpy(p, x.data(), sizeof(double) * PL_ROWS, hipMemcpyHostToDevice);
    if (e != hipSuccess) (void)hipFree(p);
    FH_HIP(e);
    dx[dev] = static_cast<double*>(p);
  }
  return dx[dev];
}

// Per-round time estimates (seconds).  The persistent kernel streams every
// operator through one CU (~100 GB/s), and an entry of a row longer than it
// loads ahead (PW_PF entries, or dense) is a dependent load: dense 90 ns (10.7
// us per operator of a 128 x 100 chain), sparse 75 ns while few rows are long,
// 120 to 200 ns by the number of rows when many are (more than 1000 entries
// beyond two per row), whose loads together get 12 GB/s.  The wide form pays a
// launch per operator but spreads the rows over the chip, leaving each row's
// fma chain as its floor: 4 ns per term of a dense row, 44 ns of a sparse one
// (the gather from LDS is in the chain); the rounds queued past the end and the
// host's waits come to 15%.  Of 160 chains of 1 to 10 factors of 128 to 2000
// rows all but two ran within 6% of the quicker form (those 13%).  us per
// round, persistent / wide, 5 factors of 1024 rows of 2: one row of 128 70 / 78; 64
// rows of 64 111 / 81; all rows of 20 163 / 62, of 8 60 / 54.
// FH_POWER_WIDE=0/1 forces a form.
static bool use_wide_form(const std::vector<PwOp>& h) {
  if (const char* e = getenv("FH_POWER_WIDE")) {
    if (e[0] == '0') return false;
    if (e[0] == '1') return true;
  }
  double single = 3e-6, wide = 1e-6;
  for (const PwOp& o : h) {
    const double entries = o.kind == 1 ? (double)o.nnz : (double)o.rows * o.cols;
    const bool sparse = o.kind == 1;
    const double bytes = entries * (sparse ? 12.0 : 8.0);
    const double row = sparse ? (o.width >= 0 ? o.width : entries / std::max(o.rows, 1)) : o.cols;
    single += bytes / 100e9 + 0.4e-6;
    if (row > PW_PF) {
      const double more = sparse ? entries - 2.0 * o.rows : 0.0;
      const double load = !sparse ? 90e-9 : more <= 1000.0 ? 75e-9 : o.rows <= 512 ? 120e-9 : o.rows <= 1024 ? 150e-9 : 200e-9;
      single += std::max(row * load, more * 12.0 / 12e9);
    }
    wide += 4e-6 + row * (sparse ? 44e-9 : 4e-9) + bytes / 3e12;
  }
  return 1.15 * wide < single;
}

static double power_iteration_wide(const std::vector<PwOp>& h, int n, const std::vector<double>& x0, int maxit,
                                   double thr, int* flag, hipStream_t st) {
  int vmax = n;
  for (const PwOp& o : h) vmax = std::max(vmax, std::max(o.rows, o.cols));
  // the chain's output and the normalised vector alternate between two halves:
  // a boundary reads the previous round's while its launch writes this one's
  DBuf xa(sizeof(double) * 2 * n), xn(sizeof(double) * 2 * n), b0(sizeof(double) * vmax), b1(sizeof(double) * vmax),
      ds(sizeof(PwState) * 2);
  PwState* dst = ds.as<PwState>();
  double* res = mail() + MAIL_POWER;
  res[3] = 0.0;  // set by the boundary that ends the iteration
  const double* start = xa.as<double>();
  if (n <= PL_ROWS)
    start = pl_x0();
  else
    FH_HIP(hipMemcpyAsync(xa.p, x0.data(), sizeof(double) * n, hipMemcpyHostToDevice, st));
  hipLaunchKernelGGL(k_pw_init, dim3(1), dim3(64), 0, st, dst);
  FH_LAUNCH_CHECK();
  const int nops = (int)h.size();
  const bool fused = h.back().cols <= PW_VMAX;  // the boundary runs in the first operator's launch
  int next_check = 4;
  PwBound b{};
  b.n = n;
  b.maxit = maxit;
  b.thr = thr;
  b.res = res;
  for (int round = 1; round <= maxit + 1; ++round) {
    b.mode = round > 1;
    b.xa = round > 1 ? xa.as<double>() + (size_t)((round - 1) & 1) * n : start;
    double* const xa_out = xa.as<double>() + (size_t)(round & 1) * n;
    b.xn_in = xn.as<double>() + (size_t)((round - 1) & 1) * n;
    b.xn_out = xn.as<double>() + (size_t)(round & 1) * n;
    b.in = dst + ((round - 1) & 1);
    b.out = dst + (round & 1);
    const bool last = round > maxit;  // every round ran: the loop test alone
    // the host looks whether the iteration is over before rounds 5, 13, ...:
    // their boundary is a launch of its own, so that it is decided by then
    const bool look = round - 1 == next_check;
    const bool alone = !fused || last || look;
    b.first = 0;
    if (alone) {
      hipLaunchKernelGGL(k_pw_step, dim3(1), dim3(PW_THREADS), 0, st, b);
      FH_LAUNCH_CHECK();
      if (last) break;
    }
    if (look) {
      FH_HIP(hipStreamSynchronize(st));
      if (res[3] != 0.0) break;
      next_check += 8;
    }
    const double* cur = b.xn_out;
    for (int s = nops - 1; s >= 0; --s) {
      const PwOp& o = h[s];
      b.first = !alone && s == nops - 1;
      double* out = (s == 0) ? xa_out : (((nops - 1 - s) & 1) ? b1.as<double>() : b0.as<double>());
      if (o.cols > PW_VMAX) {  // x does not fit LDS: read it from global memory
        const dim3 gg((o.rows + PW_WIDE_THREADS - 1) / PW_WIDE_THREADS);
        if (o.kind == 1)
          hipLaunchKernelGGL(k_pw_csr_g, gg, dim3(PW_WIDE_THREADS), 0, st, o.rp, o.ci, o.v, o.rows, cur, out,
                             (const PwState*)b.out);
        else
          hipLaunchKernelGGL(k_pw_dense_g, gg, dim3(PW_WIDE_THREADS), 0, st, o.v, o.lda, o.trans, o.rows, o.cols,
                             cur, out, (const PwState*)b.out);
      } else if (o.kind == 1) {
        int R = 1;
        while (R < 8 && (o.rows + 2 * R - 1) / (2 * R) >= 256) R *= 2;
        hipLaunchKernelGGL(k_pw_csr, dim3((o.rows + R - 1) / R), dim3(PW_WIDE_THREADS), 0, st, o.rp, o.ci, o.v,
                           o.rows, o.cols, R, cur, out, (const PwState*)b.out, b);
      } else {
        const int nb = (o.rows + PD_ROWS - 1) / PD_ROWS;
        const dim3 grid((unsigned)((nb + 7) / 8 * 8));
        if (o.trans)
          hipLaunchKernelGGL(k_pw_dense<true>, grid, dim3(PW_WIDE_THREADS), 0, st, o.v, o.lda, o.rows, o.cols, cur,
                             out, (const PwState*)b.out, b);
        else
          hipLaunchKernelGGL(k_pw_dense<false>, grid, dim3(PW_WIDE_THREADS), 0, st, o.v, o.lda, o.rows, o.cols, cur,
                             out, (const PwState*)b.out, b);
      }
      FH_LAUNCH_CHECK();
      cur = out;
    }
  }
  FH_HIP(hipStreamSynchronize(st));
  if (res[2] == 1.0) throw Error(FH_ERR_NUMERIC, "Can't normalize a zero-norm vector.");
  if (flag) *flag = (int)res[1];
  return res[0];
}

static std::vector<PwOp> pw_ops(const std::vector<ChainOp>& ops) {
  FH_CHECK(!ops.empty(), "power_iteration: empty chain");
  std::vector<PwOp> h(ops.size());
  for (size_t s = 0; s < ops.size(); ++s) {
    const DMat& M = *ops[s].M;
    const bool tr = ops[s].op != 'N';
    PwOp& o = h[s];
    o.rpo = -1;
    o.rows = tr ? M.n : M.m;
    o.cols = tr ? M.m : M.n;
    if (M.kind == K_CSR) {
      FH_CHECK(M.dtype == FH_F64, "power_iteration: FP64 dense or CSR factors only");
      o.kind = 1;
      o.trans = 0;
      o.lda = 0;
      o.nnz = M.nnz;
      o.width = tr ? M.max_col : M.max_row;
      if (tr) {
        FH_CHECK(M.has_csc, "power_iteration: CSC twin missing");
        o.rp = M.cp.as<int>();
        o.ci = M.ri.as<int>();
        o.v = M.cv.as<double>();
      } else {
        o.rp = M.rp.as<int>();
        o.ci = M.ci.as<int>();
        o.v = M.v.as<double>();
      }
    } else {
      FH_CHECK(M.kind == K_DENSE && M.dtype == FH_F64, "power_iteration: FP64 dense or CSR factors only");
      o.kind = 0;
      o.trans = tr ? 1 : 0;
      o.v = M.d.as<double>();
      // read (and unused) by the persistent kernel's unconditional loads
      o.rp = o.ci = reinterpret_cast<const int*>(o.v);
      o.lda = M.m;
      o.nnz = 0;
      o.width = -1;
    }
  }
  return h;
}

// the persistent kernel keeps every vector in LDS: up to PW_VMAX entries
static bool pw_persistent(const std::vector<PwOp>& h, int n) {
  bool fits = n <= PW_VMAX && h.size() <= (size_t)PW_MAX_OPS;
  for (const PwOp& o : h) fits = fits && o.rows >= 1 && o.rows <= PW_VMAX && o.cols <= PW_VMAX;
  return fits && !use_wide_form(h);
}

// Dynamic LDS the persistent kernel may take for row pointers: PW_RP_LDS
// once the attribute is granted, else none (every operator then reads its
// row pointers from global memory).  Queried once per process.
static size_t pw_rp_budget() {
  static int budget = -1;
  if (budget < 0)
    budget = hipFuncSetAttribute((const void*)k_power_iteration<true, false>,
                                 hipFuncAttributeMaxDynamicSharedMemorySize, PW_RP_LDS) == hipSuccess &&
                     hipFuncSetAttribute((const void*)k_power_iteration<true, true>,
                                         hipFuncAttributeMaxDynamicSharedMemorySize, PW_RP_LDS) == hipSuccess
                 ? PW_RP_LDS
                 : 0;
  (void)hipGetLastError();
  return (size_t)budget;
}

// Row-pointer copies of a chain's sparse operators in LDS (an array shared by
// two operators is copied once); returns the ints used, or -1 (and no
// copies) when they do not all fit the budget.
static long pw_assign_rp(std::vector<PwOp>& ops, size_t budget_ints) {
  size_t used = 0, maxrows = 0;
  for (size_t s = 0; s < ops.size(); ++s) {
    PwOp& o = ops[s];
    o.rpo = -1;
    maxrows = std::max(maxrows, (size_t)o.rows);
    if (o.kind != 1) {
      o.rpo = 0;  // a dense operator's (unused) row-pointer reads stay inside the array
      continue;
    }
    for (size_t q = 0; q < s; ++q)
      if (ops[q].kind == 1 && ops[q].rp == o.rp) o.rpo = ops[q].rpo;
    if (o.rpo >= 0) continue;
    o.rpo = (int)used;
    used += o.rows + 1;
  }
  used = std::max(used, maxrows + 1);
  if (used > budget_ints) {
    for (PwOp& o : ops) o.rpo = -1;
    return -1;
  }
  return (long)used;
}

// chains[k] (ops, n) in one launch, one workgroup each; lam[k] and flags[k]
// receive each chain's result.  A zero-norm start vector throws, for the
// first such chain in order.
static void power_iteration_persistent(const std::vector<std::vector<PwOp>>& hs_in, const std::vector<int>& ns,
                                       int maxit, double thr, double* lam, int* flags, hipStream_t st) {
  const int J = (int)hs_in.size();
  std::vector<std::vector<PwOp>> hs = hs_in;
  size_t nops = 0, nx = 0;
  long dyn_ints = 0;
  const size_t budget = pw_rp_budget() / sizeof(int);
  bool rp_lds = true;
  for (int k = 0; k < J; ++k) {
    nops += hs[k].size();
    nx += ns[k];
    const long used = pw_assign_rp(hs[k], budget);
    rp_lds = rp_lds && used >= 0;
    dyn_ints = std::max(dyn_ints, used);
  }
  if (!rp_lds) {
    for (auto& h : hs)
      for (PwOp& o : h) o.rpo = -1;
    dyn_ints = 0;
  }
  DBuf dops(sizeof(PwOp) * nops), dx(sizeof(double) * nx), dout(sizeof(double) * 3 * J), djobs(sizeof(PwJob) * J);
  std::vector<PwOp> allops;
  std::vector<PwJob> jobs(J);
  size_t oo = 0, ox = 0;
  for (int k = 0; k < J; ++k) {
    allops.insert(allops.end(), hs[k].begin(), hs[k].end());
    FH_HIP(hipMemcpyAsync(dx.as<double>() + ox, power_x0(ns[k]).data(), sizeof(double) * ns[k],
                          hipMemcpyHostToDevice, st));
    jobs[k] = PwJob{dops.as<PwOp>() + oo, (int)hs[k].size(), ns[k], dx.as<double>() + ox, dout.as<double>() + 3 * k};
    oo += hs[k].size();
    ox += ns[k];
  }
  FH_HIP(hipMemcpyAsync(dops.p, allops.data(), sizeof(PwOp) * nops, hipMemcpyHostToDevice, st));
  FH_HIP(hipMemcpyAsync(djobs.p, jobs.data(), sizeof(PwJob) * J, hipMemcpyHostToDevice, st));
  bool two = false;  // some vector or operator longer than one row per thread
  for (int k = 0; k < J; ++k) {
    two = two || ns[k] > PW_THREADS;
    for (const PwOp& o : hs[k]) two = two || o.rows > PW_THREADS;
  }
  const size_t dyn = rp_lds ? sizeof(int) * dyn_ints : 0;
  auto kern = rp_lds ? (two ? k_power_iteration<true, true> : k_power_iteration<true, false>)
                     : (two ? k_power_iteration<false, true> : k_power_iteration<false, false>);
  hipLaunchKernelGGL(kern, dim3(J), dim3(PW_THREADS), dyn, st, djobs.as<PwJob>(), maxit, thr);
  FH_LAUNCH_CHECK();
  std::vector<double> res(3 * J);
  FH_HIP(hipMemcpyAsync(res.data(), dout.p, sizeof(double) * 3 * J, hipMemcpyDeviceToHost, st));
  FH_HIP(hipStreamSynchronize(st));
  for (int k = 0; k < J; ++k) {
    if (res[3 * k + 2] == 1.0) throw Error(FH_ERR_NUMERIC, "Can't normalize a zero-norm vector.");
    lam[k] = res[3 * k];
    flags[k] = (int)res[3 * k + 1];
  }
}

// the LDS form's job for a chain, when it fits: every operator dense or of
// known width, at most PL_ROWS rows and columns, all entries in PL_LDS_BYTES;
// lds receives the bytes.  No estimate decides between this form and the wide
// one: over the dense and sparse chains that fit it took 1/1.8 to 1/4 of the
// others' best, and lost only with few long rows (dense 4 x 1024: 1681 us per
// norm against 1457 wide; 128^2 with one row of 128 entries: 568 against 532
// persistent).
static bool pl_job(const std::vector<PwOp>& h, int n, PlJob& j, size_t* lds) {
  if (getenv("FH_POWER_WIDE")) return false;  // one of the other forms is asked for
  if (h.empty() || h.size() > (size_t)PL_MAX_OPS || n < 1 || n > PL_ROWS) return false;
  int longest = n;
  size_t nval = 0, ncol = 0;
  for (size_t s = 0; s < h.size(); ++s) {
    const PwOp& o = h[s];
    if (o.rows < 1 || o.cols < 1 || o.rows > PL_ROWS || o.cols > PL_ROWS || (o.kind == 1 && o.width < 0)) return false;
    longest = std::max({longest, o.rows, o.cols});
    const int w = o.kind == 1 ? std::max(2, (o.width + 1) & ~1) : o.cols;
    nval += (size_t)o.rows * w;
    if (o.kind == 1) ncol += (size_t)o.rows * w;
    j.ops[s] = PlOp{o.rp, o.ci, o.v, o.kind, o.trans, o.rows, o.cols, w, o.lda};
  }
  j.nops = (int)h.size();
  j.n = n;
  j.ld = longest + 1;
  *lds = sizeof(double) * (nval + 3 * (size_t)j.ld) + sizeof(int) * ncol;
  j.nval = (int)std::min<size_t>(nval, INT_MAX);
  return *lds <= PL_LDS_BYTES;
}

template <int NT>
static void pl_go(const PlArgs& a, int jobs, size_t lds, int maxit, double thr, double* out, hipStream_t st) {
  static const hipError_t attr = hipFuncSetAttribute((const void*)k_power_lds<NT>,
                                                     hipFuncAttributeMaxDynamicSharedMemorySize, PL_LDS_BYTES);
  FH_HIP(attr);
  hipLaunchKernelGGL(k_power_lds<NT>, dim3(jobs), dim3(NT), lds, st, a, pl_x0(), maxit, thr, out);
  FH_LAUNCH_CHECK();
}

// one or two chains in the LDS form; false (and nothing done) when one does not fit it
static bool power_iteration_lds(const std::vector<std::vector<PwOp>>& hs, const std::vector<int>& ns, int maxit,
                                double thr, double* lam, int* flags, hipStream_t st) {
  const int J = (int)hs.size();
  PlArgs a;
  size_t lds = 0;
  int longest = 1;
  for (int k = 0; k < J; ++k) {
    size_t b = 0;
    if (!pl_job(hs[k], ns[k], a.job[k], &b)) return false;
    lds = std::max(lds, b);
    longest = std::max(longest, a.job[k].ld - 1);
  }
  double* out = mail() + MAIL_POWER;
  if (longest <= 64)
    pl_go<64>(a, J, lds, maxit, thr, out, st);
  else if (longest <= 128)
    pl_go<128>(a, J, lds, maxit, thr, out, st);
  else if (longest <= 256)
    pl_go<256>(a, J, lds, maxit, thr, out, st);
  else if (longest <= 512)
    pl_go<512>(a, J, lds, maxit, thr, out, st);
  else
    pl_go<1024>(a, J, lds, maxit, thr, out, st);
  FH_HIP(hipStreamSynchronize(st));
  const double* res = out;
  for (int k = 0; k < J; ++k) {
    if (res[3 * k + 2] == 1.0) throw Error(FH_ERR_NUMERIC, "Can't normalize a zero-norm vector.");
    lam[k] = res[3 * k];
    flags[k] = (int)res[3 * k + 1];
  }
  return true;
}

double power_iteration_f64(const std::vector<ChainOp>& ops, int n, int maxit, double thr, int* flag,
                           hipStream_t st) {
  FH_CHECK(maxit > 0, "power_iteration: nbr_iter_max <= 0");
  std::vector<PwOp> h = pw_ops(ops);
  double lam;
  int fl;
  if (power_iteration_lds({h}, {n}, maxit, thr, &lam, &fl, st)) {
    if (flag) *flag = fl;
    return lam;
  }
  if (!pw_persistent(h, n)) return power_iteration_wide(h, n, power_x0(n), maxit, thr, flag, st);
  power_iteration_persistent({h}, {n}, maxit, thr, &lam, &fl, st);
  if (flag) *flag = fl;
  return lam;
}

void power_iteration_pair_f64(const std::vector<ChainOp>& ops1, int n1, const std::vector<ChainOp>& ops2, int n2,
                              int maxit, double thr, double* lam1, double* lam2, int* flag, hipStream_t st) {
  FH_CHECK(maxit > 0, "power_iteration: nbr_iter_max <= 0");
  std::vector<PwOp> h1 = pw_ops(ops1), h2 = pw_ops(ops2);
  double lam[2];
  int fl[2];
  if (power_iteration_lds({h1, h2}, {n1, n2}, maxit, thr, lam, fl, st)) {
    *lam1 = lam[0];
    *lam2 = lam[1];
    if (flag) *flag = fl[1];
    return;
  }
  if (!pw_persistent(h1, n1) || !pw_persistent(h2, n2)) {
    *lam1 = power_iteration_f64(ops1, n1, maxit, thr, flag, st);
    *lam2 = power_iteration_f64(ops2, n2, maxit, thr, flag, st);
    return;
  }
  power_iteration_persistent({h1, h2}, {n1, n2}, maxit, thr, lam, fl, st);
  *lam1 = lam[0];
  *lam2 = lam[1];
  if (flag) *flag = fl[1];
}

}  // namespace fh
