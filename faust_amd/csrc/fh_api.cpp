// fh_api.cpp -- C ABI: matrix handles, products, Faust chains, projectors.
#include <algorithm>
#include <map>
#include <mutex>
#include <string>
#include <cstring>
#include <vector>

#include "fh_api_common.hpp"

using namespace fh;

namespace fh {

// Host-side CSR -> CSC (counting sort by column, stable in row order, so rows
// ascend inside each column).
static void host_csc(int m, int n, const int32_t* rp, const int32_t* ci, const void* vals, size_t esz,
                     std::vector<int>& cp, std::vector<int>& ri, std::vector<char>& cv) {
  const int64_t nnz = rp[m];
  cp.assign(n + 1, 0);
  ri.resize(nnz);
  cv.resize(nnz * esz);
  for (int64_t p = 0; p < nnz; ++p) cp[ci[p] + 1]++;
  for (int j = 0; j < n; ++j) cp[j + 1] += cp[j];
  std::vector<int> fill(cp.begin(), cp.end() - 1);
  const char* v = static_cast<const char*>(vals);
  for (int i = 0; i < m; ++i)
    for (int p = rp[i]; p < rp[i + 1]; ++p) {
      int q = fill[ci[p]]++;
      ri[q] = i;
      std::memcpy(&cv[q * esz], v + p * esz, esz);
    }
}

DMatP make_csr_from_host(int dtype, int m, int n, int nnz, const int32_t* rp, const int32_t* ci, const void* vals,
                         hipStream_t st) {
  FH_CHECK(m >= 0 && n >= 0 && nnz >= 0, "csr: negative size");
  FH_CHECK(rp[0] == 0 && rp[m] == nnz, "csr: rowptr inconsistent with nnz");
  // columns must be sorted and in range inside each row (canonical k order)
  for (int i = 0; i < m; ++i) {
    FH_CHECK(rp[i] <= rp[i + 1], "csr: rowptr not non-decreasing");
    for (int p = rp[i]; p < rp[i + 1]; ++p) {
      FH_CHECK(ci[p] >= 0 && ci[p] < n, "csr: column index out of range");
      FH_CHECK(p == rp[i] || ci[p] > ci[p - 1], "csr: column indices must be strictly increasing in each row");
    }
  }
  const size_t esz = dtype_size(dtype);
  auto M = std::make_shared<DMat>();
  M->kind = K_CSR;
  M->dtype = dtype;
  M->m = m;
  M->n = n;
  M->nnz = nnz;
  std::vector<int> cp, ri;
  std::vector<char> cv;
  host_csc(m, n, rp, ci, vals, esz, cp, ri, cv);
  M->rp.alloc(sizeof(int) * (m + 1));
  M->ci.alloc(sizeof(int) * std::max(nnz, 1));
  M->v.alloc(esz * std::max(nnz, 1));
  M->cp.alloc(sizeof(int) * (n + 1));
  M->ri.alloc(sizeof(int) * std::max(nnz, 1));
  M->cv.alloc(esz * std::max(nnz, 1));
  FH_HIP(hipMemcpyAsync(M->rp.p, rp, sizeof(int) * (m + 1), hipMemcpyHostToDevice, st));
  FH_HIP(hipMemcpyAsync(M->cp.p, cp.data(), sizeof(int) * (n + 1), hipMemcpyHostToDevice, st));
  if (nnz > 0) {
    FH_HIP(hipMemcpyAsync(M->ci.p, ci, sizeof(int) * nnz, hipMemcpyHostToDevice, st));
    FH_HIP(hipMemcpyAsync(M->v.p, vals, esz * nnz, hipMemcpyHostToDevice, st));
    FH_HIP(hipMemcpyAsync(M->ri.p, ri.data(), sizeof(int) * nnz, hipMemcpyHostToDevice, st));
    FH_HIP(hipMemcpyAsync(M->cv.p, cv.data(), esz * nnz, hipMemcpyHostToDevice, st));
  }
  M->has_csc = true;
  M->max_row = 0;
  for (int i = 0; i < m; ++i) M->max_row = std::max(M->max_row, rp[i + 1] - rp[i]);
  M->max_col = 0;
  for (int j = 0; j < n; ++j) M->max_col = std::max(M->max_col, cp[j + 1] - cp[j]);
  if (dtype == FH_F64 && std::max(m, n) > 1024) {
    // from rows of some 1000 entries in all, spread as by chance (5 ns an entry:
    // all of them doubled the upload); chains of smaller factors run in one launch
    auto far = [nnz](int nr, const int* ptr, const int* idx) -> int64_t {
      int64_t seen = 0, n = 0;
      const int rows = nr - 1;
      const int look = (int)std::min<int64_t>(rows, std::max<int64_t>(8, (int64_t)nr * 1000 / std::max(nnz, 1)));
      for (int i = 0; i < look; ++i) {
        const int r = 1 + (int)((uint64_t)i * 2654435761u % (unsigned)rows);
        int q = ptr[r - 1];
        for (int e = ptr[r]; e < ptr[r + 1]; ++e) {
          while (q < ptr[r] && idx[q] < idx[e] - 16) ++q;
          n += !(q < ptr[r] && idx[q] <= idx[e] + 16);
        }
        seen += ptr[r + 1] - ptr[r];
      }
      return seen > 0 ? n * nnz / seen : nnz;
    };
    M->far_row = far(m, rp, ci);
    M->far_col = far(n, cp.data(), ri.data());
  }
  if (dtype == FH_F32 || dtype == FH_F64) {
    // ELL views for the gather kernels (rows of S, rows of S^T).  FP32: the
    // widest row rounded up to 4, at most 16 slots, a row's slots together (its
    // lanes load them).  FP64: rounded up to 2, 4 or a multiple of 8, at most
    // 32, pair of slots by pair (a lane per row, so a wave's loads are contiguous)
    const bool by_pair = dtype == FH_F64;
    auto ell = [&](int nr, const int* ptr, const int* idx, const char* val, int widest, int& w, DBuf& dc, DBuf& dv) {
      w = 0;
      if (nr == 0 || widest > (by_pair ? 32 : 16)) return;
      w = by_pair ? (widest <= 2 ? 2 : widest <= 4 ? 4 : (widest + 7) / 8 * 8) : std::max(4, (widest + 3) / 4 * 4);
      std::vector<int> hc((size_t)nr * w, -1);
      std::vector<char> hv((size_t)nr * w * esz, 0);
      for (int r = 0; r < nr; ++r)
        for (int e = ptr[r]; e < ptr[r + 1]; ++e) {
          const size_t q = e - ptr[r], at = by_pair ? (q / 2 * nr + r) * 2 + q % 2 : (size_t)r * w + q;
          hc[at] = idx[e];
          std::memcpy(hv.data() + at * esz, val + (size_t)e * esz, esz);
        }
      dc.alloc(sizeof(int) * hc.size());
      dv.alloc(hv.size());
      FH_HIP(hipMemcpyAsync(dc.p, hc.data(), sizeof(int) * hc.size(), hipMemcpyHostToDevice, st));
      FH_HIP(hipMemcpyAsync(dv.p, hv.data(), hv.size(), hipMemcpyHostToDevice, st));
      FH_HIP(hipStreamSynchronize(st));  // the host vectors go out of scope
    };
    ell(m, rp, ci, (const char*)vals, M->max_row, M->csr_ell_w, M->csr_ell_ci, M->csr_ell_v);
    ell(n, cp.data(), ri.data(), cv.data(), M->max_col, M->csr_tell_w, M->csr_tell_ci, M->csr_tell_v);
  }
  FH_HIP(hipStreamSynchronize(st));
  return M;
}

DMatP make_dense(int dtype, int m, int n, const void* data, int ld, bool on_device, hipStream_t st) {
  FH_CHECK(m >= 0 && n >= 0 && ld >= std::max(m, 1), "dense: bad shape or leading dimension");
  const size_t esz = dtype_size(dtype);
  auto M = std::make_shared<DMat>();
  M->kind = K_DENSE;
  M->dtype = dtype;
  M->m = m;
  M->n = n;
  M->nnz = -1;
  M->d.alloc(esz * std::max<size_t>((size_t)m * n, 1));
  if (m > 0 && n > 0 && data)
    FH_HIP(hipMemcpy2DAsync(M->d.p, esz * m, data, esz * ld, esz * m, n,
                            on_device ? hipMemcpyDeviceToDevice : hipMemcpyHostToDevice, st));
  FH_HIP(hipStreamSynchronize(st));
  return M;
}

// The chain as op'd FP64 CSR factors in application order; false when it is
// not one.  widest: the longest op'd row (1 << 30 when a factor does not know
// its own), mean_max: the largest mean row length.
static bool chain_csr_ops(const std::vector<DMatP>& f, char op, std::vector<ChainCsrOp>& ops, int* widest,
                          double* mean_max) {
  const int J = (int)f.size();
  const char* e_ell = getenv("FH_CSR_ELL");
  const bool ell_on = !(e_ell && e_ell[0] == '0');
  int r = (op == 'N') ? f.back()->n : f.front()->m;
  *widest = 0;
  *mean_max = 0.0;
  for (int i = 0; i < J; ++i) {
    const DMat& S = (op == 'N') ? *f[J - 1 - i] : *f[i];
    if (S.kind != K_CSR || S.dtype != FH_F64 || ((op == 'N') ? S.n : S.m) != r || (op != 'N' && !S.has_csc))
      return false;
    const bool tr = op != 'N';
    const int wr = tr ? S.max_col : S.max_row;
    *widest = std::max(*widest, wr < 0 ? (1 << 30) : wr);
    const int rows = tr ? S.n : S.m;
    *mean_max = std::max(*mean_max, (double)S.nnz / std::max(rows, 1));
    const int ew = tr ? S.csr_tell_w : S.csr_ell_w;
    const int64_t far = tr ? S.far_col : S.far_row;
    ops.push_back({tr ? S.cp.as<int>() : S.rp.as<int>(), tr ? S.ri.as<int>() : S.ci.as<int>(),
                   tr ? S.cv.as<double>() : S.v.as<double>(), rows, (int)S.nnz,
                   ell_on && ew > 0 && ew <= 32 ? ew : 0,
                   tr ? S.csr_tell_ci.as<int>() : S.csr_ell_ci.as<int>(),
                   tr ? S.csr_tell_v.as<double>() : S.csr_ell_v.as<double>(), far < 0 ? S.nnz : far});
    r = rows;
  }
  return true;
}

// Bytes of each of the (at most two) intermediates of an FP64 chain product;
// *nbuf: how many of them the product uses.
size_t faust_ws_need_f64(const std::vector<DMatP>& f, char op, int p, int* nbuf) {
  int maxr = 0;
  for (auto& x : f) maxr = std::max(maxr, op == 'N' ? x->m : x->n);
  *nbuf = std::min(2, (int)f.size() - 1);
  return sizeof(double) * std::max<size_t>((size_t)maxr * p, 1);
}

// Grow a Faust's own intermediates to `need` bytes (hipMalloc only when a
// larger product than any before is requested) and return their addresses.
ChainWs faust_ws_grow(DBuf* ws, size_t need, int nbuf, hipStream_t st, DBuf* ctl) {
  ChainWs w{{nullptr, nullptr}, nullptr, need};
  for (int b = 0; b < nbuf; ++b) {
    if (ws[b].bytes < need) {
      FH_HIP(hipStreamSynchronize(st));  // the old buffer may still be in use
      ws[b].alloc(need);
    }
    w.p[b] = ws[b].p;
  }
  if (ctl) {
    if (ctl->bytes < bsr_chain_ctl_bytes()) {
      ctl->alloc(bsr_chain_ctl_bytes());
      bsr_chain_ctl_clear(ctl->as<int>(), st);
    }
    w.ctl = ctl->as<int>();
  }
  return w;
}

// The same with room for a form that takes more (want bytes in want_nbuf
// buffers, 0: none such) where that is to be had without refusing the call:
// under capture, when memory is short, and once a captured graph holds the
// buffers (its replays write them where they are), the product keeps to `need`.
ChainWs faust_ws_take(DBuf* ws, size_t need, int nbuf, size_t want, int want_nbuf, WsLimits* lim, hipStream_t st,
                      DBuf* ctl) {
  const bool capturing = (need > 0 || want > 0) && stream_capturing(st);
  lim->in_graph = lim->in_graph || capturing;
  if (want > 0) {
    want = std::max(want, need);
    want_nbuf = std::max(want_nbuf, nbuf);
    bool room = true, enough = true;
    for (int b = 0; b < want_nbuf; ++b) room = room && ws[b].bytes >= want;
    for (int b = 0; b < nbuf; ++b) enough = enough && ws[b].bytes >= need;
    if (room) return faust_ws_grow(ws, want, want_nbuf, st, ctl);
    if (want < lim->short_of && !capturing && !(lim->in_graph && enough)) {
      try {
        return faust_ws_grow(ws, want, want_nbuf, st, ctl);
      } catch (const Error&) {
        (void)hipGetLastError();
        lim->short_of = want;
      }
    }
  }
  return faust_ws_grow(ws, need, nbuf, st, ctl);
}

// Y = op(F) X for an FP64 chain; X, Y col-major with ld = rows; ws holds the
// intermediates (faust_ws_need_f64 bytes each).
// ---------------------------------------------------------------- autotune
namespace {
std::mutex g_tune_mu;
std::map<std::string, ChainForm> g_tune;  // chain signature -> quickest form measured
std::map<std::string, int> g_tune_mode;   // BSR / FP32 CSR chain signature -> FH_MUL_* mode
}  // namespace

// FH_AUTOTUNE=0 turns the measurement off (the default forms are used).
bool autotune_on() {
  const char* e = getenv("FH_AUTOTUNE");
  return !(e && e[0] == '0');
}

bool autotune_get_mode(const std::string& key, int* mode) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  auto it = g_tune_mode.find(key);
  if (it == g_tune_mode.end()) return false;
  *mode = it->second;
  return true;
}

void autotune_put_mode(const std::string& key, int mode) {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune_mode[key] = mode;
}

bool stream_capturing(hipStream_t st) {
  hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
  const hipError_t e = hipStreamIsCapturing(st, &cs);
  (void)hipGetLastError();
  return e != hipSuccess || cs != hipStreamCaptureStatusNone;
}

// What the quickest form depends on: direction, columns, each op'd factor's
// shape, entries and whether half of them lie far from the row before (the
// gathers of column-major X are quick where they do not), the ELL slots that
// decide which kernels the forms run (all factors with at most 8, at most 16;
// finer, matrices that differ by a column's count would each be measured), and
// the device.
static std::string chain_sig(char op, int p, int in_rows, const std::vector<ChainCsrOp>& ops) {
  int dev = 0;
  (void)hipGetDevice(&dev);
  std::string k = std::to_string(dev) + op + ":" + std::to_string(p) + ":" + std::to_string(in_rows);
  int slots = 0;
  for (const auto& o : ops) {
    k += "," + std::to_string(o.rows) + "/" + std::to_string(o.nnz) + (o.far * 2 >= o.nnz ? "f" : "n");
    slots = std::max(slots, o.ell > 0 ? o.ell : 99);
  }
  k += slots <= 8 ? "/8" : slots <= 16 ? "/16" : "";
  return k;
}

// AUTO mode on an all-CSR chain uses the form measured quickest for this chain
// signature (measured on its first call outside graph capture: every candidate
// once untimed, then the minimum of three timings of five back-to-back
// products, HIP events on the launch stream; the default form stays unless
// another is at least 3% quicker); otherwise, and when measuring is off or
// impossible, the prefetched one-launch chain where the shape allows it (8
// entries ahead unless the rows are long on average and some exceed 8), else
// row-major intermediates for blocks of columns, else the staged chain where
// the planner takes it, else one launch per factor.  `tune` false
// (allocation-free callers) never measures.
ChainPlan64 chain_plan_f64(const std::vector<DMatP>& f, char op, int p, bool tune, hipStream_t st) {
  FH_CHECK(!f.empty(), "Faust::multiply: empty Faust");
  ChainPlan64 P;
  P.need = faust_ws_need_f64(f, op, p, &P.nbuf);
  double mean_max = 0.0;
  P.csr = chain_csr_ops(f, op, P.ops, &P.widest, &mean_max);
  if (!P.csr) return P;
  P.in_rows = (op == 'N') ? f.back()->n : f.front()->m;
  const char* e_pf = getenv("FH_CHAIN_PF");
  const bool plain = mul_mode() == FH_MUL_AUTO && !getenv("FH_CHAIN_FUSED") && !(e_pf && e_pf[0] == '0');
  const int pwc = csr_chain_pf_plan_f64(P.ops, P.in_rows, p);
  const int swc = pwc > 0 ? 0 : csr_chain_plan_f64(P.ops, P.in_rows, p);
  if (pwc > 0)
    P.def = {2, pwc, (P.widest <= 8 || mean_max <= 4.0) ? 8 : 16};
  else if (swc > 0)
    P.def = {1, swc, 0};
  const bool tunable = plain && autotune_on();
  if (tunable) {
    P.key = chain_sig(op, p, P.in_rows, P.ops);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tune.find(P.key);
    if (it != g_tune.end()) {
      P.form = it->second;
      P.known = true;
    }
  }
  P.measure = tunable && !P.known && tune && !stream_capturing(st);
  // chains that fit the one-launch form keep to that and to one launch per factor
  if (plain && csr_rm_fits(P.ops, P.in_rows, p) && !csr_chain_pf_fits(P.ops, P.in_rows, p)) {
    int64_t far = 0;
    for (const auto& o : P.ops) far = std::max(far, o.far);
    P.rm_rule = far * p >= (f.size() > 1 ? RM_TERMS_DEFAULT : RM_TERMS_SINGLE);
    if (P.known ? P.form.kind == 3 : P.measure || P.rm_rule) {
      int r = P.in_rows;  // the last factor's output is Y
      for (size_t i = 0; i + 1 < P.ops.size(); ++i) r = std::max(r, P.ops[i].rows);
      P.rm_nbuf = std::min(2, (int)f.size());
      P.rm_need = sizeof(double) * csr_rm_size(r, p);
    }
  }
  return P;
}

// Y = op(F) X for an FP64 chain; X, Y col-major with ld = rows; ws holds the
// intermediates (plan.need bytes each; the row-major form runs where it holds
// plan.rm_need).
ChainForm faust_multiply_f64(const std::vector<DMatP>& f, char op, const double* X, int p, double* Y, hipStream_t st,
                             const ChainPlan64& plan, const ChainWs& ws, FaustTimers* tm, int* launches) {
  const int J = (int)f.size();
  double* const t1 = static_cast<double*>(ws.p[0]);
  double* const t2 = static_cast<double*>(ws.p[1]);
  const int in_rows0 = (op == 'N') ? f.back()->n : f.front()->m;

  auto per_factor = [&](FaustTimers* tmr) {
    const double* in = X;
    int in_rows = in_rows0;
    for (int i = 0; i < J; ++i) {
      const DMat& S = (op == 'N') ? *f[J - 1 - i] : *f[i];
      const int out_rows = (op == 'N') ? S.m : S.n;
      FH_CHECK(((op == 'N') ? S.n : S.m) == in_rows, "Faust::multiply: factor dimensions do not chain");
      double* out = (i == J - 1) ? Y : ((i & 1) ? t2 : t1);
      FH_CHECK(S.dtype == FH_F64, "Faust::multiply: FP64 chain expected");
      const size_t slot = (op == 'N') ? (size_t)(J - 1 - i) : (size_t)i;
      if (tmr) tmr->begin(slot, st);
      if (S.kind == K_CSR)
        csr_spmm_f64(S, op, in, in_rows, p, out, out_rows, 1.0, 0.0, st);
      else if (S.kind == K_DENSE)
        gemm_f64(op == 'N' ? 'N' : 'T', 'N', out_rows, p, in_rows, 1.0, S.d.as<double>(), S.m, in, in_rows, 0.0,
                 out, out_rows, st);
      else
        throw Error(FH_ERR_UNSUPPORTED, "Faust::multiply: BSR factors need the FP32/BF16 chain");
      if (tmr) tmr->end(slot, st);
      in = out;
      in_rows = out_rows;
    }
  };
  if (!plan.csr) {
    per_factor(tm);
    if (launches) *launches = J;
    return {0, 0, 0};
  }

  const std::vector<ChainCsrOp>& ops = plan.ops;
  const int out_rows = ops.back().rows;
  auto run = [&](const ChainForm& c, FaustTimers* tmr) {
    if (c.kind == 0) {
      per_factor(tmr);
      return;
    }
    if (c.kind == 3) {
      if (tmr) tmr->begin((size_t)J, st);
      csr_rm_from_col(in_rows0, p, X, t1, st);
      if (tmr) tmr->end((size_t)J, st);
      const double* in = t1;
      int in_rows = in_rows0;
      for (int i = 0; i < J; ++i) {
        const size_t slot = (op == 'N') ? (size_t)(J - 1 - i) : (size_t)i;
        double* out = i == J - 1 ? Y : ((i & 1) ? t1 : t2);
        if (tmr) tmr->begin(slot, st);
        csr_rm_mul(ops[i], in_rows, p, in, out, i == J - 1, st);
        if (tmr) tmr->end(slot, st);
        in = out;
        in_rows = ops[i].rows;
      }
      return;
    }
    if (tmr) tmr->begin(0, st);
    if (c.kind == 1)
      csr_chain_run_f64(ops, in_rows0, c.wc, X, in_rows0, p, Y, out_rows, 1.0, 0.0, st);
    else
      csr_chain_pf_run_f64(ops, in_rows0, c.wc, c.pf, X, in_rows0, p, Y, out_rows, 1.0, 0.0, st);
    if (tmr) tmr->end(0, st);
  };

  const bool rm_fits = plan.rm_need > 0 && ws.cap >= plan.rm_need && t1 && (plan.rm_nbuf < 2 || t2);
  const ChainForm def = plan.rm_rule && rm_fits ? ChainForm{3, 0, 0} : plan.def;
  ChainForm use = plan.known && (plan.form.kind != 3 || rm_fits) ? plan.form : def;
  // a choice made without the row-major form, for want of room, is not kept
  if (plan.measure && (plan.rm_need == 0 || rm_fits)) {
    // the default form first: another replaces the quickest so far only
    // when it is at least 3% quicker, so near-ties keep the default and
    // the choice does not flip between processes on timing noise
    std::vector<ChainForm> cand{def};
    auto add = [&](ChainForm c) {
      if (c.kind != def.kind || c.wc != def.wc || c.pf != def.pf) cand.push_back(c);
    };
    add({0, 0, 0});
    if (rm_fits) add({3, 0, 0});
    const int fwc = csr_chain_fit_wc(ops, in_rows0, p);
    if (fwc > 0) add({1, fwc, 0});
    if (csr_chain_pf_fits(ops, in_rows0, p))
      for (int pf : {8, 16}) {
        if (pf == 16 && plan.widest <= 8) continue;
        for (int wc : {1, 2, 4})
          if (wc == 1 || (p + wc - 1) / wc >= 8) add({2, wc, pf});
      }
    hipEvent_t e0, e1;
    FH_HIP(hipEventCreate(&e0));
    FH_HIP(hipEventCreate(&e1));
    float best_ms = 1e30f;
    // each timing covers five back-to-back products: the steady state a
    // caller's loop or graph sees
    for (const ChainForm& c : cand) {
      run(c, nullptr);
      float m = 1e30f;
      for (int rep = 0; rep < 3; ++rep) {
        FH_HIP(hipEventRecord(e0, st));
        for (int r = 0; r < 5; ++r) run(c, nullptr);
        FH_HIP(hipEventRecord(e1, st));
        FH_HIP(hipEventSynchronize(e1));
        float ms = 0.f;
        FH_HIP(hipEventElapsedTime(&ms, e0, e1));
        m = std::min(m, ms);
      }
      if (m < 0.97f * best_ms) {
        best_ms = m;
        use = c;
      }
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tune[plan.key] = use;
  }
  run(use, tm);
  if (launches) *launches = use.kind == 0 ? J : use.kind == 3 ? J + 1 : 1;
  return use;
}

void autotune_clear() {
  std::lock_guard<std::mutex> lk(g_tune_mu);
  g_tune.clear();
  g_tune_mode.clear();
}

// Transform::get_product (faust_Transform.hpp:599-626)
DMatP faust_get_product_f64(const std::vector<DMatP>& f, hipStream_t st, int64_t view_min) {
  FH_CHECK(!f.empty(), "get_product: empty Faust");
  const size_t n = f.size();
  if (n == 1) return dense_of(*f[0], st);
  auto mat = std::make_shared<DMat>();
  matmul_f64(*f[n - 2], 'N', *f[n - 1], 'N', 1.0, 0.0, *mat, st, view_min);
  for (int i = (int)n - 3; i >= 0; --i) {
    auto nm = std::make_shared<DMat>();
    matmul_f64(*f[i], 'N', *mat, 'N', 1.0, 0.0, *nm, st, view_min);
    mat = nm;
  }
  return mat;
}

// count: dense factors whose entries have not been counted are counted now
// (a wait); without it only the known counts are looked at: a chain with an
// all-zero factor gives norm 0 by its first round's product, or NaN where that
// meets infinities, which zero_or_nan looks into
static bool chain_is_zero(const std::vector<DMatP>& f, bool count, hipStream_t st) {
  for (auto& x : f)
    if ((count || x->nnz >= 0) && nnz_of(*x, st) == 0) return true;
  return false;
}

// a norm computed without the counts: 0 where NaN came of an all-zero factor
static double zero_or_nan(const std::vector<DMatP>& f, double lam, hipStream_t st) {
  if (std::isnan(lam) && chain_is_zero(f, true, st)) return 0.0;
  return std::fabs(std::sqrt(lam));
}

// the power-iteration chain of F^H F (or F F^H, the smaller side); false when
// the norm is known without it (*known: 1 for an empty Faust, 0 for a zero one)
static bool spectral_chain(const std::vector<DMatP>& f, std::vector<ChainOp>& ops, int& n, double* known,
                           bool count, hipStream_t st) {
  if (f.empty()) {
    *known = 1.0;
    return false;
  }
  if (chain_is_zero(f, count, st)) {
    *known = 0.0;
    return false;
  }
  const int nr = f.front()->m, nc = f.back()->n;
  if (nc < nr) {
    for (int i = (int)f.size() - 1; i >= 0; --i) ops.push_back({f[i].get(), 'T'});
    for (auto& x : f) ops.push_back({x.get(), 'N'});
    n = nc;
  } else {
    for (auto& x : f) ops.push_back({x.get(), 'N'});
    for (int i = (int)f.size() - 1; i >= 0; --i) ops.push_back({f[i].get(), 'T'});
    n = nr;
  }
  return true;
}

// Transform::spectralNorm (faust_Transform.hpp:684-709)
double faust_spectral_norm_f64(const std::vector<DMatP>& f, int maxit, double thr, int* flag, hipStream_t st,
                               bool count) {
  std::vector<ChainOp> ops;
  int n = 0;
  double known;
  if (!spectral_chain(f, ops, n, &known, count, st)) return known;
  return zero_or_nan(f, power_iteration_f64(ops, n, maxit, thr, flag, st), st);
}

// the 2-norms of two Fausts (PALM's R and L of one factor update), their
// power iterations sharing a launch; the same values as two calls of
// faust_spectral_norm_f64 (f1 first), flag from the last one computed
void faust_spectral_norm_pair_f64(const std::vector<DMatP>& f1, const std::vector<DMatP>& f2, int maxit, double thr,
                                  int* flag, double* n1, double* n2, hipStream_t st) {
  std::vector<ChainOp> o1, o2;
  int m1 = 0, m2 = 0;
  double k1, k2;
  const bool p1 = spectral_chain(f1, o1, m1, &k1, false, st), p2 = spectral_chain(f2, o2, m2, &k2, false, st);
  if (p1 && p2) {
    double l1, l2;
    power_iteration_pair_f64(o1, m1, o2, m2, maxit, thr, &l1, &l2, flag, st);
    *n1 = zero_or_nan(f1, l1, st);
    *n2 = zero_or_nan(f2, l2, st);
    return;
  }
  *n1 = p1 ? zero_or_nan(f1, power_iteration_f64(o1, m1, maxit, thr, flag, st), st) : k1;
  *n2 = p2 ? zero_or_nan(f2, power_iteration_f64(o2, m2, maxit, thr, flag, st), st) : k2;
}

}  // namespace fh

namespace fh {
static thread_local int tl_mul_mode = FH_MUL_AUTO;
int mul_mode() { return tl_mul_mode; }
MulModeScope::MulModeScope(int m) : prev(tl_mul_mode) { tl_mul_mode = m; }
MulModeScope::~MulModeScope() { tl_mul_mode = prev; }
}  // namespace fh

extern "C" {

int fh_mat_dense_create(int dtype, int nrows, int ncols, const void* data, int ld, int src_on_device, fh_mat_t* out) {
  FH_API_BEGIN
  FH_CHECK(out, "null output handle");
  FH_CHECK(dtype == FH_F64 || dtype == FH_F32 || dtype == FH_BF16, "unknown dtype");
  auto M = make_dense(dtype, nrows, ncols, data, ld, src_on_device != 0, nullptr);
  *out = new fh_mat_s{M};
  FH_API_END
}

int fh_mat_csr_create(int dtype, int nrows, int ncols, int nnz, const int32_t* rowptr, const int32_t* colind,
                      const void* vals, int src_on_device, fh_mat_t* out) {
  FH_API_BEGIN
  FH_CHECK(out && rowptr && (nnz == 0 || (colind && vals)), "null argument");
  FH_CHECK(dtype == FH_F64 || dtype == FH_F32 || dtype == FH_BF16, "unknown dtype");
  const size_t esz = dtype_size(dtype);
  if (src_on_device) {
    std::vector<int32_t> rp(nrows + 1), ci(nnz);
    std::vector<char> v(esz * nnz);
    FH_HIP(hipMemcpy(rp.data(), rowptr, sizeof(int) * (nrows + 1), hipMemcpyDeviceToHost));
    if (nnz) {
      FH_HIP(hipMemcpy(ci.data(), colind, sizeof(int) * nnz, hipMemcpyDeviceToHost));
      FH_HIP(hipMemcpy(v.data(), vals, esz * nnz, hipMemcpyDeviceToHost));
    }
    *out = new fh_mat_s{make_csr_from_host(dtype, nrows, ncols, nnz, rp.data(), ci.data(), v.data(), nullptr)};
  } else {
    *out = new fh_mat_s{make_csr_from_host(dtype, nrows, ncols, nnz, rowptr, colind, vals, nullptr)};
  }
  FH_API_END
}

int fh_mat_info(fh_mat_t M, int* kind, int* dtype, int* nrows, int* ncols, int64_t* nnz) {
  FH_API_BEGIN
  FH_CHECK(M, "null handle");
  const DMat& d = *M->m;
  if (kind) *kind = (int)d.kind;
  if (dtype) *dtype = d.dtype;
  if (nrows) *nrows = d.m;
  if (ncols) *ncols = d.n;
  if (nnz) {
    if (d.kind == K_DENSE)
      *nnz = nnz_of(*M->m, nullptr);
    else if (d.kind == K_BSR)
      *nnz = (int64_t)d.bnnz * d.bm * d.bn;
    else
      *nnz = d.nnz;
  }
  FH_API_END
}

int fh_mat_tocpu(fh_mat_t M, void* data_or_vals, int32_t* rowptr, int32_t* colind) {
  FH_API_BEGIN
  FH_CHECK(M, "null handle");
  const DMat& d = *M->m;
  const size_t esz = dtype_size(d.dtype);
  if (d.kind == K_DENSE) {
    if (d.m * (size_t)d.n)
      FH_HIP(hipMemcpy(data_or_vals, d.d.p, esz * (size_t)d.m * d.n, hipMemcpyDeviceToHost));
  } else if (d.kind == K_CSR) {
    if (rowptr) FH_HIP(hipMemcpy(rowptr, d.rp.p, sizeof(int) * (d.m + 1), hipMemcpyDeviceToHost));
    if (d.nnz) {
      if (colind) FH_HIP(hipMemcpy(colind, d.ci.p, sizeof(int) * d.nnz, hipMemcpyDeviceToHost));
      if (data_or_vals) FH_HIP(hipMemcpy(data_or_vals, d.v.p, esz * d.nnz, hipMemcpyDeviceToHost));
    }
  } else {
    bsr_to_host(d, data_or_vals, rowptr, colind);
  }
  FH_API_END
}

int fh_mat_to_dense(fh_mat_t M, void* dense_dev, void* stream) {
  FH_API_BEGIN
  FH_CHECK(M && dense_dev, "null argument");
  hipStream_t st = (hipStream_t)stream;
  const DMat& d = *M->m;
  if (d.dtype == FH_F64) {
    if (d.kind == K_DENSE)
      FH_HIP(hipMemcpyAsync(dense_dev, d.d.p, sizeof(double) * (size_t)d.m * d.n, hipMemcpyDeviceToDevice, st));
    else if (d.kind == K_CSR)
      csr_to_dense_f64(d, (double*)dense_dev, st);
    else
      throw Error(FH_ERR_UNSUPPORTED, "to_dense: FP64 BSR not supported");
  } else {
    mixed_to_dense(d, dense_dev, st);
  }
  FH_API_END
}

int fh_mat_free(fh_mat_t M) {
  FH_API_BEGIN
  delete M;
  FH_API_END
}

int fh_mat_mul_dense(fh_mat_t M, char op, const void* X, int ldx, int ncols, void* Y, int ldy, const void* alpha,
                     const void* beta, void* stream) {
  FH_API_BEGIN
  FH_CHECK(M, "null argument");
  FH_CHECK(op == 'N' || op == 'T' || op == 'H', "op must be N, T or H");
  FH_CHECK(ncols >= 0, "negative column count");
  if (ncols == 0) return FH_OK;  // nothing to compute (X and Y may be null)
  FH_CHECK(X && Y, "null argument");
  hipStream_t st = (hipStream_t)stream;
  const DMat& S = *M->m;
  if (S.dtype == FH_F64) {
    const double a = alpha ? *(const double*)alpha : 1.0, b = beta ? *(const double*)beta : 0.0;
    const int orows = op == 'N' ? S.m : S.n, irows = op == 'N' ? S.n : S.m;
    FH_CHECK(ldx >= std::max(irows, 1) && ldy >= std::max(orows, 1), "bad leading dimension");
    if (S.kind == K_CSR)
      csr_spmm_f64(S, op, (const double*)X, ldx, ncols, (double*)Y, ldy, a, b, st);
    else if (S.kind == K_DENSE)
      gemm_f64(op == 'N' ? 'N' : 'T', 'N', orows, ncols, irows, a, S.d.as<double>(), S.m, (const double*)X, ldx, b,
               (double*)Y, ldy, st);
    else
      throw Error(FH_ERR_UNSUPPORTED, "FP64 BSR products are not supported");
  } else {
    mixed_mul_dense(S, op, X, ldx, ncols, Y, ldy, alpha, beta, st);
  }
  FH_API_END
}

int fh_gemm(int dtype, char opA, char opB, int m, int n, int k, const void* alpha, const void* A, int lda,
            const void* B, int ldb, const void* beta, void* C, int ldc, void* stream) {
  FH_API_BEGIN
  FH_CHECK(dtype == FH_F64, "fh_gemm: FP64 only");
  FH_CHECK(m >= 0 && n >= 0 && k >= 0, "fh_gemm: negative size");
  gemm_f64(opA, opB, m, n, k, alpha ? *(const double*)alpha : 1.0, (const double*)A, lda, (const double*)B, ldb,
           beta ? *(const double*)beta : 0.0, (double*)C, ldc, (hipStream_t)stream);
  FH_API_END
}

int fh_faust_create(fh_faust_t* out) {
  FH_API_BEGIN
  FH_CHECK(out, "null output handle");
  *out = new fh_faust_s();
  FH_API_END
}

int fh_faust_push_back(fh_faust_t F, fh_mat_t M) {
  FH_API_BEGIN
  FH_CHECK(F && M, "null handle");
  if (!F->f.empty()) FH_CHECK(F->f.back()->n == M->m->m, "push_back: dimensions do not chain");
  F->f.push_back(M->m);
  FH_API_END
}

int fh_faust_size(fh_faust_t F, int* n) {
  FH_API_BEGIN
  FH_CHECK(F && n, "null argument");
  *n = (int)F->f.size();
  FH_API_END
}

int fh_faust_factor(fh_faust_t F, int i, fh_mat_t* out) {
  FH_API_BEGIN
  FH_CHECK(F && out, "null argument");
  FH_CHECK(i >= 0 && i < (int)F->f.size(), "factor index out of range");
  auto* h = new fh_mat_s();
  h->m = F->f[i];
  *out = h;
  FH_API_END
}

int fh_faust_free(fh_faust_t F) {
  FH_API_BEGIN
  delete F;
  FH_API_END
}

int fh_faust_set_mul_mode(fh_faust_t F, int mode) {
  FH_API_BEGIN
  FH_CHECK(F, "null handle");
  const bool ok = mode == FH_MUL_AUTO || mode == FH_MUL_PER_FACTOR || mode == FH_MUL_FUSED ||
                  (mode >= FH_MUL_BSR_KERNEL(0) && mode <= FH_MUL_BSR_KERNEL(5)) || mode == FH_MUL_CSR_ROWS1 ||
                  mode == FH_MUL_CSR_ROWS2;
  FH_CHECK(ok, "fh_faust_set_mul_mode: unknown mode");
  F->mul_mode = mode;
  FH_API_END
}

int fh_faust_set_act_dtype(fh_faust_t F, int dtype) {
  FH_API_BEGIN
  FH_CHECK(F, "null handle");
  FH_CHECK(dtype == FH_BF16 || dtype == FH_F32, "activation dtype must be FH_BF16 or FH_F32");
  if (dtype == FH_F32)
    for (auto& x : F->f)
      if (x->kind != K_BSR || x->dtype != FH_F32)
        throw Error(FH_ERR_UNSUPPORTED, "FP32 activations are offered for chains of FP32 BSR factors");
  for (auto& x : F->f) FH_CHECK(x->kind == K_BSR, "the activation dtype is chosen for BSR chains");
  F->act_dtype = dtype;
  FH_API_END
}

int fh_faust_get_act_dtype(fh_faust_t F, int* dtype) {
  FH_API_BEGIN
  FH_CHECK(F && dtype, "null argument");
  FH_CHECK(!F->f.empty(), "empty Faust");
  if (F->f.front()->dtype == FH_F64)
    *dtype = FH_F64;
  else if (F->f.front()->kind == K_BSR)
    *dtype = F->act_dtype == FH_F32 ? FH_F32 : FH_BF16;
  else
    *dtype = FH_F32;
  FH_API_END
}

int fh_faust_get_mul_mode(fh_faust_t F, int* mode) {
  FH_API_BEGIN
  FH_CHECK(F && mode, "null argument");
  *mode = F->mul_mode;
  FH_API_END
}

// A dense FP32 factor in an FP32 chain runs as its CSR twin (built once from
// a host copy of the factor, kept with it): the FP32 chain kernels take CSR.
static std::vector<DMatP> fp32_chain_factors(const std::vector<DMatP>& f, hipStream_t st) {
  std::vector<DMatP> out = f;
  for (auto& x : out) {
    if (x->kind != K_DENSE || x->dtype != FH_F32) continue;
    if (!x->csr_twin) {
      const int m = x->m, n = x->n;
      std::vector<float> h((size_t)m * n);
      if (!h.empty()) FH_HIP(hipMemcpyAsync(h.data(), x->d.p, sizeof(float) * h.size(), hipMemcpyDeviceToHost, st));
      FH_HIP(hipStreamSynchronize(st));
      std::vector<int32_t> rp(m + 1, 0), ci;
      std::vector<float> v;
      for (int r = 0; r < m; ++r) {
        for (int c = 0; c < n; ++c) {
          const float a = h[(size_t)c * m + r];
          if (a != 0.0f) {
            ci.push_back(c);
            v.push_back(a);
          }
        }
        rp[r + 1] = (int32_t)ci.size();
      }
      x->csr_twin = make_csr_from_host(FH_F32, m, n, (int)ci.size(), rp.data(), ci.data(), v.data(), st);
    }
    x = x->csr_twin;
  }
  return out;
}

int fh_faust_multiply(fh_faust_t F, char op, const void* X, int p, void* Y, void* stream) {
  FH_API_BEGIN
  FH_CHECK(F, "null argument");
  MulModeScope mode_scope(F->mul_mode);
  FH_CHECK(op == 'N' || op == 'T' || op == 'H', "op must be N, T or H");
  FH_CHECK(!F->f.empty(), "Faust::multiply: empty Faust");
  FH_CHECK(p >= 0, "negative column count");
  if (p == 0) {  // nothing to compute (X and Y may be null)
    F->last_launches = 0;
    return FH_OK;
  }
  FH_CHECK(X && Y, "null argument");
  hipStream_t st = (hipStream_t)stream;
  if (F->f.front()->dtype == FH_F64) {
    ChainPlan64 pl = chain_plan_f64(F->f, op, p, true, st);
    if (F->f.size() == 1 && pl.rm_need > 0) {
      // a one-factor product uses no workspace but the row-major form's copy
      // of X: that stays out of captured graphs and belongs to the stream that
      // had it first, and products on other streams run without it
      const bool mine = st != hipStreamPerThread && !stream_capturing(st) && (!F->ws_owned || F->ws_stream == st);
      if (mine) {
        F->ws_owned = true;
        F->ws_stream = st;
      } else {
        pl.rm_need = 0;
        pl.measure = false;
      }
    }
    const size_t had[2] = {F->ws[0].bytes, F->ws[1].bytes};
    const ChainWs ws = faust_ws_take(F->ws, pl.need, pl.nbuf, pl.rm_need, pl.rm_nbuf, &F->ws_lim, st);
    const ChainForm ran =
        faust_multiply_f64(F->f, op, (const double*)X, p, (double*)Y, st, pl, ws, &F->timers, &F->last_launches);
    if (pl.measure && pl.rm_need > 0 && ran.kind != 3)
      // the row-major form was measured and not kept: nor is its room
      for (int b = 0; b < 2; ++b) {
        const size_t keep = std::max(had[b], b < pl.nbuf ? pl.need : 0);
        if (F->ws[b].bytes <= keep) continue;
        FH_HIP(hipStreamSynchronize(st));
        F->ws[b].alloc(keep);
      }
  } else {
    const std::vector<DMatP> f = fp32_chain_factors(F->f, st);
    const bool act_f32 = F->act_dtype == FH_F32;
    int nbuf = 0, tbuf = 0;
    const size_t need = faust_ws_need_mixed(f, op, p, &nbuf, act_f32);
    const size_t padded = act_f32                        ? faust_ws_need_f32_tiled(f, op, p, &tbuf)
                          : f.front()->kind == K_CSR ? faust_ws_need_f32_panels(f, op, p, &tbuf)
                                                         : 0;
    const ChainWs ws = faust_ws_take(F->ws, need, nbuf, padded, tbuf, &F->ws_lim, st,
                                     (f.front()->kind == K_BSR && !act_f32) ? &F->ctl : nullptr);
    F->last_launches = faust_multiply_mixed(f, op, X, p, Y, st, ws, &F->timers, act_f32);
  }
  FH_API_END
}

int fh_faust_last_launches(fh_faust_t F, int* launches) {
  FH_API_BEGIN
  FH_CHECK(F && launches, "null argument");
  *launches = F->last_launches;
  FH_API_END
}

int fh_faust_enable_timers(fh_faust_t F, int on) {
  FH_API_BEGIN
  FH_CHECK(F, "null handle");
  if (!on) F->timers.collect();
  F->timers.on = on != 0;
  F->timers.resize(F->f.size() + 1);
  FH_API_END
}

int fh_faust_timers(fh_faust_t F, double* ms, int64_t* counts) {
  FH_API_BEGIN
  FH_CHECK(F && ms && counts, "null argument");
  F->timers.resize(F->f.size() + 1);
  F->timers.collect();
  for (size_t s = 0; s <= F->f.size(); ++s) {
    ms[s] = F->timers.ms[s];
    counts[s] = F->timers.count[s];
    F->timers.ms[s] = 0.0;
    F->timers.count[s] = 0;
  }
  FH_API_END
}

int fh_faust_get_product(fh_faust_t F, void* out_dev, void* stream) {
  FH_API_BEGIN
  FH_CHECK(F && out_dev, "null argument");
  for (auto& x : F->f)
    if (x->dtype != FH_F64 || x->kind == K_BSR)
      throw Error(FH_ERR_UNSUPPORTED, "get_product: FP64 dense / CSR chains only (multiply other chains by the identity)");
  hipStream_t st = (hipStream_t)stream;
  const auto give = [&](const DMatP& P) {
    FH_HIP(hipMemcpyAsync(out_dev, P->d.p, sizeof(double) * (size_t)P->m * P->n, hipMemcpyDeviceToDevice, st));
  };
  DMatP P = faust_get_product_f64(F->f, st);
  give(P);
  // Operands of 64K .. VIEW_MIN entries are multiplied zeros and all, and a zero
  // against an infinity makes NaN where the product of the other terms need
  // not be one: with NaN in the result they are looked at for zeros too.
  constexpr int64_t VIEW_LOOK = 1 << 16;
  bool look = false;
  if (F->f.size() > 1)
    for (auto& x : F->f)
      for (const int64_t n : {(int64_t)x->n, (int64_t)P->n}) look = look || (x->m * n >= VIEW_LOOK && x->m * n < VIEW_MIN);
  double* nan = mail() + MAIL_SUM;
  *nan = 0.0;
  if (look) any_nan_f64(P->d.as<double>(), (int64_t)P->m * P->n, nan, st);
  FH_HIP(hipStreamSynchronize(st));
  if (*nan != 0.0) {
    P = faust_get_product_f64(F->f, st, VIEW_LOOK);
    give(P);
    FH_HIP(hipStreamSynchronize(st));
  }
  FH_API_END
}

int fh_faust_spectral_norm(fh_faust_t F, int max_iter, double threshold, double* norm, int* flag, void* stream) {
  FH_API_BEGIN
  FH_CHECK(F && norm, "null argument");
  for (auto& x : F->f)
    if (x->dtype != FH_F64 || x->kind == K_BSR)
      throw Error(FH_ERR_UNSUPPORTED, "spectral_norm: FP64 dense / CSR chains only");
  *norm = faust_spectral_norm_f64(F->f, max_iter, threshold, flag, (hipStream_t)stream);
  FH_API_END
}

int fh_prox(int dtype, int name, void* M, int nrows, int ncols, int64_t k, int normalized, int pos, const void* supp,
            void* stream) {
  FH_API_BEGIN
  FH_CHECK(dtype == FH_F64, "fh_prox: FP64 only");
  FH_CHECK(M && nrows >= 0 && ncols >= 0, "bad argument");
  prox_f64(name, (double*)M, nrows, ncols, k, normalized != 0, pos != 0, (const double*)supp, (hipStream_t)stream);
  FH_API_END
}

int fh_prox_real(int dtype, int name, void* M, int nrows, int ncols, double s, int normalized, int pos,
                 void* stream) {
  FH_API_BEGIN
  FH_CHECK(dtype == FH_F64, "fh_prox_real: FP64 only");
  FH_CHECK(M && nrows >= 0 && ncols >= 0, "bad argument");
  prox_real_f64(name, (double*)M, nrows, ncols, s, normalized != 0, pos != 0, (hipStream_t)stream);
  FH_API_END
}

int fh_norm_frob(int dtype, const void* M, int64_t n, double* out, void* stream) {
  FH_API_BEGIN
  FH_CHECK(dtype == FH_F64 && out, "fh_norm_frob: FP64 only");
  hipStream_t st = (hipStream_t)stream;
  double* s = mail() + MAIL_SUM;
  reduce_dot_f64((const double*)M, (const double*)M, n, s, st);
  FH_HIP(hipStreamSynchronize(st));
  *out = std::sqrt(*s);
  FH_API_END
}

int fh_dot(int dtype, const void* x, const void* y, int64_t n, double* out, void* stream) {
  FH_API_BEGIN
  FH_CHECK(dtype == FH_F64 && out, "fh_dot: FP64 only");
  hipStream_t st = (hipStream_t)stream;
  double* s = mail() + MAIL_SUM;
  reduce_dot_f64((const double*)x, (const double*)y, n, s, st);
  FH_HIP(hipStreamSynchronize(st));
  *out = *s;
  FH_API_END
}

}  // extern "C"
