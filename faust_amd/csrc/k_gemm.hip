// k_gemm.hip -- dense FP64 GEMM in the canonical order on the matrix cores.
//
// v_mfma_f64_16x16x4_f64 accumulates its four k terms as four fused
// multiply-adds in ascending k, each rounded, starting from C (checked bit
// for bit against fma chains, denormals, cancellation and overflow included),
// so a tile's accumulator register is the canonical chain of its entry and the
// oracle's bits are kept.  A dependent chain of these instructions issues at
// the full rate (64 cycles each), so one accumulator per wave is enough.
//
// Tiling: four waves (2 x 2) compute a 32 TX x 32 TY tile of C, each wave
// TX x TY accumulators of 16 x 16.  K advances in steps of 32 through
// double-buffered LDS tiles; the next step's global values are loaded into
// registers while the current step computes, the fragments of the next four k
// are read from LDS while the current four multiply, and one barrier ends a
// step.  op(B)'s fragment is passed as the instruction's A operand and
// op(A)'s as its B operand, so lane l holds row l % 16 of C and the 16 lanes
// of a row group store 128 contiguous bytes.
//
// Tile choice: a wave's time is its chains' length times its accumulators, so
// small outputs want many small tiles side by side and large ones the LDS
// reuse of big tiles.  us for (TX, TY) = (1,1) / (1,2) / (2,2), square NN:
// 256: 7.9 / 11.2 / 18.0; 512: 14.0 / 20.9 / 33.1; 768: 35.6 / 42.7 / 48.7;
// 1024: 63.1 / 56.0 / 63.9; 2048: 433 / 416 / 360.  The bound is FP64 MFMA
// issue (78.6 TFLOP/s): 1024^3 runs at 38 TFLOP/s, the rest is the step's LDS
// stores and barrier.  64 x 64 tiles of v_fma_f64 took 32, 61, 91, 119 and
// 600 us.
#include "fh_internal.hpp"

namespace fh {

constexpr int GK = 32;  // k step

typedef double gm_d4 __attribute__((ext_vector_type(4)));

// An E x GK tile of an operand.  KC (element (r, kk) at P[r * ld + kk], k
// contiguous): kept as S[r][kk], rows of GK + 2; else (P[kk * ld + r]) as
// S[kk][r], rows of E + 16.  Either way the loads are coalesced and neither
// the stores nor the fragment reads (16 rows x 2 k per half-wave) conflict.
template <int E, bool KC>
struct GmTile {
  static constexpr int NR = E * GK / 256;  // values per thread
  static constexpr int LD = KC ? GK + 2 : E + 16, SIZE = KC ? E * LD : GK * LD;
  // Indices are clamped to the operand, so every load is unconditional (a
  // conditional one would wait for the ones before it); rows past the end
  // only feed outputs that are not stored.
  static __device__ __forceinline__ void load(const double* __restrict__ P, int ld, int rows, int kdim, int r0,
                                              int k0, int t, double (&reg)[NR]) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int e = t + 256 * q;
      const int gr = min(r0 + (KC ? e / GK : e % E), rows - 1), gk = k0 + (KC ? e % GK : e / E);
      const int ck = min(gk, kdim - 1);
      reg[q] = KC ? P[(size_t)gr * ld + ck] : P[(size_t)ck * ld + gr];
    }
  }
  // krem: k values left from the step's first; those past it are stored as 0
  // (here and not at the load, where it would wait for the load)
  static __device__ __forceinline__ void store(double* S, int t, int krem, const double (&reg)[NR]) {
#pragma unroll
    for (int q = 0; q < NR; ++q) {
      const int e = t + 256 * q;
      S[KC ? (e / GK) * LD + e % GK : (e / E) * LD + e % E] = (KC ? e % GK : e / E) < krem ? reg[q] : 0.0;
    }
  }
  static __device__ __forceinline__ double get(const double* S, int r, int kk) {
    return S[KC ? r * LD + kk : kk * LD + r];
  }
};

// op(A) is m x k: element (i, kk) = transA ? A[i*lda + kk] : A[kk*lda + i]
// op(B) is k x n: element (kk, j) = transB ? B[kk*ldb + j] : B[j*ldb + kk]
// B is held as the row operand of its transpose: row j, column kk.
template <int TX, int TY, bool TA, bool TB>
__global__ __launch_bounds__(256) void k_gemm_f64(int m, int n, int k, double alpha, const double* __restrict__ A,
                                                   int lda, const double* __restrict__ B, int ldb, double beta,
                                                   double* __restrict__ C, int ldc) {
  using OA = GmTile<32 * TX, TA>;
  using OB = GmTile<32 * TY, !TB>;
  __shared__ double As[2][OA::SIZE];
  __shared__ double Bs[2][OB::SIZE];
  const int t = threadIdx.x, lane = t & 63, li = lane & 15, lk = lane >> 4;
  const int wi = ((t >> 6) & 1) * 16 * TX, wj = (t >> 7) * 16 * TY;  // this wave's corner of the tile
  const int i0 = blockIdx.x * 32 * TX, j0 = blockIdx.y * 32 * TY;
  gm_d4 acc[TX][TY];
#pragma unroll
  for (int a = 0; a < TX; ++a)
#pragma unroll
    for (int b = 0; b < TY; ++b) acc[a][b] = gm_d4{0.0, 0.0, 0.0, 0.0};
  if (k > 0) {
    double ra[OA::NR], rb[OB::NR];
    OA::load(A, lda, m, k, i0, 0, t, ra);
    OB::load(B, ldb, n, k, j0, 0, t, rb);
    OA::store(As[0], t, k, ra);
    OB::store(Bs[0], t, k, rb);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < k; k0 += GK) {
      const bool more = k0 + GK < k;
      if (more) {
        OA::load(A, lda, m, k, i0, k0 + GK, t, ra);
        OB::load(B, ldb, n, k, j0, k0 + GK, t, rb);
      }
      // the fragments of the next four k are read while the current ones multiply
      double a[2][TX], b[2][TY];
      auto frag = [&](int kk, double (&fa)[TX], double (&fb)[TY]) {
#pragma unroll
        for (int q = 0; q < TX; ++q) fa[q] = OA::get(As[buf], wi + 16 * q + li, kk + lk);
#pragma unroll
        for (int q = 0; q < TY; ++q) fb[q] = OB::get(Bs[buf], wj + 16 * q + li, kk + lk);
      };
      frag(0, a[0], b[0]);
#pragma unroll
      for (int kk = 0; kk < GK; kk += 4) {
        const int c = (kk >> 2) & 1;
        if (kk + 4 < GK) frag(kk + 4, a[c ^ 1], b[c ^ 1]);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < TX; ++x)
#pragma unroll
          for (int y = 0; y < TY; ++y)
            acc[x][y] = __builtin_amdgcn_mfma_f64_16x16x4f64(b[c][y], a[c][x], acc[x][y], 0, 0, 0);
        __builtin_amdgcn_sched_barrier(0);
      }
      if (more) {  // the other buffer was last read before the previous barrier
        OA::store(As[buf ^ 1], t, k - k0 - GK, ra);
        OB::store(Bs[buf ^ 1], t, k - k0 - GK, rb);
        __syncthreads();
        buf ^= 1;
      }
    }
  }
  // register r of lane l: row l % 16, column l / 16 + 4 r of the 16 x 16 tile
#pragma unroll
  for (int x = 0; x < TX; ++x) {
    const int gi = i0 + wi + 16 * x + li;
    if (gi >= m) continue;
#pragma unroll
    for (int y = 0; y < TY; ++y)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int gj = j0 + wj + 16 * y + lk + 4 * r;
        if (gj >= n) continue;
        const double tt = alpha * acc[x][y][r];
        double* cp = C + (size_t)gj * ldc + gi;
        *cp = (beta == 0.0) ? tt : fma(beta, *cp, tt);
      }
  }
}

template <int TX, int TY>
static void gemm_go(bool ta, bool tb, int m, int n, int k, double alpha, const double* A, int lda, const double* B,
                    int ldb, double beta, double* C, int ldc, hipStream_t st) {
  const dim3 grid((m + 32 * TX - 1) / (32 * TX), (n + 32 * TY - 1) / (32 * TY));
  auto kern = ta ? (tb ? k_gemm_f64<TX, TY, true, true> : k_gemm_f64<TX, TY, true, false>)
                 : (tb ? k_gemm_f64<TX, TY, false, true> : k_gemm_f64<TX, TY, false, false>);
  hipLaunchKernelGGL(kern, grid, dim3(256), 0, st, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc);
}

void gemm_f64(char opA, char opB, int m, int n, int k, double alpha, const double* A, int lda, const double* B,
              int ldb, double beta, double* C, int ldc, hipStream_t st) {
  if (m <= 0 || n <= 0) return;
  const bool ta = opA != 'N', tb = opB != 'N';
  const int64_t tiles = (int64_t)((m + 31) / 32) * ((n + 31) / 32);
  if (tiles <= 640)
    gemm_go<1, 1>(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, st);
  else if (tiles <= 3072)
    gemm_go<1, 2>(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, st);
  else
    gemm_go<2, 2>(ta, tb, m, n, k, alpha, A, lda, B, ldb, beta, C, ldc, st);
  FH_LAUNCH_CHECK();
}

}  // namespace fh
