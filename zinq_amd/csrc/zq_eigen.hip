// Symmetric eigen-decomposition of the SCF's small dense matrices (n <= 192), the work of eigh /
// geigh in src/linear_algebra.zig:45-71, :184-199 (LAPACKE_dsyevd / dsygvd) on the GPU.
//
// rocSOLVER's dsyevd spends most of its time at these sizes launching the many small kernels of its
// tridiagonal reduction (about 2.4 ms of 3.9 ms at n = 192).  Here the reduction is one workgroup of 512 threads
// that hold the matrix in registers: Householder reduction of the lower triangle as LAPACK dsytd2 (A = Q T Q^T,
// Q = H_0 ... H_(n-3)), step k:
//     row k -> LDS; alpha = A[k+1][k], beta = -sign(alpha) |A[k+1:][k]|, tau = (beta - alpha) / beta,
//     v = (1, A[k+2:][k] / (alpha - beta));  p = tau A v;  w = p - tau/2 (p.v) v;  A -= v w^T + w v^T.
// A step is bound by its serial chain, which every wave computes for itself, in the same order, so all
// agree bitwise.  Two forms:
// k_tridiag (n <= 32): two barriers a step, each quantity formed directly.
// k_tridiag_wide (33 <= n <= 192): one barrier a step, the rank-2 update and the next product in one pass.  Its
//   rounding differs; n <= 32 keeps the first form since the eigenvectors of a symmetric molecule (one water)
//   take their signs from rounding there.  It is also the faster there: n = 24 29 us.
// The reflectors stay in LDS until the end, when they go to global memory.
// k_tridiag_q: Q^T = H_(n-3) ... H_0 accumulated in registers (same layout) by right multiplications
//   M <- M H_k, whose row sums (quad sums) need no barrier.  It runs on a second stream while the
//   tridiagonal problem is solved, which needs only d and e.
// The tridiagonal problem T = Z diag(w) Z^T is rocSOLVER dstedc's divide and conquer, and the
// eigenvectors Q Z are one MFMA product once both streams are done.

#include <rocblas/rocblas.h>
#include <rocsolver/rocsolver.h>

#include <algorithm>
#include <cstring>
#include <map>
#include <mutex>
#include <vector>

#include "../../include/zinq_scf.h"
#include "zq_internal.h"

namespace {

constexpr int kTridiagMax = 192;  // 16 * the largest RB instantiated

// DPP lane moves within a 16-lane row; a source outside the row reads 0.
template <int CTRL>
__device__ inline double dpp_move(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}

// Sum over the 16 lanes of a DPP row, complete in the row's last lane (tc == 15).
__device__ inline double row_sum_last(double v) {
  v += dpp_move<0xB1>(v);   // quad_perm 1 0 3 2
  v += dpp_move<0x4E>(v);   // quad_perm 2 3 0 1: every lane holds its quad's sum
  v += dpp_move<0x114>(v);  // row_shr 4
  v += dpp_move<0x118>(v);  // row_shr 8: lanes 12..15 hold the row's sum
  return v;
}

// Offset of reflector k in the packed store: entries k+1 .. n-1.
__device__ inline int vofs(int k, int n) { return k * (n - 1) - k * (k - 1) / 2; }

// A (n x n symmetric, ld lda) -> d (n), e (n - 1) and the reflectors R (refl_words(n): tau, scal, the
// packed row tails) of A = Q T Q^T, n <= 16 RB.
// One workgroup of 16 TR threads.  Thread (tr, tc) = (tid / 16, tid % 16) owns rows tr + TR a (a < RA) and
// columns tc + 16 b (b < RB); a DPP row of 16 lanes holds one thread row, so a row sum is four DPP steps.  Row k
// (= column k, A symmetric) reaches LDS from the 16 lanes that own it, together with |A[k+2:][k]|^2, which they
// sum on the way.  p.v is summed per wave into LDS before the step's second barrier and then added up in a
// fixed order, so no step waits on a 64-lane shuffle reduction.  Row vectors in LDS are stored column-permuted,
// [c % 16][c / 16] with a padded stride, so a lane reads its own columns contiguously and the 16
// column groups fall in different banks.  Sized for 32 (8 waves, two columns a lane) rather than the 64 it
// used to serve (16 waves, four): n = 7 13 -> 8 us, n = 24 46 -> 29, n = 32 62 -> 39, the same bits.
template <int RB, int TR>
__global__ __launch_bounds__(16 * TR) void k_tridiag(const double *__restrict__ A, int lda, int n, double *__restrict__ d,
                                                  double *__restrict__ e, double *__restrict__ R) {
  constexpr int NT = 16 * TR, NM = 16 * RB, RA = (NM + TR - 1) / TR, CS = RB + 1;
  __shared__ double cbp[2][16 * CS];  // row k, permuted
  __shared__ double pvp[16 * CS];     // p = tau A v, permuted
  __shared__ double xn[2], pdot[2][TR / 4];
  __shared__ double taus[NM], scals[NM], dl[NM], el[NM];
  __shared__ double vl[(NM - 2) * (NM + 1) / 2];
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15, wv = tid >> 6;
  auto P = [](int j) { return (j & 15) * CS + (j >> 4); };
  double a[RA][RB];
#pragma unroll
  for (int ai = 0; ai < RA; ++ai)
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const int r = tr + TR * ai, c = tc + 16 * bj;
      a[ai][bj] = (r < n && c < n) ? A[size_t(r) * lda + c] : 0.0;
    }
  // p stays 0 on the padding columns (no row >= n writes it), so the update leaves them 0
  for (int t = tid; t < 16 * CS; t += NT) pvp[t] = 0.0;
  // row k of the registers -> dst (permuted) by the 16 lanes that own it, and |A[k][k+2:]|^2 -> *xsq.
  // (the row block is picked with 0/1 weights: branches per block get merged into an indexed access,
  // which moves the register array to scratch memory)
  auto gather_row = [&](int k, double *dst, double *xsq) {
    if (tr == k % TR) {
      const int ak = k / TR;
      double s2 = 0.0;
#pragma unroll
      for (int bj = 0; bj < RB; ++bj) {
        double x = 0.0;
#pragma unroll
        for (int ai = 0; ai < RA; ++ai) x = fma(ai == ak ? 1.0 : 0.0, a[ai][bj], x);
        dst[tc * CS + bj] = x;
        s2 += tc + 16 * bj >= k + 2 ? x * x : 0.0;
      }
      s2 = row_sum_last(s2);
      if (tc == 15 && xsq) *xsq = s2;
    }
  };

  for (int k = 0; k + 2 < n; ++k) {
    const int par = k & 1;
    double *cb = cbp[par];
    gather_row(k, cb, &xn[par]);
    __syncthreads();
    const double alpha = cb[P(k + 1)], xnorm2 = xn[par];
    double beta = alpha, tau = 0.0, scal = 0.0;
    if (xnorm2 != 0.0) {
      beta = -copysign(sqrt(alpha * alpha + xnorm2), alpha);
      tau = (beta - alpha) / beta;
      scal = 1.0 / (alpha - beta);
    }
    if (tid == 0) {
      dl[k] = cb[P(k)];
      el[k] = beta;
      taus[k] = tau;
      scals[k] = scal;
    }
    // raw tail of row k for the back-accumulation: v_k[j] = scal * tail[j] for j > k + 1, v_k[k+1] = 1
    for (int j = k + 1 + tid; j < n; j += NT) vl[vofs(k, n) + j - k - 1] = cb[P(j)];
    auto vval = [&](int i) { return i == k + 1 ? 1.0 : (i > k + 1 && i < n ? cb[P(i)] * scal : 0.0); };
    // v on this lane's columns (0 at and left of k), read from the row in LDS at each use: registers
    // hold A
    auto vcol = [&](int bj) {
      const int j = tc + 16 * bj;
      const double x = cb[tc * CS + bj] * scal;
      return j > k + 1 ? x : (j == k + 1 ? 1.0 : 0.0);
    };
    // p = tau A v on this lane's rows; the row's last lane stores p_i and adds p_i v_i to its partial
    double pt[RA];
#pragma unroll
    for (int ai = 0; ai < RA; ++ai) pt[ai] = 0.0;
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const double v = vcol(bj);
#pragma unroll
      for (int ai = 0; ai < RA; ++ai) pt[ai] += a[ai][bj] * v;
      if (bj % 4 == 3) __builtin_amdgcn_sched_barrier(0);  // bounds the loads in flight (registers hold A)
    }
    double pd = 0.0;
#pragma unroll
    for (int ai = 0; ai < RA; ++ai) {
      const double t = tau * row_sum_last(pt[ai]);
      const int r = tr + TR * ai;
      if (tc == 15 && r > k && r < n) {
        pvp[P(r)] = t;
        pd += t * vval(r);
      }
    }
    // per-wave sum of p.v over the wave's 4 row-last lanes (15, 31, 47, 63)
    pd = pd + __shfl_xor(pd, 16, 64);
    pd = pd + __shfl_xor(pd, 32, 64);
    if ((tid & 63) == 63) pdot[par][wv] = pd;
    __syncthreads();
    double dot = 0.0;
#pragma unroll
    for (int q = 0; q < TR / 4; ++q) dot += pdot[par][q];
    const double K = -0.5 * tau * dot;
    double vr[RA], wr[RA];
#pragma unroll
    for (int ai = 0; ai < RA; ++ai) {
      const int r = tr + TR * ai;
      vr[ai] = vval(r);
      wr[ai] = (r > k && r < n) ? pvp[P(r)] + K * vr[ai] : 0.0;
    }
    // A -= v w^T + w v^T on the trailing block (w = 0 at and left of k)
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const double v = vcol(bj), w = tc + 16 * bj > k ? pvp[tc * CS + bj] + K * v : 0.0;
#pragma unroll
      for (int ai = 0; ai < RA; ++ai) a[ai][bj] -= vr[ai] * w + wr[ai] * v;
      if (bj % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
  // the last 2 x 2 block (or the 1 x 1 matrix)
  __syncthreads();
  gather_row(n >= 2 ? n - 2 : 0, cbp[0], nullptr);
  if (n >= 2) gather_row(n - 1, cbp[1], nullptr);
  __syncthreads();
  if (tid == 0) {
    if (n >= 2) {
      dl[n - 2] = cbp[0][P(n - 2)];
      el[n - 2] = cbp[1][P(n - 2)];
      dl[n - 1] = cbp[1][P(n - 1)];
    } else {
      dl[0] = cbp[0][P(0)];
    }
  }
  __syncthreads();  // reflectors, taus, d and e complete
  for (int t = tid; t < n; t += NT) d[t] = dl[t];
  for (int t = tid; t + 1 < n; t += NT) e[t] = el[t];
  // the reflectors for k_tridiag_q: tau_k and scal_k (k < n - 2), then the packed row tails
  const int nk = n > 2 ? n - 2 : 0, nv = n > 2 ? vofs(n - 2, n) : 0;
  for (int t = tid; t < nk; t += NT) R[t] = taus[t], R[n + t] = scals[t];
  for (int t = tid; t < nv; t += NT) R[2 * n + t] = vl[t];
}

// The same reduction for 32 < n <= 192 with one barrier a step and one pass over the registers.  512 threads,
// thread (tr, tc) = (tid / 16, tid % 16) owns rows tr + 32 a and columns tc + 16 b.  With u the reflector's
// direction scaled by a power of two near 1 / |beta| (u_(k+1) = (alpha - beta) s, u_j = A[k][j] s) and
// g = 2 / u.u, step k is p = A u, w = g p - g^2 / 2 (p.u) u, A -= u w^T + w u^T.  Between two barriers:
//   from p of the last step and the not yet updated row k, both in LDS, every 16-lane row works out p.u, w, the
//   updated row k, its norm and the next u for its own columns and rows by itself;
//   one pass then applies the last step's update and multiplies by the next u, three FMAs an element;
//   the row sums p and the next row, k + 1, go to LDS.
// The quotient g is needed only after the barrier, so it passes in the shadow of the pass; tau and
// 1 / (alpha - beta) of the stored reflectors are computed at the end.  The steps run in stages of 32, one per row
// block AK, which makes the finished rows and columns (blocks below AK, 2 AK) drop out at compile time;
// smaller matrices start at a later stage (index shift 32 AK0), so one kernel serves every n.
// Against the two-barrier form, which went over all of A twice a step: n = 150 709 -> 235 us, n = 64 130 -> 68,
// n = 33 64 -> 37.
constexpr int kWideRB = 12, kWideRA = kWideRB / 2, kWideN = 16 * kWideRB;

// Sum over the 16 lanes of a DPP row, on every lane.
__device__ inline double row_sum_all(double v) {
  v += dpp_move<0xB1>(v);   // quad_perm 1 0 3 2
  v += dpp_move<0x4E>(v);   // quad_perm 2 3 0 1
  v += dpp_move<0x141>(v);  // half-row mirror
  v += dpp_move<0x128>(v);  // rotate by 8
  return v;
}

struct WideShared {
  static constexpr int CS = kWideRB + 1;
  double row[2][16 * CS], p[2][16 * CS];  // columns permuted, [c % 16][c / 16]
  double alpha[kWideN], beta[kWideN], d[kWideN];
  double tail[(kWideN - 2) * (kWideN + 1) / 2];
};

// What a step hands on to the next.
struct WideState {
  double a[kWideRA][kWideRB];        // this thread's elements
  double uc[kWideRB], ur[kWideRA];   // the last u on its columns and rows
  double g, u1, s;                   // the last g, u_(k+1) and scale
};

// The steps whose next row, k + 1, lies in row block AK: kk + 1 in [32 AK, 32 AK + 32), kk = k + shift.
template <int AK>
__device__ inline void wide_stage(WideState &t, WideShared &sh, int n, int shift) {
  constexpr int CS = WideShared::CS, B0 = 2 * AK;
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15, end = n + shift;
  auto P = [](int j) { return (j & 15) * CS + (j >> 4); };
  const int k0 = max(32 * AK - 1, shift), k1 = min(32 * AK + 31, end - 1);
  for (int kk = k0; kk < k1; ++kk) {
    const int k = kk - shift, cur = kk & 1;
    const double *row = sh.row[cur], *pl = sh.p[cur];
    // w of the last step
    // a stage's first u starts at column 32 AK - 1, which its blocks leave out
    double dot = AK && kk == 32 * AK - 1 && tc == 15 ? pl[P(kk)] * t.u1 : 0.0;
#pragma unroll
    for (int b = B0; b < kWideRB; ++b) dot = fma(pl[tc * CS + b], t.uc[b], dot);
    const double K = -0.5 * t.g * t.g * row_sum_all(dot);
    double wc[kWideRB], wr[kWideRA];
#pragma unroll
    for (int b = B0; b < kWideRB; ++b) wc[b] = fma(K, t.uc[b], t.g * pl[tc * CS + b]);
#pragma unroll
    for (int a = AK; a < kWideRA; ++a) wr[a] = fma(K, t.ur[a], t.g * pl[P(tr + 32 * a)]);
    // row k, updated, on this thread's columns; its norm beyond k + 1
    const double wk = fma(K, t.u1, t.g * pl[P(kk)]);
    double x[kWideRB], norm2 = 0.0;
#pragma unroll
    for (int b = B0; b < kWideRB; ++b) {
      x[b] = fma(-wk, t.uc[b], fma(-t.u1, wc[b], row[tc * CS + b]));
      const double y = tc + 16 * b >= kk + 2 ? x[b] : 0.0;
      norm2 = fma(y, y, norm2);
    }
    norm2 = row_sum_all(norm2);
    const double u2 = k > 0 ? sh.tail[vofs(k - 1, n) + 1] * t.s : 0.0;  // the last u at k + 1
    const double alpha = fma(-wk, u2, fma(-t.u1, fma(K, u2, t.g * pl[P(kk + 1)]), row[P(kk + 1)]));
    double beta = alpha;
    if (norm2 != 0.0) beta = -copysign(sqrt(fma(alpha, alpha, norm2)), alpha);
    const double s = __builtin_ldexp(1.0, min(1000, 1 - __builtin_amdgcn_frexp_exp(beta)));
    const double as = alpha * s, bs = beta * s, u1 = as - bs;
    // the row's raw tail for the back-accumulation: v_k[j] = tail[j] / (alpha - beta)
    if (tr == 0 && k < n - 2) {
#pragma unroll
      for (int b = B0; b < kWideRB; ++b) {
        const int j = tc + 16 * b;
        if (j > kk && j < end) sh.tail[vofs(k, n) + j - kk - 1] = j == kk + 1 ? alpha : x[b];
      }
    }
    if (tid == 0) sh.d[k] = fma(-2.0 * t.u1, wk, row[P(kk)]), sh.alpha[k] = alpha, sh.beta[k] = beta;
    double xr[kWideRA], pt[kWideRA];
#pragma unroll
    for (int a = AK; a < kWideRA; ++a) {
      const int r = tr + 32 * a;
      const double y = fma(-wk, t.ur[a], fma(-t.u1, wr[a], row[P(r)])) * s;
      xr[a] = r > kk + 1 ? y : (r == kk + 1 ? u1 : 0.0);
      pt[a] = 0.0;
    }
#pragma unroll
    for (int b = B0; b < kWideRB; ++b) {
      const int j = tc + 16 * b;
      x[b] = j > kk + 1 ? x[b] * s : (j == kk + 1 ? u1 : 0.0);
#pragma unroll
      for (int a = AK; a < kWideRA; ++a) {
        t.a[a][b] = fma(-wr[a], t.uc[b], fma(-t.ur[a], wc[b], t.a[a][b]));
        pt[a] = fma(t.a[a][b], x[b], pt[a]);
      }
      t.uc[b] = x[b];
    }
    if (tr == ((kk + 1) & 31))
#pragma unroll
      for (int b = B0; b < kWideRB; ++b) sh.row[cur ^ 1][tc * CS + b] = t.a[AK][b];
#pragma unroll
    for (int a = AK; a < kWideRA; ++a) {
      const double q = row_sum_last(pt[a]);
      if (tc == 15) sh.p[cur ^ 1][P(tr + 32 * a)] = q;
      t.ur[a] = xr[a];
    }
    t.g = norm2 != 0.0 ? 1.0 / (bs * bs - as * bs) : 0.0;
    t.u1 = u1, t.s = s;
    __syncthreads();
  }
}

__global__ __launch_bounds__(512) void k_tridiag_wide(const double *__restrict__ A, int lda, int n, double *__restrict__ d,
                                                      double *__restrict__ e, double *__restrict__ R) {
  constexpr int CS = WideShared::CS;
  __shared__ WideShared sh;
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15;
  const int start = kWideRA - (n + 31) / 32, shift = 32 * start;
  auto P = [](int j) { return (j & 15) * CS + (j >> 4); };
  WideState t;
#pragma unroll
  for (int a = 0; a < kWideRA; ++a)
#pragma unroll
    for (int b = 0; b < kWideRB; ++b) {
      const int r = tr + 32 * a - shift, c = tc + 16 * b - shift;
      t.a[a][b] = (r >= 0 && c >= 0 && r < n && c < n) ? A[size_t(r) * lda + c] : 0.0;
    }
#pragma unroll
  for (int b = 0; b < kWideRB; ++b) t.uc[b] = 0.0;
#pragma unroll
  for (int a = 0; a < kWideRA; ++a) t.ur[a] = 0.0;
  t.g = t.u1 = 0.0, t.s = 1.0;
  for (int x = tid; x < 2 * 16 * CS; x += 512) (&sh.p[0][0])[x] = (&sh.row[0][0])[x] = 0.0;
  __syncthreads();
  for (int c = tid; c < n; c += 512) sh.row[shift & 1][P(c + shift)] = A[c];  // row 0
  __syncthreads();
  if (start <= 0) wide_stage<0>(t, sh, n, shift);
  if (start <= 1) wide_stage<1>(t, sh, n, shift);
  if (start <= 2) wide_stage<2>(t, sh, n, shift);
  if (start <= 3) wide_stage<3>(t, sh, n, shift);
  wide_stage<4>(t, sh, n, shift);
  wide_stage<5>(t, sh, n, shift);
  // the last step (n - 2, no reflector) left row n - 1; d and e, then the reflectors
  const int nk = n - 2, nv = vofs(n - 2, n), last = n - 1 + shift;
  for (int k = tid; k < n; k += 512) d[k] = k < n - 1 ? sh.d[k] : sh.row[last & 1][P(last)];
  for (int k = tid; k < n - 1; k += 512) e[k] = sh.beta[k];
  for (int k = tid; k < nk; k += 512) {
    const double al = sh.alpha[k], be = sh.beta[k];
    R[k] = be != al ? (be - al) / be : 0.0;
    R[n + k] = be != al ? 1.0 / (al - be) : 0.0;
  }
  for (int x = tid; x < nv; x += 512) R[2 * n + x] = sh.tail[x];
}

// Q from the reflectors k_tridiag left in R (one workgroup, the same thread
// layout): M = Q^T = H_(n-3) ... H_0, from M = I by M <- M H_k = M - tau (M v) v^T for k = n-3 .. 0,
// whose row sums (quad sums) need no barrier; then Q[c][r] = M[r][c].  It runs beside the tridiagonal
// eigensolver, which needs only d and e.
template <int RB, int TR>
__global__ __launch_bounds__(16 * TR) void k_tridiag_q(const double *__restrict__ R, int n, double *__restrict__ Q) {
  constexpr int NT = 16 * TR, NM = 16 * RB, RA = (NM + TR - 1) / TR;
  __shared__ double taus[NM], scals[NM];
  __shared__ double vl[(NM - 2) * (NM + 1) / 2];
  const int tid = threadIdx.x, tr = tid >> 4, tc = tid & 15;
  const int nk = n > 2 ? n - 2 : 0, nv = n > 2 ? vofs(n - 2, n) : 0;
  for (int t = tid; t < nk; t += NT) taus[t] = R[t], scals[t] = R[n + t];
  for (int t = tid; t < nv; t += NT) vl[t] = R[2 * n + t];
  __syncthreads();
  double a[RA][RB];
#pragma unroll
  for (int ai = 0; ai < RA; ++ai)
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const int r = tr + TR * ai, c = tc + 16 * bj;
      a[ai][bj] = (r == c && r < n) ? 1.0 : 0.0;
    }
  for (int k = n - 3; k >= 0; --k) {
    const double tau = taus[k], scal = scals[k];
    const double *tail = vl + vofs(k, n) - k - 1;  // tail[j], j > k
    auto vcol = [&](int bj) {
      const int j = tc + 16 * bj, jc = min(max(j, k + 1), n - 1);  // reads stay inside reflector k
      const double x = tail[jc] * scal;
      return (j > k + 1 && j < n) ? x : (j == k + 1 ? 1.0 : 0.0);
    };
    // rows <= k of M are still those of I and v vanishes there, so their u is 0
    double u[RA];
#pragma unroll
    for (int ai = 0; ai < RA; ++ai) u[ai] = 0.0;
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const double v = vcol(bj);
#pragma unroll
      for (int ai = 0; ai < RA; ++ai) u[ai] += a[ai][bj] * v;
      if (bj % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
#pragma unroll
    for (int ai = 0; ai < RA; ++ai) u[ai] = tau * __shfl(row_sum_last(u[ai]), (tid & ~15) | 15, 64);
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const double v = vcol(bj);
#pragma unroll
      for (int ai = 0; ai < RA; ++ai) a[ai][bj] -= u[ai] * v;
      if (bj % 4 == 3) __builtin_amdgcn_sched_barrier(0);
    }
  }
  // Q[c][r] = M[r][c]
#pragma unroll
  for (int ai = 0; ai < RA; ++ai)
#pragma unroll
    for (int bj = 0; bj < RB; ++bj) {
      const int r = tr + TR * ai, c = tc + 16 * bj;
      if (r < n && c < n) Q[size_t(c) * n + r] = a[ai][bj];
    }
}

// Words of the reflector store of one n x n matrix: tau and scal per step, the packed row tails.
inline size_t refl_words(int n) { return 2 * size_t(n) + (n > 2 ? size_t(n - 2) * (n + 1) / 2 : 0); }

// The reduction on s; Q on s2, which waits for it, while s goes on (the caller joins s2 back).
hipError_t launch_tridiag(hipStream_t s, hipStream_t s2, hipEvent_t fork, const double *A, int lda, int n, double *d,
                          double *e, double *R, double *Q) {
  if (n <= 32)
    hipLaunchKernelGGL((k_tridiag<2, 32>), dim3(1), dim3(512), 0, s, A, lda, n, d, e, R);
  else
    hipLaunchKernelGGL(k_tridiag_wide, dim3(1), dim3(512), 0, s, A, lda, n, d, e, R);
  if (hipError_t err = hipEventRecord(fork, s)) return err;
  if (hipError_t err = hipStreamWaitEvent(s2, fork, 0)) return err;
  if (n <= 64)
    hipLaunchKernelGGL((k_tridiag_q<4, 64>), dim3(1), dim3(1024), 0, s2, R, n, Q);
  else if (n <= 128)
    hipLaunchKernelGGL((k_tridiag_q<8, 64>), dim3(1), dim3(1024), 0, s2, R, n, Q);
  else
    hipLaunchKernelGGL((k_tridiag_q<12, 32>), dim3(1), dim3(512), 0, s2, R, n, Q);
  return hipGetLastError();
}

}  // namespace

// The context's rocBLAS handle, on its stream, with atomics off so that every product is reproducible.
void *zq_blas(zq_ctx *ctx) {
  if (!ctx->solver) {
    rocblas_handle h = nullptr;
    if (rocblas_create_handle(&h) != rocblas_status_success) return nullptr;
    rocblas_set_stream(h, ctx->stream);
    rocblas_set_atomics_mode(h, rocblas_atomics_not_allowed);
    ctx->solver = h;
  }
  return ctx->solver;
}

namespace {

rocblas_handle eig_handle(zq_ctx *ctx) { return (rocblas_handle)zq_blas(ctx); }

// The stream the Q accumulations of every context on a device share, created on first use and kept
// until the process ends: a stream per context would add a hardware queue per context, and streams
// beyond the hardware queues share them, ordering unrelated work.  Two contexts' accumulations may
// queue behind each other here; each still waits only for its own reduction.
hipError_t device_eig_stream(int device, hipStream_t *out) {
  static std::mutex mu;
  static std::map<int, hipStream_t> streams;
  std::lock_guard<std::mutex> lock(mu);
  hipStream_t &st = streams[device];
  if (!st)
    if (hipError_t err = hipStreamCreateWithFlags(&st, hipStreamNonBlocking)) {
      st = nullptr;
      return err;
    }
  *out = st;
  return hipSuccess;
}

}  // namespace

int zq_syev_rows(zq_ctx *ctx, double *A, int n, double *w, double *offd, int *info) {
  if (n < 1) return zq_fail(ctx, ZQ_ERR_INVALID, "zq_syev_rows: n < 1");
  rocblas_handle h = eig_handle(ctx);
  if (!h) return zq_fail(ctx, ZQ_ERR_LAPACK, "rocblas handle");
  zq_prof_begin(ctx, "scf_eig");
  if (n > kTridiagMax) {
    const rocblas_status st = rocsolver_dsyevd(h, rocblas_evect_original, rocblas_fill_upper, n, A, n, w, offd, info);
    zq_prof_end(ctx);
    if (st != rocblas_status_success) return zq_fail(ctx, ZQ_ERR_LAPACK, "rocsolver_dsyevd");
    return ZQ_OK;
  }
  const size_t nn = size_t(n) * n;
  auto *Qm = (double *)zq_scratch(ctx, "eig_Q", nn * sizeof(double));
  auto *Z = (double *)zq_scratch(ctx, "eig_Z", nn * sizeof(double));
  // no captured SCF iteration holds the reflector store, so growing it keeps the capture cache
  auto *R = (double *)zq_scratch(ctx, "eig_refl", refl_words(n) * sizeof(double), nullptr, false);
  if (!Qm || !Z || !R) {
    zq_prof_end(ctx);
    return zq_fail(ctx, ZQ_ERR_OOM, "eigen-solver buffers");
  }
  hipStream_t s2 = nullptr;
  ZQ_TRY(ctx, device_eig_stream(ctx->device, &s2));
  for (hipEvent_t &ev : ctx->eig_events)
    if (!ev) ZQ_TRY(ctx, hipEventCreateWithFlags(&ev, hipEventDisableTiming));
  hipStream_t s = ctx->stream;
  hipEvent_t fork = ctx->eig_events[0], join = ctx->eig_events[1];
  const hipError_t le = launch_tridiag(s, s2, fork, A, n, n, w, offd, R, Qm);
  if (le != hipSuccess) {
    zq_prof_end(ctx);
    return zq_check(ctx, le, "k_tridiag");
  }
  // T = Z diag(w) Z^T: column k of the column-major Z (= row k of Z as stored) is eigenvector k; Q is
  // accumulated on s2 meanwhile
  const rocblas_status st = rocsolver_dstedc(h, rocblas_evect_tridiagonal, n, w, offd, Z, n, info);
  // s waits for Q even when the solver failed, so no later work on s overtakes it
  const hipError_t je = hipEventRecord(join, s2);
  const hipError_t we = je == hipSuccess ? hipStreamWaitEvent(s, join, 0) : je;
  zq_prof_end(ctx);  // before the product, which times itself (profile regions do not nest)
  if (we != hipSuccess) return zq_check(ctx, we, "eigen-solver join");
  if (st != rocblas_status_success) return zq_fail(ctx, ZQ_ERR_LAPACK, "rocsolver_dstedc");
  // row k of A = (Q z_k)^T: A[k][p] = sum_q Z[k][q] Q[p][q]
  return zq_gemm_nt(ctx, Z, n, Qm, n, A, n, n, n, n, 1.0, "scf_eig");
}

namespace {
// out[i n + k] = V[k n + i] (16 x 16 tiles through LDS), then w (n) and info, into pinned memory.
__global__ __launch_bounds__(256) void k_eigh_out(const double *__restrict__ V, const double *__restrict__ w,
                                                  const int *__restrict__ info, int n, double *__restrict__ out) {
  __shared__ double t[16][17];
  const int x = threadIdx.x & 15, y = threadIdx.x >> 4, i0 = blockIdx.y * 16, k0 = blockIdx.x * 16;
  if (k0 + y < n && i0 + x < n) t[y][x] = V[size_t(k0 + y) * n + i0 + x];
  __syncthreads();
  if (i0 + y < n && k0 + x < n) out[size_t(i0 + y) * n + k0 + x] = t[x][y];
  if (blockIdx.y == 0 && threadIdx.x < 16 && k0 + x < n) out[size_t(n) * n + k0 + x] = w[k0 + x];
  if (blockIdx.x == 0 && blockIdx.y == 0 && threadIdx.x == 0) out[size_t(n) * n + n] = *info;
}
}  // namespace

extern "C" int zq_eigh(zq_ctx *ctx, size_t n, const double *A, double *W, double *U) {
  ZqGate _gate;
  if (!ctx || !A || !W || !U || n < 1) return zq_fail(ctx, ZQ_ERR_INVALID, "zq_eigh: null argument or n = 0");
  if (n > 8192) return zq_fail(ctx, ZQ_ERR_INVALID, "zq_eigh: n too large");
  ZQ_TRY(ctx, hipSetDevice(ctx->device));
  const size_t nn = n * n;
  auto *dA = (double *)zq_scratch(ctx, "eigh_A", nn * sizeof(double));
  auto *dw = (double *)zq_scratch(ctx, "eigh_w", 2 * n * sizeof(double));
  auto *dinfo = (int *)zq_scratch(ctx, "eigh_info", sizeof(int));
  if (!dA || !dw || !dinfo) return zq_fail(ctx, ZQ_ERR_OOM, "zq_eigh buffers");
  if (nn <= kZqStageMax) {
    // A through pinned memory; U (the transpose of the eigenvector rows), W and info back in it
    ZqStage st;
    if (int rc = st.take(ctx, nn + n + 1)) return rc;
    std::memcpy(st.host, A, nn * sizeof(double));
    zq_pad(ctx, st.dev, 1, int(n), int(n), dA);
    if (int rc = zq_syev_rows(ctx, dA, int(n), dw, dw + n, dinfo)) return rc;
    hipLaunchKernelGGL(k_eigh_out, dim3(unsigned((n + 15) / 16), unsigned((n + 15) / 16)), dim3(256), 0, ctx->stream, dA,
                       dw, dinfo, int(n), st.dev);
    ZQ_LAUNCH_CHECK(ctx, "k_eigh_out");
    ZQ_TRY(ctx, hipStreamSynchronize(ctx->stream));
    st.done();
    if (st.host[nn + n] != 0.0) return zq_fail(ctx, ZQ_ERR_LAPACK, "zq_eigh: tridiagonal eigensolver did not converge");
    std::memcpy(U, st.host, nn * sizeof(double));
    std::memcpy(W, st.host + nn, n * sizeof(double));
    return ZQ_OK;
  }
  ZQ_TRY(ctx, hipMemcpyAsync(dA, A, nn * sizeof(double), hipMemcpyHostToDevice, ctx->stream));
  if (int rc = zq_syev_rows(ctx, dA, int(n), dw, dw + n, dinfo)) return rc;
  std::vector<double> V(nn);
  int info = 0;
  ZQ_TRY(ctx, hipMemcpyAsync(V.data(), dA, nn * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  ZQ_TRY(ctx, hipMemcpyAsync(W, dw, n * sizeof(double), hipMemcpyDeviceToHost, ctx->stream));
  ZQ_TRY(ctx, hipMemcpyAsync(&info, dinfo, sizeof(int), hipMemcpyDeviceToHost, ctx->stream));
  ZQ_TRY(ctx, hipStreamSynchronize(ctx->stream));
  if (info != 0) return zq_fail(ctx, ZQ_ERR_LAPACK, "zq_eigh: tridiagonal eigensolver did not converge");
  for (size_t i = 0; i < n; ++i)  // eigenvector k is row k of V and column k of U
    for (size_t k = 0; k < n; ++k) U[i * n + k] = V[k * n + i];
  return ZQ_OK;
}
