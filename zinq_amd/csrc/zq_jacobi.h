// Eigenpairs of small symmetric matrices (n <= 96), one workgroup each: cyclic Jacobi, the matrix in LDS and
// the vectors in registers.
//
// The m = 2 h indices (n rounded up to an even number, padding rows zero) sit on a line of positions.  Even
// steps rotate the pairs of positions (2i, 2i + 1), odd steps (2i + 1, 2i + 2), and every rotation also swaps its
// pair, so in the m steps of a sweep every two indices meet once (odd-even transposition) and the line ends
// reversed, while every lane keeps its addresses.  In odd steps the two ends form a pair that is to stay where it
// is: (cos, sin) = (0, 1), which with the swap leaves both in place and turns the sign of position 0.  One step:
//   rotation   each lane takes one pair and every wave computes all of them for itself, so no barrier parts the
//              rotations from their use.  The angle is the textbook one (tan of it the smaller root), in single
//              precision: that only decides how much of the pivot is left (1e-7 of it, which the next sweep
//              takes).  The rotation is orthogonal to double precision: tau = tan(angle / 2) is taken as exact,
//              sin = 2 tau / (1 + tau^2), cos = 1 - tau sin;
//   vectors    rows of V by wave, positions 2i and 2i + 1 in lane i; odd steps shift the even positions by one
//              lane and back (DPP), so V needs no LDS;
//   matrix     the lower triangle in LDS, in four planes by the parities of row and column (lanes then fall in
//              different banks).  The lane of pair i takes the 2 x 2 blocks of pairs (i, i + d mod h), d <= h / 2,
//              its waves the distances d in turn: each block meets both rotations once, in place.
// The diagonal and the pivots of the next step are kept apart, one copy for even and one for odd steps, so a
// step ends in one barrier.  Sweeps end when no element off the diagonal is above 2^-51 of the largest of
// the start, after 4 to 8 of them; a matrix with infinities or NaN runs kSweeps and reports it.
//
// What bounds it: the serial chain of a step (LDS read, rotation, LDS exchange, blocks, barrier) and, at n = 72,
// the waves' issue of it; 72 steps a sweep.  8 waves, since each repeats the rotations: a form of 16 waves with V
// and a movable matrix in LDS took 1.5 ms where this takes 0.7.  For 96 molecules of n = 7 .. 72 this
// replaced dsyevd_strided_batched once per distinct n on three streams: 3.5 to 10.7 ms (by ROCm release, its
// tridiagonal reductions are many small launches) -> 0.7 ms, F' and C included.
#pragma once

#include <hip/hip_runtime.h>

namespace zqj {

constexpr int kThreads = 512, kWaves = kThreads / 64, kMaxN = 96, kSweeps = 30;

// Lanes that hold a step's pairs, and pairs at most.
__host__ __device__ constexpr int lanes_of(int n) { return n <= 32 ? 16 : n <= 64 ? 32 : 64; }
__host__ __device__ constexpr int pairs_of(int W) { return W == 64 ? kMaxN / 2 : W; }

// LDS doubles of an n x n problem: the four planes, rotations per wave, two copies of the diagonal and of the
// pivots, a slot per wave.
__host__ __device__ constexpr int lds_doubles(int n) {
  const int h = pairs_of(lanes_of(n));
  return 4 * h * h + kWaves * 2 * h + 6 * h + kWaves;
}

// Lane i of the wave takes lane i + 1's value (the last the first's), and back.
template <int CTRL>
__device__ inline double wave_turn(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xF, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xF, 0xF, false);
  return __hiloint2double(hi, lo);
}
__device__ inline double from_next(double v) { return wave_turn<0x134>(v); }  // wave_rol:1
__device__ inline double from_prev(double v) { return wave_turn<0x13C>(v); }  // wave_ror:1

__device__ inline double wg_max(double v, double *red) {
  for (int w = 32; w; w >>= 1) {
    const double o = __shfl_xor(v, w, 64);
    v = o > v || o != o ? o : v;  // NaN stays
  }
  if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  double r = red[0];
  for (int w = 1; w < kWaves; ++w) r = red[w] > r || red[w] != red[w] ? red[w] : r;
  __syncthreads();
  return r;
}

// One problem: W = lanes_of(n).  Row r of V is held by group r mod kGroups of W lanes, as v[r / kGroups].
template <int W>
struct Jacobi {
  static constexpr int G = 64 / W, kGroups = kWaves * G, HM = pairs_of(W);
  static constexpr int kRows = (2 * HM + kGroups - 1) / kGroups, kBlocks = (HM / 2 + kGroups - 1) / kGroups;
  double *A, *diag, *piv, *red;
  double2 *rot;
  int h, i, g, wave;
  double v[kRows][2];    // positions 2i and 2i + 1
  int adr[2][kBlocks][4];  // [step parity]: elements (first, first), (first, second), (second, first), (second, second)
  int mate[kBlocks];     // the other pair, -1: no block
  double inv;

  __device__ static int at(int x, int y) {
    const int r = max(x, y), c = min(x, y);
    return ((r & 1) * 2 + (c & 1)) * HM * HM + (r >> 1) * HM + (c >> 1);
  }
  __device__ int first(int par, int pair) const { return 2 * pair + par; }
  __device__ int second(int par, int pair) const { return par && pair == h - 1 ? 0 : 2 * pair + par + 1; }

  // load(i, j): element i >= j of the matrix; row(r, k): column k of row r of V.  Both are asked for n only.
  template <class L, class R>
  __device__ Jacobi(double *lds, int n, L &&load, R &&row) {
    rot = reinterpret_cast<double2 *>(lds);
    A = lds + kWaves * 2 * HM;
    diag = A + 4 * HM * HM, piv = diag + 4 * HM, red = piv + 2 * HM;
    const int lane = threadIdx.x & 63;
    wave = threadIdx.x >> 6;
    rot += wave * HM;
    h = max(3, (n + 1) / 2), i = lane % W, g = wave * G + lane / W;
    double big = 0.0;
    for (int x = threadIdx.x; x < 4 * h * h; x += kThreads) {
      const int r = x / (2 * h), c = x - r * 2 * h;
      if (c > r) continue;
      const double e = r < n ? load(r, c) : 0.0, f = fabs(e);
      big = f > big || f != f ? f : big;
      A[at(r, c)] = e;
      if (r == c) diag[r] = e;
      if (r == c + 1 && (r & 1)) piv[c >> 1] = e;
    }
    big = wg_max(big, red);
    inv = big > 0.0 ? 1.0 / big : 0.0;
#pragma unroll
    for (int k = 0; k < kRows; ++k) {
      const int r = g + kGroups * k;
#pragma unroll
      for (int b = 0; b < 2; ++b) v[k][b] = i < h && r < n && 2 * i + b < n ? row(r, 2 * i + b) : 0.0;
    }
#pragma unroll
    for (int k = 0; k < kBlocks; ++k) {
      const int d = kGroups - g + kGroups * k;  // the waves with the fewest rows of V take a distance more
      const bool on = i < h && 2 * d <= h && !(2 * d == h && i >= d);
      mate[k] = on ? (i + d >= h ? i + d - h : i + d) : -1;
      if (on)
#pragma unroll
        for (int par = 0; par < 2; ++par) {
          const int x1 = first(par, i), x2 = second(par, i), y1 = first(par, mate[k]), y2 = second(par, mate[k]);
          adr[par][k][0] = at(x1, y1), adr[par][k][1] = at(x1, y2), adr[par][k][2] = at(x2, y1), adr[par][k][3] = at(x2, y2);
        }
    }
  }

  // PAR: 0 an even, 1 an odd step.
  template <int PAR>
  __device__ void step() {
    const bool act = i < h, ends = PAR && i >= h - 1;
    const int p = act ? first(PAR, i) : 0, q = act ? second(PAR, i) : 0;
    const double app = diag[PAR * 2 * HM + p], aqq = diag[PAR * 2 * HM + q], apq = piv[PAR * HM + (act ? i : 0)];
    double a[kBlocks][4];  // in flight while the rotation is computed
#pragma unroll
    for (int k = 0; k < kBlocks; ++k)
      if (mate[k] >= 0)
#pragma unroll
        for (int e = 0; e < 4; ++e) a[k][e] = A[adr[PAR][k][e]];
    const double gap = aqq - app;
    const float hf = float(0.5 * gap * inv), af = float(apq * inv);
    const float den = fabsf(hf) + __builtin_amdgcn_sqrtf(hf * hf + af * af);
    // below the normal numbers the reciprocal is infinite; gap and pivot are then 1e-19 of the largest at most
    const float t = den >= 0x1p-126f ? copysignf(1.0f, hf) * af * __builtin_amdgcn_rcpf(den) : 0.0f;
    const double tau = double(t * __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_sqrtf(1.0f + t * t)));
    const double x = fma(tau, tau, 1.0);
    double y = __builtin_amdgcn_rcp(x);
    y = fma(y, fma(-x, y, 1.0), y);
    y = fma(y, fma(-x, y, 1.0), y);
    double sn = 2.0 * tau * y, cs = fma(-sn, tau, 1.0);
    if (ends) sn = 1.0, cs = 0.0;
    if (i < HM && (W == 64 || (threadIdx.x & 63) < W)) rot[i] = make_double2(cs, sn);
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
    if (g == 0 && act) {
      // the swapped pair's diagonal for the next step, and what is left of the pivot (turned at the ends)
      const double cross = cs * sn, move = fma(2.0 * cross, apq, -(sn * sn) * gap);
      diag[(PAR ^ 1) * 2 * HM + p] = ends ? app : aqq + move;
      diag[(PAR ^ 1) * 2 * HM + q] = ends ? aqq : app - move;
      const int o = at(p, q);
      A[o] = ends ? -A[o] : fma(-cross, gap, fma(-2.0 * sn * sn, apq, apq));
    }
#pragma unroll
    for (int k = 0; k < kRows; ++k)
      if (k == 0 || wave * G + kGroups * k < 2 * h) {
        if (PAR) {
          const double f = v[k][1], s = from_next(v[k][0]);
          v[k][1] = fma(cs, s, sn * f);
          v[k][0] = from_prev(fma(-sn, s, cs * f));
        } else {
          const double f = v[k][0], s = v[k][1];
          v[k][0] = fma(cs, s, sn * f);
          v[k][1] = fma(-sn, s, cs * f);
        }
      }
#pragma unroll
    for (int k = 0; k < kBlocks; ++k)
      if (mate[k] >= 0) {
        const double2 o = rot[mate[k]];
        double b[4];  // the mate's rotation, then this lane's
        b[0] = fma(o.x, a[k][1], o.y * a[k][0]), b[1] = fma(-o.y, a[k][1], o.x * a[k][0]);
        b[2] = fma(o.x, a[k][3], o.y * a[k][2]), b[3] = fma(-o.y, a[k][3], o.x * a[k][2]);
        const double c2 = fma(-sn, b[2], cs * b[0]);
        A[adr[PAR][k][0]] = fma(cs, b[2], sn * b[0]);
        A[adr[PAR][k][1]] = fma(cs, b[3], sn * b[1]);
        A[adr[PAR][k][2]] = c2;
        A[adr[PAR][k][3]] = fma(-sn, b[3], cs * b[1]);
        // neighbours (distance 1): the second of this pair and the first of the next meet in the next step
        if (k == 0 && g == kGroups - 1) piv[(PAR ^ 1) * HM + (PAR ? mate[k] : i)] = c2;
      }
    __syncthreads();
  }

  // Diagonalizes; returns the sweeps done, an odd number of which leaves index k at position 2 h - 1 - k.
  // The eigenvalue at position x is diag[x]; *ok: the sweeps ended by themselves.
  __device__ int run(bool *ok) {
    for (int sweep = 1; sweep <= kSweeps; ++sweep) {
      for (int s = 0; s < h; ++s) {
        step<0>();
        step<1>();
      }
      double off = 0.0;
      for (int r = wave; r < h; r += kWaves)
        for (int c = threadIdx.x & 63; c <= r; c += 64)
#pragma unroll
          for (int e = 0; e < 4; ++e)
            if (c < r || e == 2) {
              const double f = fabs(A[e * HM * HM + r * HM + c]) * inv;
              off = f > off || f != f ? f : off;
            }
      off = wg_max(off, red);
      if (off <= 0x1p-51) {
        *ok = true;
        return sweep;
      }
    }
    *ok = false;
    return kSweeps;
  }
};

}  // namespace zqj
