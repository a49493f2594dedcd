// Device pieces shared by the SCF's density and DIIS kernels, and the whole of an SCF iteration after the
// Fock build as one workgroup (scf_step), for padded sizes up to 16 kStepTiles.
//
// scf_step serves both the device SCF of one molecule (zq_scf_dev.hip) and the batch (zq_group.hip): energy,
// DIIS error, history, bordered LU and extrapolation (src/hartree_fock.zig:176-227,643-683,810-845),
// F' = X^T F X, SP2 with certified folds (see zq_dense.hip), P = f X D X^T (:621-640) and the convergence
// test (:853-870).
#pragma once

#include <hip/hip_runtime.h>

#include "zq_internal.h"
#include "zq_tile.h"

namespace zqs {

using namespace zqt;

// Sp2Bufs::est, in doubles: the fold bookkeeping kept across the SP2 runs of one device SCF.
enum : int {
  kEstValid = 0,      // 1: ref holds F' of a settled plain run, and kEstHomo / kEstLumo bound its HOMO / LUMO
  kEstHomo = 1,       // upper bound of that run's HOMO energy
  kEstLumo = 2,       // lower bound of its LUMO energy
  kEstLastPlain = 3,  // 1: the last run was plain: ref holds its F', its traces are in the history
  kEstLastLo = 4,     // and its Gershgorin interval
  kEstLastHi = 5,
  kEstFold = 6,       // this run folds, with the bounds kEstA0 (virtual) and kEstB0 (occupied) in X_0's scale
  kEstA0 = 7,
  kEstB0 = 8,
  kEstSteps = 9,      // steps the last run recorded, and whether it settled
  kEstSettled = 10,
  kEstRuns = 11,      // since the SCF's first density: densities, folded ones, SP2 steps in all
  kEstFolds = 12,
  kEstStepSum = 13,
  kEstRefSel = 14,    // which of the two n x n reference buffers holds F'_ref
  kEstHist = 16,      // history[k] = {tr X_k, tr X_k^2, 1 for a down step, fold point}
  kEstSize = kEstHist + 4 * kSp2MaxSteps
};

// HOMO (upper bound) and LUMO (lower bound) energies of the last plain run (steps steps, Gershgorin
// interval [lo, hi]) from its trace history h (a copy in LDS of est + kEstHist).
__device__ inline bool sp2_estimate(int steps, double lo, double hi, const double *h, int nocc, double &eh, double &el) {
  int ks = -1;
  for (int k = 0; k < steps && ks < 0; ++k)
    if (h[4 * k] - h[4 * k + 1] < 1e-3) ks = k;
  if (ks < 0) return false;
  const double idem = h[4 * ks] - h[4 * ks + 1], d = h[4 * ks] - double(nocc), r = 4.0 * idem * idem + 1e-12;
  double xl = fmin(fmax(0.5 * (idem + d) + r, 0.0), 1.0), xh = fmin(fmax(1.0 - (0.5 * (idem - d) + r), 0.0), 1.0);
  for (int k = ks - 1; k >= 0; --k) {
    if (h[4 * k + 2] != 0.0) {
      xl = sqrt(xl), xh = sqrt(xh);
    } else {
      xl = 1.0 - sqrt(fmax(1.0 - xl, 0.0)), xh = 1.0 - sqrt(fmax(1.0 - xh, 0.0));
    }
  }
  const double inv = 1.0 / fmax(hi - lo, 1e-10 * fmax(1.0, fabs(hi)));
  eh = hi - xh / inv;
  el = hi - xl / inv;
  return el > eh;
}

// What a run's fold decision needs of the bookkeeping in est; track as in zq_sp2_enqueue (1: the first
// density of an SCF, 2: a later one).
struct FoldBook {
  double valid, homo, lumo, lo, hi, runs, folds;
  int steps, sel;
  bool last_plain, pending;  // pending: the last run was plain and settled, its history gives the bounds
};

__device__ inline FoldBook fold_book(const double *est, int track) {
  FoldBook b;
  b.valid = est[kEstValid], b.homo = est[kEstHomo], b.lumo = est[kEstLumo];
  b.lo = est[kEstLastLo], b.hi = est[kEstLastHi], b.steps = int(est[kEstSteps]);
  b.sel = int(est[kEstRefSel]) & 1;
  b.runs = est[kEstRuns], b.folds = est[kEstFolds];
  b.last_plain = est[kEstLastPlain] != 0.0;
  b.pending = track == 2 && b.last_plain && est[kEstSettled] != 0.0;
  return b;
}

// Whether this run folds, and its bounds a0, b0 in X_0's scale.  emin, emax: its Gershgorin interval;
// dsum, dmax: ||F' - F'_ref||_F^2 and the largest row sum of |F' - F'_ref|; found, eh, el: sp2_estimate on
// the pending history.  Updates est (one thread).
__device__ inline bool fold_decide(double *est, const FoldBook &k, int track, bool found, double eh,
                                   double el, double emin, double emax, double dsum, double dmax, double &a0,
                                   double &b0) {
  bool fold = false;
  double valid = track == 1 ? 0.0 : k.valid, runs = k.runs, folds = k.folds;
  if (track == 2 && k.last_plain) {
    // ref holds the last run's F': its history gives the bounds, when it settled
    valid = 0.0;
    if (found) {
      est[kEstHomo] = eh, est[kEstLumo] = el;
      valid = 1.0;
    }
  }
  if (!found) eh = k.homo, el = k.lumo;
  est[kEstValid] = valid;
  if (valid != 0.0) {
    // ||F' - F'_ref||_2 is at most its Frobenius norm and at most its largest absolute row sum
    // (F' symmetric); the row sum is often the smaller one early in an SCF.  A relative pad covers
    // the rounding of both sums.
    const double D = fmin(sqrt(dsum), dmax) * (1.0 + 1e-12);
    const double lumo = el - D, homo = eh + D;
    if (lumo - homo > 0.5 * (el - eh)) {
      const double inv = 1.0 / fmax(emax - emin, 1e-10 * fmax(1.0, fabs(emax)));
      fold = true;
      a0 = fmin(fmax((emax - lumo) * inv, 0.0), 1.0);
      b0 = fmin(fmax((emax - homo) * inv, 0.0), 1.0);
      est[kEstA0] = a0, est[kEstB0] = b0;
    }
  }
  est[kEstFold] = fold ? 1.0 : 0.0;
  est[kEstLastPlain] = fold ? 0.0 : 1.0;
  if (!fold) est[kEstRefSel] = double(k.sel ^ 1);
  if (track == 1) runs = 0.0, folds = 0.0, est[kEstStepSum] = 0.0;
  est[kEstRuns] = runs + 1.0;
  est[kEstFolds] = folds + (fold ? 1.0 : 0.0);
  if (!fold) est[kEstLastLo] = emin, est[kEstLastHi] = emax;
  return fold;
}

// The polynomial of one step, X_(k+1) = alpha X_k^2 + beta X_k + gamma I; s is the fold point (0 plain).
struct Sp2Map {
  double alpha, beta, gamma, s;
  bool down;
};

// The stop rule and the step's map from the summed partials (t1 = tr X_k, t2 = tr X_k^2 over the m x m
// grid): count < 0 before idem < tol was first seen, then the number of steps taken since; the step that
// brings count to 2 produces the settled projector.  Plain: X^2 or 2X - X^2, whichever keeps the trace
// closer to N.  Folding (bounds a < b carried in a, b): the folded map of the side whose bound lags,
// down when a > 1 - b, else up; both bounds go through it.  (The trace rule cannot choose between
// folded maps: a folded down step lifts every eigenvalue near 0, the zero padding included, to
// s^2/(1-s)^2, which makes its trace look worse than it is and keeps the iteration going up.)
__device__ inline Sp2Map sp2_map(double t1, double t2, double tol, int nocc, int &count, bool fold, double &a,
                                 double &b) {
  const double N = double(nocc);
  if (count < 0 && t1 - t2 < tol) count = 0;
  if (count >= 0) ++count;
  Sp2Map p;
  if (!fold || !(b > a)) {
    p.down = fabs(t2 - N) <= fabs(2.0 * t1 - t2 - N);
    p.alpha = p.down ? 1.0 : -1.0, p.beta = p.down ? 0.0 : 2.0, p.gamma = 0.0, p.s = 0.0;
    return p;
  }
  const double sd = 0.5 * a, su = 0.5 * (1.0 - b);
  const double cd = 1.0 / (1.0 - sd), cu = 1.0 / (1.0 - su);
  p.down = a > 1.0 - b;
  if (p.down)
    p.alpha = cd * cd, p.beta = -2.0 * sd * cd * cd, p.gamma = sd * sd * cd * cd, p.s = sd;
  else
    p.alpha = -cu * cu, p.beta = 2.0 * cu, p.gamma = 0.0, p.s = su;
  // the roundings written out: every kernel that inlines this takes the same bounds to the last bit
  a = fma(a, p.alpha * a, p.beta * a) + p.gamma;
  b = fma(b, p.beta, b * (p.alpha * b)) + p.gamma;
  return p;
}

constexpr int kMaxHist = 16;

struct ScfState {
  int done;       // 0 running, 1 converged, 2 iteration limit reached, 3 SP2 did not settle in its budget
  int it;         // iterations completed
  int sp2_steps;  // SP2 steps of the last density
  int sp2_max;    // most SP2 steps of any density so far
  int hist_n, cur, combine;
  int resets;          // singular DIIS systems met (the history reset to the current entry)
  int hist[kMaxHist];  // DIIS slots, oldest first
  int sp2[6];          // SP2 {count, steps} pairs, the settled buffer's parity, the abort flag
  double e_old, e_new, rms, dE;
  double coef[kMaxHist + 1];
  double B[kMaxHist * kMaxHist];  // B[slot][slot] = <err_slot, err_slot'>
};

// The host's view of a device SCF, in pinned memory: word holds done << 32 | iterations completed and is
// written last, once per iteration; the rest is valid once done is set.
struct ScfProgress {
  unsigned long long word;
  double energy;
  int it, resets;
  int sp2[3];  // densities, folded ones, SP2 steps
};

// One thread, at the end of an iteration (or of one that found done already set).
__device__ inline void report(const ScfState *st, const double *est, ScfProgress *p) {
  if (st->done) {
    p->energy = st->e_new, p->it = st->it, p->resets = st->resets;
    for (int k = 0; k < 3; ++k) p->sp2[k] = int(est[kEstRuns + k]);
  }
  __hip_atomic_store(&p->word, (unsigned long long)(st->done) << 32 | unsigned(st->it), __ATOMIC_RELEASE,
                     __HIP_MEMORY_SCOPE_SYSTEM);
}

// Slot of the next iteration's error/Fock pair: the oldest when the history is full, else the lowest
// free.  Taken at the end of the previous iteration (k_converge) or by k_state_init for the first.
__device__ inline void diis_next_slot(ScfState *st, int diis) {
  int slot;
  if (st->hist_n >= diis) {
    slot = st->hist[0];
    for (int k = 1; k < st->hist_n; ++k) st->hist[k - 1] = st->hist[k];
    --st->hist_n;
  } else {
    slot = 0;
    for (bool used = true; used; ) {
      used = false;
      for (int k = 0; k < st->hist_n; ++k) used |= st->hist[k] == slot;
      if (used) ++slot;
    }
  }
  st->hist[st->hist_n++] = slot;
  st->cur = slot;
}

// Orders this wave's LDS accesses before it against those after it, for exchanges inside one wave.
__device__ inline void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// LU with partial pivoting and the triangular solves of the host zq::getrf/getrs, on one wave: row i
// of A (n <= kLuMax) in LDS at A[i * kLuLd], b[i] in lane i's register.  Every element sees the same
// operations in the same order as in the serial steps: the same pivot (the first row with the largest
// |A[i][k]|), the same multipliers and updates, the forward sums in ascending j, the backward sums in
// ascending j.  The rows of b are swapped as the pivots are found, which permutes b exactly as applying
// the swaps afterwards does.  The loops run to n, not to kLuMax: the code stays small, which matters for
// a kernel that runs once per iteration with its instructions not in the cache.  Returns false, on every
// lane, for a zero pivot; otherwise lane i < n holds x[i] in b.
// (LDS hand-overs inside the wave only: other waves of the workgroup need not take part.)
constexpr int kLuMax = kMaxHist + 1;
constexpr int kLuLd = kLuMax + 1;  // row stride of A in LDS

// lane src's v on every lane; src is wave-uniform, so this is two v_readlane, not an LDS permute
__device__ inline double lane_bcast(double v, int src) {
  return __hiloint2double(__builtin_amdgcn_readlane(__double2hiint(v), src),
                          __builtin_amdgcn_readlane(__double2loint(v), src));
}

__device__ inline bool lu_solve_lds(int n, double *A, double &b) {
  const int lane = threadIdx.x & 63;
  for (int k = 0; k < n; ++k) {
    // pivot: every lane scans column k in row order, so all find the same row
    int p = k;
    double best = fabs(A[k * kLuLd + k]);
    for (int i = k + 1; i < n; ++i) {
      const double v = fabs(A[i * kLuLd + k]);
      if (v > best) best = v, p = i;
    }
    if (best == 0.0) return false;
    p = __builtin_amdgcn_readfirstlane(p);
    if (p != k) {
      if (lane < n) {  // lane j swaps column j of rows k and p
        const double rk = A[k * kLuLd + lane], rp = A[p * kLuLd + lane];
        A[k * kLuLd + lane] = rp;
        A[p * kLuLd + lane] = rk;
      }
      const double bk = lane_bcast(b, k), bp = lane_bcast(b, p);
      b = lane == k ? bp : (lane == p ? bk : b);
      wave_lds_sync();
    }
    if (lane > k && lane < n) {
      const double f = A[lane * kLuLd + k] / A[k * kLuLd + k];
      A[lane * kLuLd + k] = f;
      for (int j = k + 1; j < n; ++j) A[lane * kLuLd + j] -= f * A[k * kLuLd + j];
    }
    wave_lds_sync();
  }
  for (int j = 0; j < n; ++j) {
    const double bj = lane_bcast(b, j);
    if (lane > j && lane < n) b -= A[lane * kLuLd + j] * bj;
  }
  for (int i = n - 1; i >= 0; --i) {
    double acc = b;
    for (int j = i + 1; j < n; ++j) {
      const double bj = lane_bcast(b, j);
      if (lane < n) acc -= A[lane * kLuLd + j] * bj;
    }
    if (lane == i) b = acc / A[i * kLuLd + i];
  }
  return true;
}

// lu_solve_lds for systems of at most kLuSmall rows (a DIIS history of 8), the same operations in the same
// order on rows that stay in the registers of their lane: a swap exchanges two lanes' positions, not their
// data.  After step k the columns shift by one, so that the pivot column is always element 0 and the step
// loop stays rolled (its instructions are rarely in the cache).  The pivot is the row of largest |A[i][k]|,
// the first in position order among equals: a 16-lane maximum of the high words, then of the low words and
// positions only where rows tie.  Finished rows of U and their right-hand sides go to LDS at A[k * kLuLd],
// from where the back-substitution reads them once.  Dependent LDS reads and writes per element made it
// 17,000 cycles for a history of 8; this takes about 7,000.
constexpr int kLuSmall = 9;

// Largest v over each 16-lane row, on all of its lanes.
__device__ inline int row_max(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0xB1, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x4E, 0xF, 0xF, false));
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x141, 0xF, 0xF, false));
  return max(v, __builtin_amdgcn_update_dpp(0, v, 0x128, 0xF, 0xF, false));
}

__device__ inline bool lu_solve_small(int n, double *A, double &b) {
  const int lane = threadIdx.x & 63;
  double a[kLuSmall + 1];
#pragma unroll
  for (int j = 0; j < kLuSmall; ++j) a[j] = lane < n && j < n ? A[lane * kLuLd + j] : 0.0;
  a[kLuSmall] = 0.0;
  int pos = lane < n ? lane : kLuMax;  // position of this lane's row
  wave_lds_sync();
  for (int k = 0; k < n; ++k) {
    const bool open = pos >= k && pos < n;
    const double v = fabs(a[0]);
    const int hi = open ? __double2hiint(v) : -1;
    const int most = __builtin_amdgcn_readfirstlane(row_max(hi));  // on every lane: a butterfly needs them all
    unsigned long long cand = __ballot(open && hi == most);
    if (cand & (cand - 1)) {  // (rare) equal high words: the low words (biased to signed order), then the positions
      const bool in = cand >> lane & 1;
      const int lo = in ? int(unsigned(__double2loint(v)) ^ 0x80000000u) : int(0x80000000u);
      const int most_lo = __builtin_amdgcn_readfirstlane(row_max(lo));
      cand = __ballot(in && lo == most_lo);
      const bool in2 = cand >> lane & 1;
      const int first = -__builtin_amdgcn_readfirstlane(row_max(in2 ? -pos : -kLuMax - 1));
      cand = __ballot(in2 && pos == first);
    }
    const int p = __builtin_amdgcn_readfirstlane(__ffsll(cand) - 1);  // the pivot row's lane
    const double piv = lane_bcast(a[0], p), bk = lane_bcast(b, p);
    if (piv == 0.0) return false;
    const int ppos = __builtin_amdgcn_readlane(pos, p);
    pos = lane == p ? k : (pos == k ? ppos : pos);
    if (lane == p) {
#pragma unroll
      for (int j = 0; j < kLuSmall; ++j)
        if (k + j < n) A[k * kLuLd + k + j] = a[j];
      A[k * kLuLd + kLuMax] = b;
    }
    const double f = pos > k && pos < n ? a[0] / piv : 0.0;  // 0 leaves a finished row as it is
    b = fma(-f, bk, b);
#pragma unroll
    for (int j = 1; j < kLuSmall; ++j) a[j - 1] = fma(-f, lane_bcast(a[j], p), a[j]);
    a[kLuSmall - 1] = 0.0;
  }
  wave_lds_sync();
  const double rhs = lane < n ? A[lane * kLuLd + kLuMax] : 0.0;
#pragma unroll
  for (int j = 0; j < kLuSmall; ++j) a[j] = lane < n && j >= lane && j < n ? A[lane * kLuLd + j] : 1.0;
  double x[kLuSmall];
#pragma unroll
  for (int i = kLuSmall - 1; i >= 0; --i) {
    double acc = rhs;
#pragma unroll
    for (int j = i + 1; j < kLuSmall; ++j)
      if (j < n) acc = fma(-a[j], x[j], acc);
    x[i] = lane_bcast(acc / a[i], i);
    if (lane == i && i < n) b = x[i];
  }
  return true;
}

__device__ inline bool lu_solve(int n, double *A, double &b) {
  return n <= kLuSmall ? lu_solve_small(n, A, b) : lu_solve_lds(n, A, b);
}

// ------------------------------------------------------------------------------------------ scf_step
// One SCF iteration after the Fock build (or the core-Hamiltonian guess density) as one workgroup.
//
// At these sizes the iteration is a chain of ~16 dependent steps of a microsecond or less each, so as
// separate launches it costs their ~5 us of launch and drain each, and SP2 spread over workgroups costs a
// 3-4 us cross-XCD hand-over per step.  Here every n x n product runs on operands in LDS: two MP x (MP + 2)
// buffers (MP = 16 T; the row stride keeps rows 16-byte aligned and the 16 rows of a tile in distinct
// banks), the tiles of a product dealt over the waves and kept in registers until every wave has read the
// operands, then written over one of them.  SP2 ping-pongs between the buffers with one barrier per step and
// forms the upper tiles only.
//
// The sums of F', D and P are taken in the order of the multi-launch form (zq_scf_dev.hip, zq_dense.hip).  The DIIS
// dot products and rms(dP) are not (that form sums both tile by tile), so the two forms agree to rounding, not to the
// bit.  The order here stays as it is: the signs of the orbitals of a symmetric molecule hang on the last bits of F'.
//
// Matrices in global memory are n x n with a leading dimension each, or n n contiguous (history, reference).
constexpr int kStepTiles = 6;  // largest T that fits: 2 x 96 x 98 doubles of LDS

enum { kStepGuess = 0, kStepIter = 1 };

struct StepArgs {
  ScfState *st;
  const double *H, *F;  // ldh
  double *P, *dP;       // ldp; dP (P_new - P_old) may be null
  const double *S, *X, *XT;  // ldm
  double *W;            // ldm: the (extrapolated) Fock matrix that is diagonalised
  double *Fh, *Eh;      // history slots
  double *ref;          // the two buffers of the fold reference
  double *est;          // fold bookkeeping
  const double *epart;  // energy partials of the J/K reduce; null: the energy is summed here
  int *done_out;        // receives st->done at the end (may be null)
  ScfProgress *progress;  // the host's view of the run (may be null)
  int nep, ldh, ldp, ldm, n, nocc, diis, maxit, nsteps, mode;
  double factor, VN, thr, err_scale;
};

struct StepShared {
  double red[16];                        // per-wave partials
  double2 part[2][kStepTiles * (kStepTiles + 1) / 2];  // the tiles' partial traces, by step parity
  double rows[4][64];                    // per virtual wave of the Gershgorin pass: min, max, dd, row-sum max
  double hist[4 * kSp2MaxSteps];
  double Bs[kMaxHist * kMaxHist], Alu[kLuMax * kLuLd], dots[kMaxHist], coef[kMaxHist];
  double scal[6];                        // emin, emax, a0, b0, HOMO and LUMO estimates
  int hs[kMaxHist];
  double map[3];                         // alpha, beta, gamma of the SP2 step
  int m, cur, comb, fold, found, count;
};

// Dynamic LDS of scf_step for padded size mp.
__host__ __device__ constexpr size_t step_lds_bytes(int mp) { return 2 * size_t(mp) * (mp + 2) * sizeof(double); }

__device__ inline double perm16_other(double v) {  // v and its partner at lane ^ 16, in either order
  const auto lo = __builtin_amdgcn_permlane16_swap(unsigned(__double2loint(v)), unsigned(__double2loint(v)), false, false);
  const auto hi = __builtin_amdgcn_permlane16_swap(unsigned(__double2hiint(v)), unsigned(__double2hiint(v)), false, false);
  return fmax(__hiloint2double(int(hi[0]), int(lo[0])), __hiloint2double(int(hi[1]), int(lo[1])));
}
__device__ inline double perm32_other(double v) {
  const auto lo = __builtin_amdgcn_permlane32_swap(unsigned(__double2loint(v)), unsigned(__double2loint(v)), false, false);
  const auto hi = __builtin_amdgcn_permlane32_swap(unsigned(__double2hiint(v)), unsigned(__double2hiint(v)), false, false);
  return fmax(__hiloint2double(int(hi[0]), int(lo[0])), __hiloint2double(int(hi[1]), int(lo[1])));
}

// Sum over the wave as a tree from lane distance 32 down to 1 (the order of a halving tree in LDS).
__device__ inline double wave_tree(double v) {
  v = add_swap32(v);
  v = add_swap16(v);
  v += dpp_mov<0x128>(v);
  v += dpp_mov<0x1B>(dpp_mov<0x141>(v));  // lane ^ 4: half-row mirror, then the quad reversed
  v += dpp_mov<0x4E>(v);
  return v + dpp_mov<0xB1>(v);
}

// The 16 x 16 tile of A B^T over K = 16 T from LDS rows A and B (row 0 of the tile each, stride LD): lane
// (r, q) reads 4 consecutive k of its rows per 16-wide chunk, element t of every lane in MFMA t.  SPLIT
// keeps chunk c's products in accumulator c & 3, added up in order (the K split of the SP2 kernels).
template <int T, bool SPLIT>
__device__ inline d4 lds_tile_nt(const double *A, const double *B) {
  constexpr int LD = 16 * T + 2, NA = SPLIT ? (T < 4 ? T : 4) : 1;
  const int lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
  const double2 *a = reinterpret_cast<const double2 *>(A + r * LD + 4 * q);
  const double2 *b = reinterpret_cast<const double2 *>(B + r * LD + 4 * q);
  d4 acc[NA];
#pragma unroll
  for (int x = 0; x < NA; ++x) acc[x] = d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
  for (int c = 0; c < T; ++c) {
    const double2 a0 = a[8 * c], a1 = a[8 * c + 1], b0 = b[8 * c], b1 = b[8 * c + 1];
    d4 &s = acc[c % NA];
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a0.x, b0.x, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a0.y, b0.y, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a1.x, b1.x, s, 0, 0, 0);
    s = __builtin_amdgcn_mfma_f64_16x16x4f64(a1.y, b1.y, s, 0, 0, 0);
  }
#pragma unroll
  for (int x = 1; x < NA; ++x) acc[0] += acc[x];
  return acc[0];
}

// Upper tile t of T (T + 1) / 2, row by row.
template <int T>
__device__ inline void upper_tile(int t, int &ti, int &tj) {
  ti = 0;
  while (t >= T - ti) t -= T - ti, ++ti;
  tj = ti + t;
}

template <int NT, int T>
struct StepBody {
  static constexpr int MP = 16 * T, LD = MP + 2, MM = MP * MP, NW = NT / 64, TU = T * (T + 1) / 2;
  static constexpr int NE = (MM + NT - 1) / NT;  // elements per thread
  static constexpr bool kEarly = T <= 4;
  static constexpr int NF = (T * T + NW - 1) / NW, NU = (TU + NW - 1) / NW;  // tiles per wave: all, upper

  // element u of this thread in the MP x MP grid; false past the end
  static __device__ bool elem(int u, int &i, int &j) {
    const int x = int(threadIdx.x) + NT * u;
    i = x / MP, j = x - i * MP;
    return MM % NT == 0 || x < MM;
  }
  static __device__ void load(double (&v)[NE], const double *src, int ld, int n) {
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      int i, j;
      v[u] = (elem(u, i, j) && i < n && j < n) ? src[size_t(i) * ld + j] : 0.0;
    }
  }
  static __device__ void put(double *dst, const double (&v)[NE]) {
#pragma unroll
    for (int u = 0; u < NE; ++u) {
      int i, j;
      if (elem(u, i, j)) dst[i * LD + j] = v[u];
    }
  }
  // every tile of A B^T, kept in registers
  static __device__ void product(d4 (&acc)[NF], const double *A, const double *B) {
    const int wave = threadIdx.x >> 6;
#pragma unroll
    for (int u = 0; u < NF; ++u) {
      const int t = wave + u * NW;
      if (t < T * T) acc[u] = lds_tile_nt<T, false>(A + (t / T) * 16 * LD, B + (t % T) * 16 * LD);
    }
  }
  // f(u, element j, row, column) for every element of this wave's tiles of a full product
  template <class Fn>
  static __device__ void each_full(Fn f) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int u = 0; u < NF; ++u) {
      const int t = wave + u * NW;
      if (t < T * T)
#pragma unroll
        for (int j = 0; j < 4; ++j) f(u, j, (t / T) * 16 + 4 * j + q, (t % T) * 16 + r);
    }
  }
  static __device__ void put_tiles(double *dst, const d4 (&acc)[NF]) {
    each_full([&](int u, int j, int row, int col) { dst[row * LD + col] = acc[u][j]; });
  }
  // This wave's upper tiles of an SP2 iterate, y(u, j, row, column) each: into dst with their mirror, and
  // their partial traces.
  template <class Fn>
  static __device__ void sp2_put(double *dst, double2 *part, Fn y) {
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, r = lane & 15, q = lane >> 4;
#pragma unroll
    for (int u = 0; u < NU; ++u) {
      const int t = wave + u * NW;
      if (t >= TU) continue;
      int ti, tj;
      upper_tile<T>(t, ti, tj);
      double s1 = 0.0, s2 = 0.0;
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int row = ti * 16 + 4 * j + q, col = tj * 16 + r;
        const double v = y(u, j, row, col);
        if (row == col) s1 += v;
        s2 = fma(v, v, s2);
        dst[row * LD + col] = v;
        if (ti != tj) dst[col * LD + row] = v;
      }
      s1 = ti == tj ? wave_sum(s1) : 0.0;
      s2 = wave_sum(s2);
      if (lane == 0) part[t] = make_double2(s1, ti == tj ? s2 : 2.0 * s2);
    }
  }

  // The DIIS system of the m entries sh.hs (the new one in slot cur) on one wave: sh.comb and sh.coef, or the
  // reset to the current entry when it is singular.  sh.dots holds the new row by history position.
  // sh.Bs holds the B of the earlier entries by slot.
  static __device__ void diis_solve(StepShared &sh, ScfState *st, int m, int cur) {
    const int lane = threadIdx.x & 63;
    if (lane < m) st->B[cur * kMaxHist + sh.hs[lane]] = st->B[sh.hs[lane] * kMaxHist + cur] = sh.dots[lane];
    if (m >= 2) {
      // the bordered system [B -1; -1 0] c = [0; -1]
      for (int idx = lane; idx < (m + 1) * (m + 1); idx += 64) {
        const int i = idx / (m + 1), j = idx - i * (m + 1);
        double v = i == j ? 0.0 : -1.0;
        if (i < m && j < m) {
          const int si = sh.hs[i], sj = sh.hs[j];
          v = (si == cur || sj == cur) ? sh.dots[si == cur ? j : i] : sh.Bs[si * kMaxHist + sj];
        }
        sh.Alu[i * kLuLd + j] = v;
      }
      double c = lane == m ? -1.0 : 0.0;
      wave_lds_sync();
      if (lu_solve(m + 1, sh.Alu, c)) {
        if (lane < m) sh.coef[lane] = c;
        if (lane == 0) sh.comb = 1;
      } else if (lane == 0) {
        st->hist[0] = cur, st->hist_n = 1;
        ++st->resets;
      }
    }
  }

  // <err_new, err_k> of every history entry k < m into sh.dots: products of 256 consecutive elements summed
  // as a halving tree, the nb (at most 36) trees by wave_sum.  er: err_new, n n contiguous in LDS; tree: nb m
  // doubles of LDS.  A wave takes (tree, entry) pairs, four of them in flight.
  static __device__ void diis_dots(StepShared &sh, const double *er, double *tree, const double *Eh, int nn, int m) {
#pragma clang fp contract(off)  // the trees sum rounded products, whatever is inlined around them
    const int wave = threadIdx.x >> 6, lane = threadIdx.x & 63, nb = (nn + 255) / 256, tot = nb * m;
    for (int i0 = wave; i0 < tot; i0 += 4 * NW) {
      double e[4][4];
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int idx = min(i0 + g * NW, tot - 1), k = idx / nb, b = idx - k * nb;
        const double *Ek = Eh + size_t(sh.hs[k]) * nn;
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int x = 256 * b + 64 * j + lane;
          e[g][j] = x < nn ? Ek[x] : 0.0;
        }
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const int idx = min(i0 + g * NW, tot - 1), k = idx / nb, b = idx - k * nb;
        double y[4];
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const int x = 256 * b + 64 * j + lane;
          y[j] = x < nn ? er[x] * e[g][j] : 0.0;
        }
        const double s = wave_tree((y[0] + y[2]) + (y[1] + y[3]));
        if (lane == 0) tree[k * nb + b] = s;
      }
    }
    __syncthreads();
    for (int k = wave; k < m; k += NW) {
      const double d = wave_sum(lane < nb ? tree[k * nb + lane] : 0.0);
      if (lane == 0) sh.dots[k] = d;
    }
  }

  static __device__ void run(const StepArgs &a, double *dyn, StepShared &sh) {
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, n = a.n, nn = n * n;
    ScfState *st = a.st;
    double *L0 = dyn, *L1 = dyn + MP * LD;
    const bool iter = a.mode == kStepIter;
    const int track = iter ? 2 : 1;
    double e_new = a.VN;
    // S, X^T and X are read before the first product where the registers allow (kEarly): a cold read costs
    // about as much as a product at small T
    double v[NE], ms[kEarly ? NE : 1], mxt[kEarly ? NE : 1], mx[kEarly ? NE : 1];
    // the bookkeeping of the density's fold, read early so that its latency hides behind the products
    const FoldBook book = fold_book(a.est, track);
    if (iter) {
      double f[NE];
      load(f, a.F, a.ldh, n);
      load(v, a.P, a.ldp, n);
      if constexpr (kEarly) {
        if (a.diis > 0) load(ms, a.S, a.ldm, n);
        load(mxt, a.XT, a.ldm, n);
        load(mx, a.X, a.ldm, n);
      }
      double e = 0.0;
      if (a.epart) {
        if (wave == 0)
          for (int b = lane; b < a.nep; b += 64) e += a.epart[b];
      } else {
#pragma unroll
        for (int u = 0; u < NE; ++u) {
          int i, j;
          if (elem(u, i, j) && i < n && j < n) e += 0.5 * v[u] * (a.H[size_t(i) * a.ldh + j] + f[u]);
        }
      }
      if (tid < kMaxHist) sh.hs[tid] = st->hist[tid];
      if (a.diis > 1)
        for (int x = tid; x < kMaxHist * kMaxHist; x += NT) sh.Bs[x] = st->B[x];
      if (tid == 0) sh.m = st->hist_n, sh.cur = st->cur, sh.comb = 0;
      if (tid == 64) sh.found = 0;
      if (book.pending)
        for (int x = tid; x < 4 * book.steps; x += NT) sh.hist[x] = a.est[kEstHist + x];
      put(L0, f);
      put(L1, v);
      e = wave_sum(e);
      if (lane == 0) sh.red[wave] = e;
      __syncthreads();
      e_new = sh.red[0];
      if (!a.epart)
#pragma unroll
        for (int w = 1; w < NW; ++w) e_new += sh.red[w];
      e_new += a.VN;
      if (a.diis > 0) {
        const int m = sh.m, cur = sh.cur;
        d4 acc[NF];
        if constexpr (!kEarly) load(v, a.S, a.ldm, n);
        product(acc, L0, L1);  // F P (P symmetric)
        __syncthreads();
        put_tiles(L0, acc);
        if constexpr (kEarly)
          put(L1, ms);
        else
          put(L1, v);
        __syncthreads();
        product(acc, L0, L1);  // F P S (S symmetric)
        __syncthreads();
        put_tiles(L0, acc);
        __syncthreads();
        double *Ec = a.Eh + size_t(cur) * nn, *Fc = a.Fh + size_t(cur) * nn;
#pragma unroll
        for (int u = 0; u < NE; ++u) {
          int i, j;
          if (elem(u, i, j) && i < n && j < n) {
            const double er = a.err_scale * (L0[i * LD + j] - L0[j * LD + i]);
            L1[i * n + j] = er;
            Ec[i * n + j] = er;
            Fc[i * n + j] = f[u];
          }
        }
        __syncthreads();  // also orders this workgroup's stores of E before the loads of diis_dots
        diis_dots(sh, L1, L0, a.Eh, nn, m);
        __syncthreads();
        // wave 0 solves the system while wave 1 inverts the last plain run's history
        if (wave == 0) diis_solve(sh, st, m, cur);
      }
      if (wave == 1 && lane == 0 && book.pending) {
        double eh = 0.0, el = 0.0;
        sh.found = sp2_estimate(book.steps, book.lo, book.hi, sh.hist, a.nocc, eh, el);
        sh.scal[4] = eh, sh.scal[5] = el;
      }
      if constexpr (!kEarly) load(v, a.XT, a.ldm, n);
      __syncthreads();
      if (sh.comb) {
        // F = sum_k c_k F_k over the history: every F_k is exactly symmetric, so the sum is too
        const int m = sh.m;
#pragma unroll
        for (int u = 0; u < NE; ++u) f[u] = 0.0;
        for (int k = 0; k < m; k += 2) {
          const int k1 = k + 1 < m ? k + 1 : k;
          const double *Fk = a.Fh + size_t(sh.hs[k]) * nn, *Fl = a.Fh + size_t(sh.hs[k1]) * nn;
          const double c0 = sh.coef[k], c1 = k1 > k ? sh.coef[k1] : 0.0;
          double fk[NE], fl[NE];
#pragma unroll
          for (int u = 0; u < NE; ++u) {
            int i, j;
            const bool in = elem(u, i, j) && i < n && j < n;
            fk[u] = in ? Fk[i * n + j] : 0.0, fl[u] = in ? Fl[i * n + j] : 0.0;
          }
#pragma unroll
          for (int u = 0; u < NE; ++u) {
            f[u] += c0 * fk[u];
            f[u] += c1 * fl[u];
          }
        }
      }
#pragma unroll
      for (int u = 0; u < NE; ++u) {
        int i, j;
        if (elem(u, i, j) && i < n && j < n) a.W[size_t(i) * a.ldm + j] = f[u];
      }
      put(L0, f);
      if constexpr (kEarly)
        put(L1, mxt);
      else
        put(L1, v);
    } else {
      if (tid == 0) {
        st->done = 0, st->it = 0, st->sp2_steps = 0, st->sp2_max = 0;
        st->hist_n = 0, st->cur = 0, st->combine = 0, st->resets = 0;
        st->e_old = a.VN, st->e_new = a.VN, st->rms = 0.0, st->dE = 0.0;
        if (a.diis > 0) diis_next_slot(st, a.diis);
        sh.found = 0;
      }
      load(v, a.H, a.ldh, n);
      put(L0, v);
      // W = H until the first iteration replaces it
#pragma unroll
      for (int u = 0; u < NE; ++u) {
        int i, j;
        if (elem(u, i, j) && i < n && j < n) a.W[size_t(i) * a.ldm + j] = v[u];
      }
      load(v, a.XT, a.ldm, n);
      put(L1, v);
      if constexpr (kEarly) load(mx, a.X, a.ldm, n);
    }
    __syncthreads();

    // F' = X^T W X into L0
    {
      d4 acc[NF];
      product(acc, L1, L0);  // T = X^T W (W symmetric)
      __syncthreads();
      put_tiles(L0, acc);
      __syncthreads();
      product(acc, L0, L1);  // F' = T X
      __syncthreads();
      put_tiles(L0, acc);
      __syncthreads();
    }

    // Gershgorin interval and the distance to the reference, as k_gershgorin's 64 waves take them (wave g rows
    // g, g + 64, ...); F' into the reference buffer not in use
    {
      const double *rold = a.ref + size_t(book.sel) * nn;
      double *rnew = a.ref + size_t(book.sel ^ 1) * nn;
      constexpr int NC = (MP + 63) / 64;
      for (int g = wave; g < 64; g += NW) {
        double lo = 1e300, hi = -1e300, dd = 0.0, dm = 0.0;
        if (g < n) {
          for (int i = g; i < n; i += 64) {
            double rs = 0.0, rd = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
              const int j = 64 * c + lane;
              const double y = j < n ? L0[i * LD + j] : 0.0;
              rs += fabs(y);
              if (track == 2) {
                const double df = y - (j < n ? rold[i * n + j] : 0.0);
                dd = fma(df, df, dd), rd += fabs(df);
              }
              if (j < n) rnew[i * n + j] = y;
            }
            const double d = L0[i * LD + i];
            rs = wave_sum(rs) - fabs(d);
            lo = fmin(lo, d - rs), hi = fmax(hi, d + rs);
            if (track == 2) dm = fmax(dm, wave_sum(rd));
          }
          dd = wave_sum(dd);
        }
        if (lane == 0) sh.rows[0][g] = lo, sh.rows[1][g] = hi, sh.rows[2][g] = dd, sh.rows[3][g] = dm;
      }
    }
    __syncthreads();
    if (wave == 0) {
      // the interval and the largest row sum as wave maxima, dd in k_gershgorin's order: groups of four waves
      // left to right, then the groups left to right
      auto wave_max = [](double x) {
        x = fmax(x, dpp_mov<0xB1>(x));
        x = fmax(x, dpp_mov<0x4E>(x));
        x = fmax(x, dpp_mov<0x141>(x));
        x = fmax(x, dpp_mov<0x128>(x));
        return perm32_other(perm16_other(x));
      };
      const double glo = -wave_max(-sh.rows[0][lane]), ghi = wave_max(sh.rows[1][lane]), gd = wave_max(sh.rows[3][lane]);
      const double pad = 1e-12 * fmax(fabs(glo), fabs(ghi)), emin = glo - pad, emax = ghi + pad;
      if (lane == 0) {
        const double *w = sh.rows[2];
        double dsum = ((w[0] + w[1]) + w[2]) + w[3];
        for (int g = 4; g < min(n, 64); g += 4) dsum += ((w[g] + w[g + 1]) + w[g + 2]) + w[g + 3];
        double a0 = 0.0, b0 = 1.0;
        sh.fold = fold_decide(a.est, book, track, sh.found, sh.scal[4], sh.scal[5], emin, emax, dsum, gd, a0, b0);
        sh.scal[0] = emin, sh.scal[1] = emax, sh.scal[2] = a0, sh.scal[3] = b0;
      }
    }
    __syncthreads();

    // SP2 from X_0 = (e_max I - F') / (e_max - e_min) in L1
    double fa = sh.scal[2], fb = sh.scal[3];
    const bool fold = sh.fold;
    {
      const double emax = sh.scal[1], inv = 1.0 / fmax(emax - sh.scal[0], 1e-10 * fmax(1.0, fabs(emax)));
      sp2_put(L1, sh.part[0], [&](int, int, int row, int col) {
        return row < n && col < n ? ((row == col ? emax : 0.0) - L0[row * LD + col]) * inv : 0.0;
      });
    }
    __syncthreads();
    // The step's map needs the traces of X_k, its products do not: the last wave (which has the fewest tiles)
    // sums the partials and forms the map while the others multiply.
    double *Xi = L1, *Xo = L0;
    int count = -1, steps = 0;
    for (int k = 0; k < a.nsteps; ++k) {
      const int par = k & 1;
      if (wave == NW - 1) {
        const double2 pt = lane < TU ? sh.part[par][lane] : make_double2(0.0, 0.0);
        const double t1 = wave_sum(pt.x), t2 = wave_sum(pt.y);
        const Sp2Map mp = sp2_map(t1, t2, 1e-9, a.nocc, count, fold, fa, fb);
        if (lane == 0) {
          sh.hist[4 * k] = t1, sh.hist[4 * k + 1] = t2;
          sh.hist[4 * k + 2] = mp.down ? 1.0 : 0.0, sh.hist[4 * k + 3] = mp.s;
          sh.map[0] = mp.alpha, sh.map[1] = mp.beta, sh.map[2] = mp.gamma;
          sh.count = count;
        }
      }
      steps = k + 1;
      d4 acc[NU];
#pragma unroll
      for (int u = 0; u < NU; ++u) {
        const int t = wave + u * NW;
        if (t < TU) {
          int ti, tj;
          upper_tile<T>(t, ti, tj);
          acc[u] = lds_tile_nt<T, true>(Xi + ti * 16 * LD, Xi + tj * 16 * LD);
        }
      }
      __syncthreads();
      const double alpha = sh.map[0], beta = sh.map[1], gamma = sh.map[2];
      count = sh.count;
      sp2_put(Xo, sh.part[par ^ 1], [&](int u, int j, int row, int col) {
        const double v = fma(alpha, acc[u][j], beta * Xi[row * LD + col]);
        return row == col ? v + gamma : v;
      });
      __syncthreads();
      double *t = Xi;
      Xi = Xo, Xo = t;
      if (count >= 2) break;
    }
    const bool settled = count >= 2;
    if (!fold)
      for (int x = tid; x < 4 * steps; x += NT) a.est[kEstHist + x] = sh.hist[x];
    if (tid == 0) {
      a.est[kEstSteps] = steps, a.est[kEstSettled] = settled ? 1.0 : 0.0, a.est[kEstStepSum] += steps;
      st->sp2_steps = steps;
      st->sp2_max = max(st->sp2_max, steps);
      if (iter) st->e_new = e_new;
      if (!settled) {  // no gap at the Fermi level within the budget: this density is not used
        st->done = 3;
        if (a.done_out) *a.done_out = 3;
        if (a.progress) report(st, a.est, a.progress);
      }
    }
    if (!settled) return;

    // P = f X D X^T; D is in Xi
    if constexpr (kEarly) {
      put(Xo, mx);
    } else {
      load(v, a.X, a.ldm, n);
      put(Xo, v);
    }
    __syncthreads();
    double s = 0.0;
    {
      d4 acc[NF], po[NF];
      product(acc, Xo, Xi);  // T = X D (D symmetric)
      __syncthreads();
      put_tiles(Xi, acc);
      // the old density of this thread's elements, its loads overlapping the product
      each_full([&](int u, int j, int row, int col) {
        po[u][j] = row < n && col < n ? a.P[size_t(row) * a.ldp + col] : 0.0;
      });
      __syncthreads();
      product(acc, Xi, Xo);  // T X^T
      each_full([&](int u, int j, int row, int col) {
        if (row >= n || col >= n) return;
        const double y = a.factor * acc[u][j], d = y - po[u][j];
        s += d * d;
        a.P[size_t(row) * a.ldp + col] = y;
        if (a.dP) a.dP[size_t(row) * a.ldp + col] = d;
      });
    }
    s = wave_sum(s);
    if (lane == 0) sh.red[wave] = s;
    __syncthreads();
    if (tid != 0) return;
    if (iter) {
      for (int w = 1; w < NW; ++w) s += sh.red[w];
      const double rms = sqrt(s / (double(n) * n)), dE = fabs(e_new - st->e_old);
      st->e_old = e_new;
      st->rms = rms, st->dE = dE;
      const bool conv = st->it > 0 && dE < a.thr && rms < a.thr;
      ++st->it;
      if (conv)
        st->done = 1;
      else if (st->it >= a.maxit)
        st->done = 2;
      else if (a.diis > 0)
        diis_next_slot(st, a.diis);
    }
    if (a.done_out) *a.done_out = st->done;
    if (a.progress) report(st, a.est, a.progress);
  }
};

}  // namespace zqs
