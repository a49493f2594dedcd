// Grouped RHF + MP2 of many small molecules (include/zinq_batch.h).
//
// Per SCF iteration, for every molecule that has not converged, three launches captured in one graph:
//   zq_jk_records / zq_jk_reduce over the grouped work plan     F = H + G(P)   (getFock, hartree_fock.zig:686-735)
//   k_batch_step, one workgroup per molecule:
//     E = 1/2 sum P (H + F) + V_NN                                (getEnergy, :643-655)
//     err = F P S - (F P S)^T, history, bordered LU, F_ext        (getError :658-683, diis :176-227, :810-845)
//     F' = X^T F_ext X, SP2 purification -> D, P = 2 X D X^T       (geigh + getDensity, :621-640)
//     rms(dP), |dE|, convergence test                            (:853-870)
//   k_batch_count: molecules done, read by the host one iteration late.
// The step is scf_step of zq_step.h, the one the device SCF of a small molecule runs, certified folds included.
// Every per-molecule matrix lives in one workspace with leading dimension mp = n rounded up to 16 and
// zero padding, so the small GEMMs of the orbitals (zq_tile.h, A B^T on FP64 MFMA, one wave per
// 16 x 16 tile) never need bounds checks.  After convergence: F' of the last extrapolated F, its eigenpairs and
// C = X V in one launch, a workgroup per molecule (zq_jacobi.h), and the MP2 energy from the OVOV transform of
// zq_transform.hip through a context that views the molecule's resident quartets.

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <string>
#include <thread>
#include <vector>

#include "../../include/zinq_batch.h"
#include "zq_internal.h"
#include "zq_jacobi.h"
#include "zq_linalg.h"
#include "zq_step.h"
#include "zq_tile.h"

using namespace zqt;
using namespace zqs;

namespace {

constexpr int kMaxN = kZqBatchMaxN;
constexpr int kHist = 8;
constexpr int kMats = 9;
enum { M_H, M_F, M_P, M_S, M_X, M_XT, M_W, M_T, M_FPR };
// matrices of mp x mp in a molecule's workspace: the above, the DIIS history of F and of the error, and the
// two buffers of the SP2 fold reference
constexpr int kWsMats = kMats + 2 * kHist + 2;
static_assert(kMaxN <= 16 * kStepTiles && kHist <= kMaxHist, "the step's limits");

struct BMol {
  long long ws;  // workspace offset (doubles): kWsMats matrices of mp x mp
  int n, mp, nocc, pad;
  double VN;
};

// What a run returns of a molecule's state.
struct BResult {
  double energy;
  int it, done;  // done: 1 converged, 2 iteration limit, 3 an SP2 density did not settle
};

// C = alpha A B^T, all mp x mp with leading dimension mp (mp a multiple of 16); the workgroup's waves
// take the 16 x 16 tiles in turn.  Ends with a barrier.
template <int NT>
__device__ void wg_gemm_nt(const double *A, const double *B, double *C, int mp, double alpha) {
  const int T = mp >> 4, waves = NT / 64, wave = threadIdx.x >> 6, lane = threadIdx.x & 63;
  const int r = lane & 15, q = lane >> 4;
  for (int t = wave; t < T * T; t += waves) {
    const int ti = t / T, tj = t - ti * T;
    const d4 acc = tile_nt<true>(A, mp, B, mp, ti * 16, tj * 16, mp, mp, mp);
#pragma unroll
    for (int j = 0; j < 4; ++j) C[size_t(ti * 16 + 4 * j + q) * mp + tj * 16 + r] = alpha * acc[j];
  }
  __syncthreads();
}

// One SCF step (kStepIter) or the core-Hamiltonian guess (kStepGuess) of molecule order[blockIdx.x]: scf_step
// on its matrices.  Against the form before it (products on operands in L2, a serial DIIS solve, all tiles of
// X^2 and no folds), per iteration of 96 molecules, n <= 72: 401 -> 198 us.
template <int NT>
__global__ __launch_bounds__(NT) void k_batch_step(double *__restrict__ ws, const BMol *__restrict__ mols,
                                                   const int *__restrict__ order, ScfState *__restrict__ st,
                                                   double *__restrict__ est, int *__restrict__ done, int mode, int diis,
                                                   double thr, int maxit) {
  extern __shared__ __attribute__((aligned(16))) double step_lds[];
  __shared__ StepShared sh;
  const int mi = order[blockIdx.x];
  if (mode == kStepIter && done[mi]) return;
  const BMol M = mols[mi];
  const size_t mm = size_t(M.mp) * M.mp;
  double *base = ws + M.ws;
  StepArgs a{};
  a.st = st + mi;
  a.H = base + M_H * mm, a.F = base + M_F * mm, a.ldh = M.mp;
  a.P = base + M_P * mm, a.ldp = M.mp;
  a.S = base + M_S * mm, a.X = base + M_X * mm, a.XT = base + M_XT * mm, a.W = base + M_W * mm, a.ldm = M.mp;
  a.Fh = base + kMats * mm, a.Eh = a.Fh + kHist * mm, a.ref = a.Eh + kHist * mm;
  a.est = est + size_t(mi) * kEstSize;
  a.done_out = done + mi;
  a.n = M.n, a.nocc = M.nocc, a.diis = diis, a.maxit = maxit, a.nsteps = 100, a.mode = mode;
  a.factor = 2.0, a.VN = M.VN, a.thr = thr, a.err_scale = 1.0;
  switch (M.mp >> 4) {
    case 1: StepBody<NT, 1>::run(a, step_lds, sh); break;
    case 2: StepBody<NT, 2>::run(a, step_lds, sh); break;
    case 3: StepBody<NT, 3>::run(a, step_lds, sh); break;
    case 4: StepBody<NT, 4>::run(a, step_lds, sh); break;
    case 5: StepBody<NT, 5>::run(a, step_lds, sh); break;
    default: StepBody<NT, 6>::run(a, step_lds, sh); break;
  }
}

__global__ void k_batch_result(const ScfState *__restrict__ st, int m, BResult *__restrict__ out) {
  const int i = blockIdx.x * blockDim.x + threadIdx.x;
  if (i < m) out[i] = BResult{st[i].e_new, st[i].it, st[i].done};
}

__global__ void k_batch_count(const int *__restrict__ done, int m, int *__restrict__ out) {
  __shared__ int red[256];
  int c = 0;
  for (int i = threadIdx.x; i < m; i += 256) c += done[i] != 0;
  red[threadIdx.x] = c;
  __syncthreads();
  for (int w = 128; w > 0; w >>= 1) {
    if (threadIdx.x < w) red[threadIdx.x] += red[threadIdx.x + w];
    __syncthreads();
  }
  if (threadIdx.x == 0) *out = red[0];
}

// Orbitals of molecule order[blockIdx.x]: F' = X^T W X (W the last extrapolated F), its eigenpairs by Jacobi
// (zq_jacobi.h) on V started as X, so the rotated V is C = X V' at once; e ascending into w + woff, C into
// cout + coff, columns in the same order, info 1 where the sweeps did not end.
template <int W>
__device__ void orbitals(double *lds, const double *X, const double *Fp, int n, int mp, double *__restrict__ e,
                         double *__restrict__ C, int *__restrict__ info) {
  zqj::Jacobi<W> J(
      lds, n, [&](int i, int j) { return 0.5 * (Fp[size_t(i) * mp + j] + Fp[size_t(j) * mp + i]); },
      [&](int r, int k) { return X[size_t(r) * mp + k]; });
  bool ok;
  const bool odd = J.run(&ok) & 1;
  int *rank = reinterpret_cast<int *>(J.A);  // by position, -1: padding
  __syncthreads();                           // A is read no more
  for (int x = threadIdx.x; x < 2 * J.h; x += zqj::kThreads) {
    const int k = odd ? 2 * J.h - 1 - x : x;  // the index that ended at position x
    int r = -1;
    if (k < n) {
      r = 0;
      const double d = J.diag[x];
      for (int y = 0; y < 2 * J.h; ++y) {
        const int l = odd ? 2 * J.h - 1 - y : y;
        if (l < n) r += J.diag[y] < d || (J.diag[y] == d && l < k);
      }
      if (!ok) r = k;  // NaN has no rank
      e[r] = d;
    }
    rank[x] = r;
  }
  __syncthreads();
#pragma unroll
  for (int k = 0; k < J.kRows; ++k) {
    const int r = J.g + J.kGroups * k;
    if (r < n && J.i < J.h)
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const int c = rank[2 * J.i + b];
        if (c >= 0) C[r * n + c] = J.v[k][b];
      }
  }
  if (threadIdx.x == 0) *info = ok ? 0 : 1;
}

__global__ __launch_bounds__(zqj::kThreads) void k_batch_orbitals(double *__restrict__ ws, const BMol *__restrict__ mols,
                                                                  const int *__restrict__ order,
                                                                  const long long *__restrict__ off, double *__restrict__ e,
                                                                  double *__restrict__ C, int *__restrict__ info) {
  extern __shared__ __attribute__((aligned(16))) double step_lds[];
  const int mi = order[blockIdx.x];
  const BMol M = mols[mi];
  const size_t mm = size_t(M.mp) * M.mp;
  double *base = ws + M.ws;
  double *X = base + M_X * mm, *XT = base + M_XT * mm, *W = base + M_W * mm, *T = base + M_T * mm, *Fp = base + M_FPR * mm;
  wg_gemm_nt<zqj::kThreads>(XT, W, T, M.mp, 1.0);
  wg_gemm_nt<zqj::kThreads>(T, XT, Fp, M.mp, 1.0);
  const long long *o = off + 2 * mi;
  switch (zqj::lanes_of(M.n)) {
    case 16: orbitals<16>(step_lds, X, Fp, M.n, M.mp, e + o[1], C + o[0], info + mi); break;
    case 32: orbitals<32>(step_lds, X, Fp, M.n, M.mp, e + o[1], C + o[0], info + mi); break;
    default: orbitals<64>(step_lds, X, Fp, M.n, M.mp, e + o[1], C + o[0], info + mi); break;
  }
}

struct HostMol {
  int n, nocc;
  double VN;
  std::vector<double> H, S, eri;
};

}  // namespace

struct zq_batch {
  int device = 0;
  hipStream_t stream = nullptr;
  std::string err;
  std::vector<HostMol> mols;
  bool uploaded = false;
  int chunk = 0, nt = 256;
  // device residency
  double *eri = nullptr, *ws = nullptr, *rec = nullptr;
  BMol *d_mols = nullptr;
  int *d_order = nullptr;  // molecules by descending padded size: the step kernel's workgroup order
  ScfState *d_state = nullptr;
  double *d_est = nullptr;  // fold bookkeeping, kEstSize per molecule
  BResult *d_res = nullptr;
  int *d_done = nullptr, *d_count = nullptr, *d_ptr = nullptr, *d_idx = nullptr;
  JKItem *d_items = nullptr;
  JKMol *d_jkm = nullptr;
  int2 *d_blk = nullptr;
  int nitems = 0, nblk = 0;
  bool jk_long = false;  // the J/K plan is run in the records kernel's long form
  std::vector<long long> eri_off, ws_off;
  size_t eri_count = 0;  // doubles in eri
  int mp_max = 16;       // largest padded size of the batch (the step's LDS)
  int n_max = 1;         // largest n (the orbitals' LDS)
  int *h_count = nullptr;
  hipGraphExec_t graph = nullptr;
  std::string graph_key;
  // the grouped MP2's FP32 copy of the quartets (FP32 forms; made once per upload) and workspace
  float *eri32 = nullptr;
  void *mp2_ws = nullptr;
  size_t mp2_ws_bytes = 0;
  // the eigenpair stage's device buffers (grow-only, kept across runs) and pinned host copies of C, e and
  // the info codes, which a second stream brings back while the MP2 runs
  double *d_c = nullptr, *d_w = nullptr;
  long long *d_eoff = nullptr;
  int *d_info = nullptr;
  size_t c_cap = 0, w_cap = 0, m_cap = 0;  // doubles of d_c, of d_w; molecules
  double *h_c = nullptr, *h_w = nullptr;
  int *h_info = nullptr;
  size_t hc_cap = 0, hw_cap = 0, hi_cap = 0;
  hipStream_t copy_stream = nullptr;
  hipEvent_t coef_done = nullptr;
  // results of the last run (C and e of molecule m at c_off[m], w_off[m] of h_c, h_w), and its stage
  // times (host wall clock, ms): SCF, eigenpairs, MP2, total
  std::vector<long long> c_off, w_off;
  std::vector<int> res_n;
  double stage_ms[4] = {0, 0, 0, 0};
};

namespace {

int bfail(zq_batch *b, int code, const std::string &msg) {
  if (b) b->err = msg;
  return code;
}

#define BTRY(b, call)                                                                     \
  do {                                                                                    \
    hipError_t _e = (call);                                                               \
    if (_e != hipSuccess) return bfail(b, ZQ_ERR_LAUNCH, std::string(#call) + ": " + hipGetErrorString(_e)); \
  } while (0)

void free_plan(zq_batch *b) {
  for (void *p : {(void *)b->rec, (void *)b->d_items, (void *)b->d_ptr, (void *)b->d_idx, (void *)b->d_blk})
    if (p) (void)hipFree(p);
  b->rec = nullptr, b->d_items = nullptr, b->d_ptr = nullptr, b->d_idx = nullptr, b->d_blk = nullptr;
  if (b->graph) (void)hipGraphExecDestroy(b->graph);
  b->graph = nullptr;
}

void free_eig(zq_batch *b) {
  if (b->copy_stream) (void)hipStreamSynchronize(b->copy_stream);  // copies into the pinned buffers
  for (void *p : {(void *)b->d_c, (void *)b->d_w, (void *)b->d_eoff, (void *)b->d_info})
    if (p) (void)hipFree(p);
  b->d_c = b->d_w = nullptr;
  b->d_eoff = nullptr, b->d_info = nullptr;
  b->c_cap = b->w_cap = b->m_cap = 0;
  for (void *p : {(void *)b->h_c, (void *)b->h_w, (void *)b->h_info})
    if (p) (void)hipHostFree(p);
  b->h_c = b->h_w = nullptr, b->h_info = nullptr;
  b->hc_cap = b->hw_cap = b->hi_cap = 0;
}

// Grow-only device and pinned host buffers of the eigenpair stage.
int eig_buffers(zq_batch *b, size_t ctot, size_t wtot, size_t M) {
  if (ctot > b->c_cap) {
    if (b->d_c) (void)hipFree(b->d_c);
    if (b->h_c) (void)hipHostFree(b->h_c);
    b->d_c = b->h_c = nullptr, b->c_cap = b->hc_cap = 0;
    BTRY(b, hipMalloc(&b->d_c, ctot * sizeof(double)));
    BTRY(b, hipHostMalloc((void **)&b->h_c, ctot * sizeof(double), hipHostMallocDefault));
    b->c_cap = b->hc_cap = ctot;
  }
  if (wtot > b->w_cap) {
    if (b->d_w) (void)hipFree(b->d_w);
    if (b->h_w) (void)hipHostFree(b->h_w);
    b->d_w = b->h_w = nullptr, b->w_cap = b->hw_cap = 0;
    BTRY(b, hipMalloc(&b->d_w, wtot * sizeof(double)));
    BTRY(b, hipHostMalloc((void **)&b->h_w, wtot * sizeof(double), hipHostMallocDefault));
    b->w_cap = b->hw_cap = wtot;
  }
  if (M > b->m_cap) {
    if (b->d_eoff) (void)hipFree(b->d_eoff);
    if (b->d_info) (void)hipFree(b->d_info);
    if (b->h_info) (void)hipHostFree(b->h_info);
    b->d_eoff = nullptr, b->d_info = nullptr, b->h_info = nullptr, b->m_cap = b->hi_cap = 0;
    BTRY(b, hipMalloc(&b->d_eoff, 2 * M * sizeof(long long)));
    BTRY(b, hipMalloc(&b->d_info, M * sizeof(int)));
    BTRY(b, hipHostMalloc((void **)&b->h_info, M * sizeof(int), hipHostMallocDefault));
    b->m_cap = b->hi_cap = M;
  }
  if (!b->copy_stream) BTRY(b, hipStreamCreateWithFlags(&b->copy_stream, hipStreamNonBlocking));
  if (!b->coef_done) BTRY(b, hipEventCreateWithFlags(&b->coef_done, hipEventDisableTiming));
  return ZQ_OK;
}

void free_all(zq_batch *b) {
  free_plan(b);
  free_eig(b);
  for (void *p : {(void *)b->eri, (void *)b->ws, (void *)b->d_mols, (void *)b->d_order, (void *)b->d_state,
                  (void *)b->d_est, (void *)b->d_res, (void *)b->d_done, (void *)b->d_count, (void *)b->d_jkm,
                  (void *)b->eri32, b->mp2_ws})
    if (p) (void)hipFree(p);
  b->eri = nullptr, b->ws = nullptr, b->d_mols = nullptr, b->d_order = nullptr, b->d_state = nullptr;
  b->d_est = nullptr, b->d_res = nullptr, b->d_done = nullptr;
  b->d_count = nullptr, b->d_jkm = nullptr, b->eri32 = nullptr, b->mp2_ws = nullptr, b->mp2_ws_bytes = 0;
  b->uploaded = false;
}

int mp_of(int n) { return (n + 15) / 16 * 16; }
int nb_of(int n) { return (n + ZQ_BLK - 1) / ZQ_BLK; }

// The grouped J/K plan for item size `chunk` (0: each molecule's default): items, records and CSR rows of all molecules
// concatenated.  With the defaults, long and short items mix; the long form is taken when all are long.  SCF of 6
// iterations without autotune, ms, short / long form / each item in its own, in two launches: 32 molecules n = 96
// 8.62 / 8.54 / 8.55, 8 n = 80 2.72 / 2.68 / 2.68, 40 n = 24 .. 96 6.36 / 6.77 / 6.34, 60 n <= 24 and one n = 96
// 3.94 / 3.91 / 3.98 (items of one quartet throughout: 9.61, 2.78, 6.59, 4.00).
int build_plan(zq_batch *b, int chunk) {
  free_plan(b);
  std::vector<JKItem> items;
  std::vector<int> ptr(1, 0), idx;
  std::vector<int2> blk;
  size_t rec_base = 0;
  b->jk_long = true;
  for (size_t m = 0; m < b->mols.size(); ++m) {
    const int nb = nb_of(b->mols[m].n), Nb = nb * (nb + 1) / 2;
    const size_t nq = size_t(Nb) * (Nb + 1) / 2;
    JKPlan pl;
    zq_jk_plan(Nb, nq, chunk, pl);
    b->jk_long = b->jk_long && zq_jk_long(nq, chunk);
    for (JKItem it : pl.items) {
      it.rec0 += int(rec_base);
      it.mol = int(m);
      items.push_back(it);
    }
    for (int o = 0; o < Nb; ++o) {
      for (int e = pl.ptr[o]; e < pl.ptr[o + 1]; ++e) {
        const int code = pl.idx[e];
        idx.push_back(int((size_t(code >> 1) + rec_base) << 1) | (code & 1));
      }
      ptr.push_back(int(idx.size()));
      blk.push_back(make_int2(int(m), o));
    }
    rec_base += pl.nrecords;
    if (rec_base >= (size_t(1) << 30)) return bfail(b, ZQ_ERR_INVALID, "batch J/K plan: too many records");
  }
  b->nitems = int(items.size());
  b->nblk = int(blk.size());
  BTRY(b, hipMalloc(&b->rec, std::max<size_t>(1, rec_base) * 64 * sizeof(double)));
  BTRY(b, hipMalloc(&b->d_items, items.size() * sizeof(JKItem)));
  BTRY(b, hipMalloc(&b->d_ptr, ptr.size() * sizeof(int)));
  BTRY(b, hipMalloc(&b->d_idx, std::max<size_t>(1, idx.size()) * sizeof(int)));
  BTRY(b, hipMalloc(&b->d_blk, blk.size() * sizeof(int2)));
  // the batch stream is non-blocking: uploads go on it, so its kernels see them
  BTRY(b, hipMemcpyAsync(b->d_items, items.data(), items.size() * sizeof(JKItem), hipMemcpyHostToDevice, b->stream));
  BTRY(b, hipMemcpyAsync(b->d_ptr, ptr.data(), ptr.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
  if (!idx.empty())
    BTRY(b, hipMemcpyAsync(b->d_idx, idx.data(), idx.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
  BTRY(b, hipMemcpyAsync(b->d_blk, blk.data(), blk.size() * sizeof(int2), hipMemcpyHostToDevice, b->stream));
  BTRY(b, hipStreamSynchronize(b->stream));  // the plan's host vectors go out of scope
  b->chunk = chunk;
  return ZQ_OK;
}

// ERIs into quartets, H/S/X/X^T into the workspace, the per-molecule tables, the plan.
int upload(zq_batch *b) {
  if (b->uploaded) return ZQ_OK;
  if (b->mols.empty()) return bfail(b, ZQ_ERR_STATE, "empty batch");
  BTRY(b, hipSetDevice(b->device));
  const size_t M = b->mols.size();
  b->eri_off.assign(M, 0);
  b->ws_off.assign(M, 0);
  size_t eri_total = 0, ws_total = 0, canon_max = 0;
  std::vector<BMol> bm(M);
  std::vector<JKMol> jm(M);
  for (size_t m = 0; m < M; ++m) {
    const HostMol &h = b->mols[m];
    const int nb = nb_of(h.n), Nb = nb * (nb + 1) / 2, mp = mp_of(h.n);
    const size_t nq = size_t(Nb) * (Nb + 1) / 2, mm = size_t(mp) * mp;
    b->eri_off[m] = (long long)eri_total;
    b->ws_off[m] = (long long)ws_total;
    eri_total += nq * ZQ_QUARTET;
    ws_total += kWsMats * mm;
    canon_max = std::max(canon_max, h.eri.size());
    bm[m] = BMol{(long long)b->ws_off[m], h.n, mp, h.nocc, 0, h.VN};
    b->mp_max = std::max(b->mp_max, mp);
    b->n_max = std::max(b->n_max, h.n);
    jm[m] = JKMol{b->eri_off[m], b->ws_off[m] + M_P * (long long)mm, b->ws_off[m] + M_H * (long long)mm,
                  b->ws_off[m] + M_F * (long long)mm, mp, h.n};
  }
  BTRY(b, hipMalloc(&b->eri, eri_total * sizeof(double)));
  b->eri_count = eri_total;
  BTRY(b, hipMalloc(&b->ws, ws_total * sizeof(double)));
  BTRY(b, hipMalloc(&b->d_mols, M * sizeof(BMol)));
  BTRY(b, hipMalloc(&b->d_order, M * sizeof(int)));
  BTRY(b, hipMalloc(&b->d_state, M * sizeof(ScfState)));
  BTRY(b, hipMalloc(&b->d_est, M * kEstSize * sizeof(double)));
  BTRY(b, hipMalloc(&b->d_res, M * sizeof(BResult)));
  BTRY(b, hipMalloc(&b->d_done, M * sizeof(int)));
  BTRY(b, hipMalloc(&b->d_count, sizeof(int)));
  BTRY(b, hipMalloc(&b->d_jkm, M * sizeof(JKMol)));
  BTRY(b, hipMemsetAsync(b->ws, 0, ws_total * sizeof(double), b->stream));
  BTRY(b, hipMemsetAsync(b->d_done, 0, M * sizeof(int), b->stream));
  BTRY(b, hipMemcpyAsync(b->d_mols, bm.data(), M * sizeof(BMol), hipMemcpyHostToDevice, b->stream));
  BTRY(b, hipMemcpyAsync(b->d_jkm, jm.data(), M * sizeof(JKMol), hipMemcpyHostToDevice, b->stream));
  // largest first: a step of a large molecule takes a compute unit for longest, so the small ones fill
  // in behind it rather than leaving a large one for the end (one workgroup per compute unit at 512
  // threads)
  std::vector<int> order(M);
  for (size_t m = 0; m < M; ++m) order[m] = int(m);
  std::stable_sort(order.begin(), order.end(), [&](int x, int y) { return bm[x].mp > bm[y].mp; });
  BTRY(b, hipMemcpyAsync(b->d_order, order.data(), M * sizeof(int), hipMemcpyHostToDevice, b->stream));
  BTRY(b, hipStreamSynchronize(b->stream));
  double *canon = nullptr;
  BTRY(b, hipMalloc(&canon, canon_max * sizeof(double)));
  for (size_t m = 0; m < M; ++m) {
    const HostMol &h = b->mols[m];
    const int nb = nb_of(h.n), Nb = nb * (nb + 1) / 2, mp = mp_of(h.n);
    const size_t nq = size_t(Nb) * (Nb + 1) / 2, mm = size_t(mp) * mp;
    hipError_t e = hipMemcpyAsync(canon, h.eri.data(), h.eri.size() * sizeof(double), hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) {
      hipLaunchKernelGGL(zq_pack_quartets, dim3(unsigned(nq)), dim3(256), 0, b->stream, canon, b->eri + b->eri_off[m], h.n,
                         nq);
      e = hipStreamSynchronize(b->stream);
    }
    // H, S, X = L^-T, X^T, zero padded to mp
    std::vector<double> stage(4 * mm, 0.0), hX(size_t(h.n) * h.n);
    if (e == hipSuccess && zq::chol_inv_t(h.n, h.S.data(), hX.data())) {
      (void)hipFree(canon);
      return bfail(b, ZQ_ERR_LAPACK, "batch molecule " + std::to_string(m) + ": overlap not positive definite");
    }
    for (int i = 0; i < h.n; ++i)
      for (int j = 0; j < h.n; ++j) {
        stage[0 * mm + size_t(i) * mp + j] = h.H[size_t(i) * h.n + j];
        stage[1 * mm + size_t(i) * mp + j] = h.S[size_t(i) * h.n + j];
        stage[2 * mm + size_t(i) * mp + j] = hX[size_t(i) * h.n + j];
        stage[3 * mm + size_t(j) * mp + i] = hX[size_t(i) * h.n + j];
      }
    double *w = b->ws + b->ws_off[m];
    if (e == hipSuccess) e = hipMemcpyAsync(w + M_H * mm, stage.data(), mm * 8, hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(w + M_S * mm, stage.data() + mm, mm * 8, hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(w + M_X * mm, stage.data() + 2 * mm, mm * 8, hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(w + M_XT * mm, stage.data() + 3 * mm, mm * 8, hipMemcpyHostToDevice, b->stream);
    if (e == hipSuccess) e = hipStreamSynchronize(b->stream);  // stage goes out of scope
    if (e != hipSuccess) {
      (void)hipFree(canon);
      return bfail(b, ZQ_ERR_LAUNCH, std::string("batch upload: ") + hipGetErrorString(e));
    }
  }
  (void)hipFree(canon);
  if (int rc = build_plan(b, b->chunk)) return rc;
  if (!b->h_count) BTRY(b, hipHostMalloc((void **)&b->h_count, 2 * sizeof(int), hipHostMallocDefault));
  b->uploaded = true;
  return ZQ_OK;
}

void launch_step(zq_batch *b, int mode, int diis, double thr, int maxit) {
  const dim3 grid(unsigned(b->mols.size()));
  const size_t lds = step_lds_bytes(b->mp_max);
  if (b->nt == 512)
    hipLaunchKernelGGL(k_batch_step<512>, grid, dim3(512), lds, b->stream, b->ws, b->d_mols, b->d_order, b->d_state,
                       b->d_est, b->d_done, mode, diis, thr, maxit);
  else
    hipLaunchKernelGGL(k_batch_step<256>, grid, dim3(256), lds, b->stream, b->ws, b->d_mols, b->d_order, b->d_state,
                       b->d_est, b->d_done, mode, diis, thr, maxit);
}

int enqueue_iteration(zq_batch *b, int diis, double thr, int maxit) {
  BTRY(b, zq_jk_group(b->stream, b->eri, b->d_items, b->nitems, b->ws, 0.5, b->rec, b->d_jkm, b->d_done, b->d_ptr,
                      b->d_idx, b->d_blk, b->nblk, b->ws, b->ws, b->mp_max, b->jk_long));
  launch_step(b, kStepIter, diis, thr, maxit);
  hipLaunchKernelGGL(k_batch_count, dim3(1), dim3(256), 0, b->stream, b->d_done, int(b->mols.size()), b->d_count);
  BTRY(b, hipGetLastError());
  return ZQ_OK;
}

// A view context on molecule m's resident quartets, for the transform code of zq_transform.hip.
void bind_view(zq_ctx *v, zq_batch *b, int m) {
  const int n = b->mols[m].n;
  if (v->eri32 && v->eri32_owned) (void)hipFree(v->eri32);  // an FP32 copy of the previous molecule
  v->eri32 = nullptr;
  v->eri32_owned = true;
  v->eri_owned = false;
  v->n = n;
  v->nb = nb_of(n);
  v->npad = v->nb * ZQ_BLK;
  v->Nb = v->nb * (v->nb + 1) / 2;
  v->nquartets = size_t(v->Nb) * (v->Nb + 1) / 2;
  v->eri = b->eri + b->eri_off[m];
}

}  // namespace

extern "C" {

zq_batch *zq_batch_create(int device) {
  ZqGate _gate;
  int count = 0;
  if (hipGetDeviceCount(&count) != hipSuccess || device < 0 || device >= count) return nullptr;
  if (hipSetDevice(device) != hipSuccess) return nullptr;
  auto *b = new zq_batch;
  b->device = device;
  if (hipStreamCreateWithFlags(&b->stream, hipStreamNonBlocking) != hipSuccess) {
    delete b;
    return nullptr;
  }
  return b;
}

void zq_batch_destroy(zq_batch *b) {
  ZqGate _gate;
  if (!b) return;
  (void)hipSetDevice(b->device);
  (void)hipStreamSynchronize(b->stream);
  if (b->copy_stream) (void)hipStreamSynchronize(b->copy_stream);
  free_all(b);
  if (b->h_count) (void)hipHostFree(b->h_count);
  if (b->coef_done) (void)hipEventDestroy(b->coef_done);
  if (b->copy_stream) (void)hipStreamDestroy(b->copy_stream);
  (void)hipStreamDestroy(b->stream);
  delete b;
}

const char *zq_batch_last_error(const zq_batch *b) { return b ? b->err.c_str() : "null batch"; }

int zq_batch_count(const zq_batch *b) { return b ? int(b->mols.size()) : 0; }

int zq_batch_add(zq_batch *b, size_t n, size_t nocc, const double *H, const double *S, double VN,
                 const double *eri_packed) {
  if (!b || !H || !S || !eri_packed) return bfail(b, ZQ_ERR_INVALID, "zq_batch_add: null argument");
  if (n == 0 || n > size_t(kMaxN) || nocc == 0 || nocc >= n)
    return bfail(b, ZQ_ERR_INVALID, "zq_batch_add: need 0 < nocc < n <= 96");
  HostMol h;
  h.n = int(n), h.nocc = int(nocc), h.VN = VN;
  h.H.assign(H, H + n * n);
  h.S.assign(S, S + n * n);
  const size_t np = n * (n + 1) / 2, nu = np * (np + 1) / 2;
  h.eri.assign(eri_packed, eri_packed + nu);
  if (b->uploaded) {
    ZqGate _gate;
    free_all(b);  // residency is rebuilt on the next run
  }
  b->mols.push_back(std::move(h));
  return int(b->mols.size()) - 1;
}

int zq_batch_autotune(zq_batch *b, int chosen[2]) {
  ZqGate _gate;
  if (!b) return ZQ_ERR_INVALID;
  BTRY(b, hipSetDevice(b->device));
  if (int rc = upload(b)) return rc;
  hipEvent_t e0, e1;
  BTRY(b, hipEventCreate(&e0));
  BTRY(b, hipEventCreate(&e1));
  auto time_it = [&](auto &&fn) -> float {
    float best = 1e30f;
    for (int rep = 0; rep < 3; ++rep) {
      (void)hipEventRecord(e0, b->stream);
      fn();
      (void)hipEventRecord(e1, b->stream);
      (void)hipEventSynchronize(e1);
      float ms = 0;
      (void)hipEventElapsedTime(&ms, e0, e1);
      best = std::min(best, ms);
    }
    return best;
  };
  int best_chunk = 1;
  float best = 1e30f;
  BTRY(b, hipMemsetAsync(b->d_done, 0, b->mols.size() * sizeof(int), b->stream));
  for (int ch : {1, 2, 4, 8, 16}) {
    if (int rc = build_plan(b, ch)) return rc;
    const float ms = time_it([&] {
      (void)zq_jk_group(b->stream, b->eri, b->d_items, b->nitems, b->ws, 0.5, b->rec, b->d_jkm, b->d_done, b->d_ptr,
                        b->d_idx, b->d_blk, b->nblk, b->ws, b->ws, b->mp_max, b->jk_long);
    });
    if (ms < best) best = ms, best_chunk = ch;
  }
  int best_nt = 256;
  best = 1e30f;
  for (int nt : {256, 512}) {
    b->nt = nt;
    const float ms = time_it([&] { launch_step(b, kStepGuess, 8, 1e-8, 100); });
    if (ms < best) best = ms, best_nt = nt;
  }
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  b->nt = best_nt;
  if (int rc = build_plan(b, best_chunk)) return rc;
  BTRY(b, hipStreamSynchronize(b->stream));
  if (chosen) chosen[0] = best_chunk, chosen[1] = best_nt;
  return ZQ_OK;
}

int zq_batch_run(zq_batch *b, const zq_scf_options *opt, int mp2_precision, double *E_rhf, double *E_corr,
                 int *iterations, int *status) {
  ZqGate _gate;
  if (!b || !opt || !E_rhf || !E_corr || !iterations || !status) return bfail(b, ZQ_ERR_INVALID, "zq_batch_run: null argument");
  if (opt->generalized || opt->fock_precision != ZQ_PREC_FP64 || opt->diis < 0 || opt->diis > kHist || opt->iterations < 1)
    return bfail(b, ZQ_ERR_INVALID, "zq_batch_run: RHF, FP64 Fock builds, diis <= 8, iterations >= 1");
  BTRY(b, hipSetDevice(b->device));
  if (int rc = upload(b)) return rc;
  const int M = int(b->mols.size());
  const auto t0 = std::chrono::steady_clock::now();
  auto since = [](std::chrono::steady_clock::time_point t) {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t).count();
  };

  // core-Hamiltonian guess, then the captured iteration until every molecule is done
  launch_step(b, kStepGuess, opt->diis, opt->threshold, opt->iterations);
  char key[128];
  snprintf(key, sizeof key, "%d/%d/%d/%a/%d/%p", b->nt, b->chunk, opt->diis, opt->threshold, opt->iterations,
           (void *)b->d_items);
  if (!b->graph || b->graph_key != key) {
    if (b->graph) (void)hipGraphExecDestroy(b->graph);
    b->graph = nullptr;
    ZqCaptureWindow window;
    BTRY(b, hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue_iteration(b, opt->diis, opt->threshold, opt->iterations);
    hipGraph_t g = nullptr;
    const hipError_t e = hipStreamEndCapture(b->stream, &g);
    if (rc) {
      if (g) (void)hipGraphDestroy(g);
      return rc;
    }
    if (e != hipSuccess) return bfail(b, ZQ_ERR_LAUNCH, std::string("hipStreamEndCapture: ") + hipGetErrorString(e));
    const hipError_t e2 = hipGraphInstantiate(&b->graph, g, nullptr, nullptr, 0);
    (void)hipGraphDestroy(g);
    if (e2 != hipSuccess) return bfail(b, ZQ_ERR_LAUNCH, std::string("hipGraphInstantiate: ") + hipGetErrorString(e2));
    b->graph_key = key;
  }
  hipEvent_t ev[2];
  BTRY(b, hipEventCreateWithFlags(&ev[0], hipEventDisableTiming));
  BTRY(b, hipEventCreateWithFlags(&ev[1], hipEventDisableTiming));
  for (int k = 0; k < opt->iterations; ++k) {
    BTRY(b, hipGraphLaunch(b->graph, b->stream));
    BTRY(b, hipMemcpyAsync(b->h_count + (k & 1), b->d_count, sizeof(int), hipMemcpyDeviceToHost, b->stream));
    BTRY(b, hipEventRecord(ev[k & 1], b->stream));
    if (k >= 1) {
      BTRY(b, hipEventSynchronize(ev[(k - 1) & 1]));
      if (b->h_count[(k - 1) & 1] >= M) break;
    }
  }
  BTRY(b, hipStreamSynchronize(b->stream));
  (void)hipEventDestroy(ev[0]);
  (void)hipEventDestroy(ev[1]);
  std::vector<BResult> hs(M);
  hipLaunchKernelGGL(k_batch_result, dim3(unsigned((M + 255) / 256)), dim3(256), 0, b->stream, b->d_state, M, b->d_res);
  BTRY(b, hipMemcpyAsync(hs.data(), b->d_res, M * sizeof(BResult), hipMemcpyDeviceToHost, b->stream));
  BTRY(b, hipStreamSynchronize(b->stream));
  b->stage_ms[0] = since(t0);
  const auto t1 = std::chrono::steady_clock::now();

  // orbitals of the last extrapolated F, one workgroup per molecule
  std::vector<long long> off(2 * size_t(M)), coff(M), woff(M);
  long long ctot = 0, wtot = 0;
  for (int m = 0; m < M; ++m) {
    off[2 * m] = coff[m] = ctot, off[2 * m + 1] = woff[m] = wtot;
    ctot += (long long)b->mols[m].n * b->mols[m].n;
    wtot += b->mols[m].n;
  }
  // the previous run's copies of C and e must have landed before their buffers are reused
  if (b->copy_stream) BTRY(b, hipStreamSynchronize(b->copy_stream));
  if (int rc = eig_buffers(b, size_t(ctot), size_t(wtot), size_t(M))) return rc;
  double *d_w = b->d_w, *d_c = b->d_c;
  int *d_info = b->d_info;
  BTRY(b, hipMemcpyAsync(b->d_eoff, off.data(), off.size() * sizeof(long long), hipMemcpyHostToDevice, b->stream));
  hipLaunchKernelGGL(k_batch_orbitals, dim3(M), dim3(zqj::kThreads), zqj::lds_doubles(b->n_max) * sizeof(double), b->stream,
                     b->ws, b->d_mols, b->d_order, b->d_eoff, d_w, d_c, d_info);
  BTRY(b, hipGetLastError());
  // C, e and the info codes go to pinned host memory on the copy stream, overlapped with the MP2
  BTRY(b, hipEventRecord(b->coef_done, b->stream));
  BTRY(b, hipStreamWaitEvent(b->copy_stream, b->coef_done, 0));
  BTRY(b, hipMemcpyAsync(b->h_c, d_c, ctot * sizeof(double), hipMemcpyDeviceToHost, b->copy_stream));
  BTRY(b, hipMemcpyAsync(b->h_w, d_w, wtot * sizeof(double), hipMemcpyDeviceToHost, b->copy_stream));
  BTRY(b, hipMemcpyAsync(b->h_info, d_info, M * sizeof(int), hipMemcpyDeviceToHost, b->copy_stream));
  b->c_off = coff, b->w_off = woff;
  b->res_n.resize(M);
  for (int m = 0; m < M; ++m) b->res_n[m] = b->mols[m].n;
  BTRY(b, hipStreamSynchronize(b->stream));
  b->stage_ms[1] = since(t1);
  const auto t2 = std::chrono::steady_clock::now();

  // MP2 of every molecule that finished its iterations
  std::vector<int> rc_m(M, ZQ_OK);
  for (int m = 0; m < M; ++m) E_corr[m] = 0.0;
  if (mp2_precision != ZQ_PREC_BF16X3) {
    // grouped: one launch per transform stage for all molecules, on the device C and e
    const bool f32 = mp2_precision == ZQ_PREC_FP32 || mp2_precision == ZQ_PREC_FP32C;
    if (f32 && !b->eri32) {
      BTRY(b, hipMalloc(&b->eri32, b->eri_count * sizeof(float)));
      zq_narrow_eri(b->stream, b->eri, b->eri_count, b->eri32);
      BTRY(b, hipGetLastError());
    }
    std::vector<ZqGroupMol> gm;
    std::vector<int> which;
    for (int m = 0; m < M; ++m) {
      if (hs[m].done != 1 && hs[m].done != 2) continue;
      gm.push_back(ZqGroupMol{b->eri + b->eri_off[m], f32 ? b->eri32 + b->eri_off[m] : nullptr, b->mols[m].n,
                              b->mols[m].nocc, d_c + coff[m], d_w + woff[m]});
      which.push_back(m);
    }
    std::vector<double> ec(gm.size(), 0.0);
    std::string err;
    if (int rc = zq_mp2_grouped(b->stream, gm, mp2_precision, &b->mp2_ws, &b->mp2_ws_bytes, ec.data(), err))
      return bfail(b, rc, err);
    for (size_t k = 0; k < which.size(); ++k) E_corr[which[k]] = ec[k];
  } else {
    // BF16X3: several view contexts at once, each with its own stream, on the host copies of C and e
    BTRY(b, hipStreamSynchronize(b->copy_stream));
    const int nworkers = std::min(M, 8);
    std::vector<zq_ctx *> views(nworkers, nullptr);
    for (int w = 0; w < nworkers; ++w) {
      views[w] = zq_create(b->device);
      if (!views[w]) {
        for (zq_ctx *v : views)
          if (v) zq_destroy(v);
        return bfail(b, ZQ_ERR_LAUNCH, "batch MP2: context creation");
      }
    }
    std::atomic<int> next{0};
    std::vector<std::thread> th;
    for (int w = 0; w < nworkers; ++w)
      th.emplace_back([&, w] {
        ZqGate gate;
        (void)hipSetDevice(b->device);
        for (int m; (m = next.fetch_add(1)) < M;) {
          if (hs[m].done != 1 && hs[m].done != 2) continue;
          bind_view(views[w], b, m);
          rc_m[m] = zq_mp2_device(views[w], b->h_c + coff[m], b->h_w + woff[m], b->mols[m].nocc, mp2_precision,
                                  &E_corr[m]);
          views[w]->eri = nullptr;
        }
      });
    for (auto &t : th) t.join();
    for (zq_ctx *v : views) {
      v->eri = nullptr;
      zq_destroy(v);
    }
  }
  b->stage_ms[2] = since(t2);
  BTRY(b, hipStreamSynchronize(b->copy_stream));  // C, e and the info codes are on the host
  b->stage_ms[3] = since(t0);
  for (int m = 0; m < M; ++m) {
    E_rhf[m] = hs[m].energy;
    iterations[m] = hs[m].it;
    status[m] = hs[m].done == 1 ? ZQ_OK : hs[m].done == 2 ? ZQ_ERR_NOT_CONVERGED : ZQ_ERR_LAPACK;
    if (b->h_info[m] && status[m] == ZQ_OK) status[m] = ZQ_ERR_LAPACK;
    if (rc_m[m] != ZQ_OK && status[m] == ZQ_OK) status[m] = rc_m[m];
  }
  return ZQ_OK;
}

int zq_batch_timings(const zq_batch *b, double ms[4]) {
  if (!b || !ms) return ZQ_ERR_INVALID;
  std::copy(b->stage_ms, b->stage_ms + 4, ms);
  return ZQ_OK;
}

int zq_batch_orbitals(const zq_batch *b, int index, double *e, double *C) {
  if (!b || index < 0 || size_t(index) >= b->res_n.size() || !e || !C || !b->h_c || !b->h_w) return ZQ_ERR_INVALID;
  const long long n = b->res_n[index];
  std::copy(b->h_w + b->w_off[index], b->h_w + b->w_off[index] + n, e);
  std::copy(b->h_c + b->c_off[index], b->h_c + b->c_off[index] + n * n, C);
  return ZQ_OK;
}

}  // extern "C"
