// Ensemble: many independent runs (own grid, Ma, Kn, CFL, tmax; each its own CFL dt)
// advanced together by one HIP-graph-captured step.
//
// Layout: the runs' states are contiguous parts of shared SoA planes ([35][Ntot]; run r
// owns cells [off_r, off_r + N_r), each in its own Julia order).  Kernels run over blocks
// of one run each: a block table maps blockIdx -> (run, first cell), so a block reads its
// run's parameters and step scalars once and a finished run costs one load per block.
// One step (begin, pass 1, dt, update, pass 2: the single run's kernels, hyq_step_kernels.h, over
// the block table) is captured once into a graph and replayed; the per-run dt reduction is an
// atomic max into the run's scalars.
//
// The block size of each of the three cell kernels is a tunable: hyq_ensemble_tune times
// every candidate on the ensemble's own state (saved and restored around the trial steps)
// and keeps the fastest per kernel.
#include <hip/hip_runtime.h>

#include <cstring>
#include <mutex>
#include <string>
#include <vector>

#include "../../include/hyqmom.h"
#include "hyq_ensemble_kernels.h"
#include "hyq_hostcopy.h"

using namespace hyq;
using namespace hyq_ens;

namespace {

thread_local std::string g_eerr;
int efail(int code, const char* what, hipError_t e = hipSuccess) {
  g_eerr = what;
  if (e != hipSuccess) {
    g_eerr += ": ";
    g_eerr += hipGetErrorString(e);
  }
  return code;
}
#define ECHK(x, msg)                                       \
  do {                                                     \
    hipError_t _e = (x);                                   \
    if (_e != hipSuccess) return efail(HYQ_EHIP, msg, _e); \
  } while (0)

constexpr int kCand[3] = {64, 128, 256};  // block-size candidates

__global__ void ke_begin(RunDev* R, int nr, StepCounts* cnt) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r == 0) clear_counts(cnt);
  if (r >= nr) return;
  RunDev& q = R[r];
  // a run whose z wave-speed solve met a non-finite Jacobian stops there (the reference throws)
  const bool act = q.t < q.tmax && q.nn < q.nnmax && q.err == 0ull;
  q.active = act ? 1.0 : 0.0;
  if (act) q.nn += 1;
  q.vmax_bits = 0ull;
}

__global__ void ke_dt(RunDev* R, int nr) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nr) return;
  RunDev& q = R[r];
  if (q.active == 0.0) return;
  const double vmax = __longlong_as_double((long long)q.vmax_bits);
  const double hmin = jmin(jmin(q.dx, q.dy), q.dz);
  double dt = jmin(q.CFL * hmin / vmax, jmin(q.dtmax, q.Kn));
  dt = jmin(dt, q.tmax - q.t);
  q.dt = dt;
  q.t += dt;
}

// A run's state between its cells of the ensemble's planes and a contiguous [35][N] array, so
// that the host copies it in one piece rather than 35.  TO: into the planes; the run's
// scalars then start over.
template <bool TO>
__global__ __launch_bounds__(256) void ke_strips(double* M, double* S, RunDev* q, long long off, long long N,
                                                 long long P) {
  const long long c = (long long)blockIdx.x * 256 + threadIdx.x;
  const int n = blockIdx.y;
  if (TO && c == 0 && n == 0) {
    q->t = 0.0;
    q->nn = 0;
    q->active = 0.0;
    q->err = 0ull;
  }
  if (c >= N) return;
  if (TO) M[(size_t)n * P + off + c] = S[(size_t)n * N + c];
  else S[(size_t)n * N + c] = M[(size_t)n * P + off + c];
}

int cand_index(int b) {
  for (int i = 0; i < 3; ++i)
    if (kCand[i] == b) return i;
  return -1;
}

}  // namespace

struct hyq_ensemble {
  int nr = 0, prec = 0;
  long long P = 0;  // total cells = plane stride
  std::vector<RunDev> runs;
  RunDev* R = nullptr;
  double *M = nullptr, *Mr = nullptr, *Mbak = nullptr;
  void *F = nullptr, *vp = nullptr;
  uint32_t* flags = nullptr;
  StepCounts* cnt = nullptr;
  Blk* T[3] = {nullptr, nullptr, nullptr};
  int nblk[3] = {0, 0, 0};
  int blocks[3] = {128, 128, 128};  // pass 1, update, pass 2
  hipStream_t stream = nullptr;
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  hipEvent_t ev[4] = {nullptr, nullptr, nullptr, nullptr};
  HostCopy* copy = nullptr;  // the states' copies from and to the host
  bool ended = false;        // every run was past its end at the last step, and none was set since
  // Held by every call that writes Mr: a state travels through it between the host's copy and
  // the gather or scatter of its cells, and each step's pass 1 writes it.
  std::mutex mu;
};

namespace {

void launch_kernel(hyq_ensemble* e, int which, int b, hipStream_t s) {
  const int ci = cand_index(b);
  const EnsPtrs p{e->M, e->Mr, e->F, e->vp, e->flags, e->R, e->P, carve_lists(e->F, e->P), e->cnt,
                  e->T[0], (unsigned)e->nblk[0]};
  static_assert(kCand[0] == 64, "k_planes runs on blocks of 64 cells");
  if (e->prec == HYQ_PREC_FP64) launch_fp64(which, b, (unsigned)e->nblk[ci], e->T[ci], p, s);
  else if (e->prec == HYQ_PREC_MIXED) launch_mixed(which, b, (unsigned)e->nblk[ci], e->T[ci], p, s);
  else launch_newton(which, b, (unsigned)e->nblk[ci], e->T[ci], p, s);
}

// One step; with ev != null, events around the three cell kernels (ev[0..3]).
void enqueue(hyq_ensemble* e, hipStream_t s, hipEvent_t* ev) {
  const unsigned gr = (unsigned)((e->nr + 63) / 64);
  hipLaunchKernelGGL(ke_begin, dim3(gr), dim3(64), 0, s, e->R, e->nr, e->cnt);
  if (ev) hipEventRecord(ev[0], s);
  launch_kernel(e, 0, e->blocks[0], s);
  if (ev) hipEventRecord(ev[1], s);
  hipLaunchKernelGGL(ke_dt, dim3(gr), dim3(64), 0, s, e->R, e->nr);
  launch_kernel(e, 1, e->blocks[1], s);
  if (ev) hipEventRecord(ev[2], s);
  launch_kernel(e, 2, e->blocks[2], s);
  if (ev) hipEventRecord(ev[3], s);
}

void drop_graph(hyq_ensemble* e) {
  if (e->exec) (void)hipGraphExecDestroy(e->exec);
  if (e->graph) (void)hipGraphDestroy(e->graph);
  e->exec = nullptr;
  e->graph = nullptr;
}

int build_graph(hyq_ensemble* e) {
  drop_graph(e);
  ECHK(hipStreamBeginCapture(e->stream, hipStreamCaptureModeThreadLocal), "begin capture");
  enqueue(e, e->stream, nullptr);
  ECHK(hipStreamEndCapture(e->stream, &e->graph), "end capture");
  ECHK(hipGraphInstantiate(&e->exec, e->graph, nullptr, nullptr, 0), "graph instantiate");
  return HYQ_OK;
}

}  // namespace

extern "C" {

const char* hyq_ensemble_last_error(void) { return g_eerr.c_str(); }

int hyq_ensemble_create(const hyq_params* runs, int32_t nruns, hyq_ensemble** out) {
  if (!runs || nruns <= 0 || !out) return efail(HYQ_EINVAL, "bad argument");
  const int prec = runs[0].precision;
  if (prec != HYQ_PREC_FP64 && prec != HYQ_PREC_MIXED && prec != HYQ_PREC_MIXED_NEWTON)
    return efail(HYQ_EINVAL, "ensemble precision must be FP64, MIXED or MIXED_NEWTON");
  hyq_ensemble* e = new hyq_ensemble();
  e->nr = nruns;
  e->prec = prec;
  long long off = 0;
  for (int r = 0; r < nruns; ++r) {
    const hyq_params& p = runs[r];
    if (p.Nmom != 35 || p.Nx < 1 || p.Ny < 1 || p.Nz < 1 || p.precision != prec) {
      delete e;
      return efail(HYQ_EINVAL, "run parameters (Nmom 35, sizes >= 1, one precision for all)");
    }
    RunDev q;
    std::memset(&q, 0, sizeof(q));
    q.off = off;
    q.N = (long long)p.Nx * p.Ny * p.Nz;
    q.Nx = p.Nx; q.Ny = p.Ny; q.Nz = p.Nz;
    q.flag2D = p.flag2D; q.positivity = p.positivity;
    q.Ma = p.Ma; q.Kn = p.Kn; q.CFL = p.CFL; q.dtmax = p.dtmax;
    q.dx = (p.xmax - p.xmin) / p.Nx; q.dy = (p.ymax - p.ymin) / p.Ny; q.dz = (p.zmax - p.zmin) / p.Nz;
    q.tmax = p.tmax;
    q.nnmax = (1ll << 62);
    e->runs.push_back(q);
    off += q.N;
    if (off >= hyq::kMaxUpdateCells) {
      delete e;
      return efail(HYQ_EINVAL, "more than 2^29 - 1 cells in all runs");
    }
  }
  e->P = off;
  const size_t fsz = prec == HYQ_PREC_FP64 ? sizeof(double) : sizeof(float);
  bool ok = hipStreamCreateWithFlags(&e->stream, hipStreamNonBlocking) == hipSuccess &&
            hipMalloc(&e->R, sizeof(RunDev) * nruns) == hipSuccess &&
            hipMalloc(&e->M, sizeof(double) * 35 * e->P) == hipSuccess &&
            hipMalloc(&e->Mr, sizeof(double) * 35 * e->P) == hipSuccess &&
            hipMalloc(&e->F, fsz * 105 * e->P) == hipSuccess &&
            hipMalloc(&e->vp, fsz * 6 * e->P) == hipSuccess &&
            hipMalloc(&e->flags, sizeof(uint32_t) * e->P) == hipSuccess &&
            hipMalloc(&e->cnt, sizeof(StepCounts)) == hipSuccess;
  for (int i = 0; i < 4 && ok; ++i) ok = hipEventCreate(&e->ev[i]) == hipSuccess;
  long long largest = 0;
  for (const RunDev& q : e->runs) largest = q.N > largest ? q.N : largest;
  if (ok) ok = (e->copy = HostCopy::create(sizeof(double) * 35 * largest)) != nullptr;
  // block tables, one per candidate block size
  for (int ci = 0; ci < 3 && ok; ++ci) {
    std::vector<Blk> tab;
    for (int r = 0; r < nruns; ++r)
      for (long long f = 0; f < e->runs[r].N; f += kCand[ci]) tab.push_back(Blk{r, 0, e->runs[r].off + f});
    e->nblk[ci] = (int)tab.size();
    ok = hipMalloc(&e->T[ci], sizeof(Blk) * tab.size()) == hipSuccess &&
         hipMemcpy(e->T[ci], tab.data(), sizeof(Blk) * tab.size(), hipMemcpyHostToDevice) == hipSuccess;
  }
  if (ok) ok = hipMemcpy(e->R, e->runs.data(), sizeof(RunDev) * nruns, hipMemcpyHostToDevice) == hipSuccess;
  // on the stream of the calls that follow, which does not wait for the null stream: hipMemset
  // may return before its fill is done, and a state set next must not be cleared by it
  if (ok)
    ok = hipMemsetAsync(e->M, 0, sizeof(double) * 35 * e->P, e->stream) == hipSuccess &&
         hipStreamSynchronize(e->stream) == hipSuccess;
  if (!ok) {
    hyq_ensemble_destroy(e);
    return efail(HYQ_ENOMEM, "ensemble allocation");
  }
  *out = e;
  return HYQ_OK;
}

int hyq_ensemble_destroy(hyq_ensemble* e) {
  if (!e) return HYQ_OK;
  if (e->stream) (void)hipStreamSynchronize(e->stream);
  drop_graph(e);
  (void)hipFree(e->R);
  (void)hipFree(e->M);
  (void)hipFree(e->Mr);
  delete e->copy;
  (void)hipFree(e->Mbak);
  (void)hipFree(e->F);
  (void)hipFree(e->vp);
  (void)hipFree(e->flags);
  (void)hipFree(e->cnt);
  for (int i = 0; i < 3; ++i) (void)hipFree(e->T[i]);
  for (int i = 0; i < 4; ++i)
    if (e->ev[i]) (void)hipEventDestroy(e->ev[i]);
  if (e->stream) (void)hipStreamDestroy(e->stream);
  delete e;
  return HYQ_OK;
}

// State of run r (host, Julia layout (Nx,Ny,Nz,35)); resets the run's t and nn to 0.
int hyq_ensemble_set_state(hyq_ensemble* e, int32_t r, const double* M) {
  if (!e || !M || r < 0 || r >= e->nr) return efail(HYQ_EINVAL, "bad argument");
  std::lock_guard<std::mutex> lk(e->mu);
  e->ended = false;
  const RunDev& q = e->runs[r];
  // Mr is free between steps: each step's pass 1 writes it before anything reads it
  ECHK(e->copy->to_device(e->Mr, M, sizeof(double) * 35 * q.N, e->stream), "state upload");
  hipLaunchKernelGGL(ke_strips<true>, dim3((unsigned)((q.N + 255) / 256), 35), dim3(256), 0, e->stream,
                     e->M, e->Mr, e->R + r, q.off, q.N, e->P);
  ECHK(hipGetLastError(), "state upload");
  ECHK(hipStreamSynchronize(e->stream), "sync");
  return HYQ_OK;
}

int hyq_ensemble_get_state(hyq_ensemble* e, int32_t r, double* M) {
  if (!e || !M || r < 0 || r >= e->nr) return efail(HYQ_EINVAL, "bad argument");
  std::lock_guard<std::mutex> lk(e->mu);
  const RunDev& q = e->runs[r];
  hipLaunchKernelGGL(ke_strips<false>, dim3((unsigned)((q.N + 255) / 256), 35), dim3(256), 0, e->stream,
                     e->M, e->Mr, e->R + r, q.off, q.N, e->P);
  ECHK(hipGetLastError(), "state download");
  ECHK(e->copy->to_host(M, e->Mr, sizeof(double) * 35 * q.N, e->stream), "state download");
  return HYQ_OK;
}

// Per-run time, last dt and step count (arrays of nruns; any may be NULL).
int hyq_ensemble_status(hyq_ensemble* e, double* t, double* dt, int64_t* nn) {
  if (!e) return efail(HYQ_EINVAL, "bad argument");
  std::vector<RunDev> h(e->nr);
  ECHK(hipStreamSynchronize(e->stream), "sync");
  ECHK(hipMemcpy(h.data(), e->R, sizeof(RunDev) * e->nr, hipMemcpyDeviceToHost), "run scalars");
  for (int r = 0; r < e->nr; ++r) {
    if (t) t[r] = h[r].t;
    if (dt) dt[r] = h[r].dt;
    if (nn) nn[r] = h[r].nn;
  }
  return HYQ_OK;
}

// nsteps steps of every run still below its tmax (runs past it stay put): graph replays
// when use_graph != 0, else direct launches.  Synchronizes before returning.
int hyq_ensemble_run(hyq_ensemble* e, int64_t nsteps, int32_t use_graph) {
  if (!e || nsteps < 0) return efail(HYQ_EINVAL, "bad argument");
  std::lock_guard<std::mutex> lk(e->mu);
  if (use_graph && !e->exec) {
    const int rc = build_graph(e);
    if (rc) return rc;
  }
  // A step after the end of every run changes nothing, and its empty launches take 28 us: no
  // step is queued once a call has seen that end, and a long call runs in pieces of 32, 64,
  // ... steps and looks for it after each.
  std::vector<RunDev> h(e->nr);
  int64_t left = e->ended ? 0 : nsteps;
  for (int64_t piece = 32;; piece *= 2) {
    const int64_t todo = left < piece ? left : piece;
    for (int64_t s = 0; s < todo; ++s) {
      if (use_graph) {
        ECHK(hipGraphLaunch(e->exec, e->stream), "graph launch");
      } else {
        enqueue(e, e->stream, nullptr);
      }
    }
    ECHK(hipGetLastError(), "ensemble launch");
    ECHK(hipStreamSynchronize(e->stream), "ensemble sync");
    ECHK(hipMemcpy(h.data(), e->R, sizeof(RunDev) * e->nr, hipMemcpyDeviceToHost), "run scalars");
    if (todo > 0) {
      e->ended = true;
      for (const RunDev& q : h) e->ended = e->ended && q.active == 0.0;
    }
    left -= todo;
    if (left == 0 || e->ended) break;
  }
  std::string bad;
  for (int r = 0; r < e->nr; ++r)
    if (h[r].err) bad += (bad.empty() ? "" : ", ") + std::to_string(r);
  if (!bad.empty())
    return efail(HYQ_ENONFINITE, ("non-finite Jacobian in the z wave-speed solve of run(s) " + bad +
                                  " (eigenvalues6z_hyperbolic_3D.jl:108,121 throws); they stopped there")
                                     .c_str());
  return HYQ_OK;
}

// Block sizes (pass 1, update, pass 2), each one of 64, 128, 256.
int hyq_ensemble_set_blocks(hyq_ensemble* e, const int32_t* blocks) {
  if (!e || !blocks) return efail(HYQ_EINVAL, "bad argument");
  for (int i = 0; i < 3; ++i)
    if (cand_index(blocks[i]) < 0) return efail(HYQ_EINVAL, "block size must be 64, 128 or 256");
  std::lock_guard<std::mutex> lk(e->mu);
  for (int i = 0; i < 3; ++i) e->blocks[i] = blocks[i];
  drop_graph(e);
  return HYQ_OK;
}

// Autotuner: for each candidate block size, `trial_steps` steps from the current state
// (saved and restored; run scalars too) timed per kernel with HIP events; each kernel
// keeps its fastest candidate.  ms_out [3][3] (candidate x kernel) may be NULL.
int hyq_ensemble_tune(hyq_ensemble* e, int32_t trial_steps, int32_t* blocks_out, double* ms_out) {
  if (!e || trial_steps < 1) return efail(HYQ_EINVAL, "bad argument");
  std::lock_guard<std::mutex> lk(e->mu);
  if (!e->Mbak) ECHK(hipMalloc(&e->Mbak, sizeof(double) * 35 * e->P), "tuner backup");
  std::vector<RunDev> rbak(e->nr);
  ECHK(hipStreamSynchronize(e->stream), "sync");
  ECHK(hipMemcpy(rbak.data(), e->R, sizeof(RunDev) * e->nr, hipMemcpyDeviceToHost), "run scalars");
  ECHK(hipMemcpyAsync(e->Mbak, e->M, sizeof(double) * 35 * e->P, hipMemcpyDeviceToDevice, e->stream),
       "tuner backup");
  double ms[3][3];
  for (int ci = 0; ci < 3; ++ci) {
    for (int k = 0; k < 3; ++k) e->blocks[k] = kCand[ci];
    for (int k = 0; k < 3; ++k) ms[ci][k] = 0.0;
    for (int s = 0; s < trial_steps; ++s) {
      enqueue(e, e->stream, e->ev);
      ECHK(hipStreamSynchronize(e->stream), "tuner step");
      float a, b, c;
      ECHK(hipEventElapsedTime(&a, e->ev[0], e->ev[1]), "event");
      ECHK(hipEventElapsedTime(&b, e->ev[1], e->ev[2]), "event");
      ECHK(hipEventElapsedTime(&c, e->ev[2], e->ev[3]), "event");
      ms[ci][0] += a;
      ms[ci][1] += b;
      ms[ci][2] += c;
    }
    ECHK(hipMemcpyAsync(e->M, e->Mbak, sizeof(double) * 35 * e->P, hipMemcpyDeviceToDevice, e->stream),
         "tuner restore");
    ECHK(hipMemcpyAsync(e->R, rbak.data(), sizeof(RunDev) * e->nr, hipMemcpyHostToDevice, e->stream),
         "tuner restore");
    ECHK(hipStreamSynchronize(e->stream), "tuner restore");
  }
  for (int k = 0; k < 3; ++k) {
    int best = 0;
    for (int ci = 1; ci < 3; ++ci)
      if (ms[ci][k] < ms[best][k]) best = ci;
    e->blocks[k] = kCand[best];
    if (blocks_out) blocks_out[k] = kCand[best];
  }
  if (ms_out)
    for (int ci = 0; ci < 3; ++ci)
      for (int k = 0; k < 3; ++k) ms_out[ci * 3 + k] = ms[ci][k] / trial_steps;
  drop_graph(e);
  return HYQ_OK;
}

}  // extern "C"
