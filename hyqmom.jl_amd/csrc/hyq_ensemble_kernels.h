// Kernels of the ensemble step (hyq_ensemble.hip), instantiated per precision mode in
// hyq_ens_fp64.hip, hyq_ens_mixed.hip and hyq_ens_newton.hip so that the three compile in
// parallel.  The layout and the block table are described in hyq_ensemble.hip.
#pragma once
#include <hip/hip_runtime.h>

#include <type_traits>

#include "hyq_step_kernels.h"
#include "hyq_update.h"

namespace hyq_ens {
using namespace hyq;

struct RunDev {
  long long off, N;
  int Nx, Ny, Nz, flag2D, positivity, pad;
  double Ma, Kn, CFL, dtmax, dx, dy, dz;
  double t, dt, tmax, active;
  unsigned long long vmax_bits;
  long long nn, nnmax;
  unsigned long long err;  // bit 0: a non-finite z Jacobian (where the reference throws)
};
struct Blk {
  int run, pad;
  long long first;
};

// The runs of an ensemble to the step's kernels: a block is one run's (block table T of the
// kernel's block size).
struct EnsRun {
  static constexpr bool kRoundFast = false, kWide = false;
  RunDev* R;
  const Blk* T;
  __device__ __forceinline__ CellCtx of_run(int run) const {
    RunDev* q = R + run;
    CellCtx x;
    x.active = q->active != 0.0;
    x.in = false;
    x.c = 0;
    x.run = run;
    x.flag2D = q->flag2D;
    x.positivity = q->positivity;
    x.Ma = q->Ma;
    x.Kn = q->Kn;
    x.dt = q->dt;
    x.vmax = &q->vmax_bits;
    x.err = &q->err;
    return x;
  }
  __device__ __forceinline__ CellCtx entry(const Lists& L, unsigned e) const { return of_run(L.run[e]); }
  __device__ __forceinline__ CellCtx cell(unsigned block, int, unsigned t) const {
    const Blk b = T[block];
    CellCtx x = of_run(b.run);
    x.c = b.first + t;
    x.in = x.c < R[b.run].off + R[b.run].N;
    return x;
  }
};

template <int B, typename FT>
__global__ __launch_bounds__(B) void ke_update(const double* __restrict__ Mr, const FT* __restrict__ F,
                                               const FT* __restrict__ vp, double* __restrict__ Mout,
                                               const RunDev* R, const Blk* __restrict__ T, long long P) {
  const Blk b = T[blockIdx.x];
  const RunDev* q = R + b.run;
  if (q->active == 0.0) return;
  const long long c = b.first + threadIdx.x;
  if (c >= q->off + q->N) return;
  const long long l = c - q->off;
  const int Nx = q->Nx, Ny = q->Ny;
  const int i = (int)(l % Nx), j = (int)((l / Nx) % Ny), k = (int)(l / ((long long)Nx * Ny));
  const double dt = q->dt;
  update_cell<FT>(Mr, F, vp, Mout, c, i, j, k, Nx, Ny, q->Nz, P, dt / q->dx, dt / q->dy, dt / q->dz);
}

// Device pointers of the ensemble's planes, its lists (in F) and their counters, and the
// blocks of 64 cells (which k_planes runs on).
struct EnsPtrs {
  double *M, *Mr;
  void *F, *vp;
  uint32_t* flags;
  RunDev* R;
  long long P;
  Lists L;
  StepCounts* cnt;
  const Blk* T64;
  unsigned nblk64;
};

// Launch one of the three phases (0 pass 1, 1 update, 2 pass 2) with block size b for the
// kernels of every cell.
template <typename FT, int EM, bool MIXED>
void launch_cells(int which, int b, unsigned nblk, const Blk* T, const EnsPtrs& p, hipStream_t s) {
  FT* F = (FT*)p.F;
  FT* vp = (FT*)p.vp;
  const EnsRun R{p.R, T}, R64{p.R, p.T64};
  auto cells = [&](auto size) {
    constexpr int B = decltype(size)::value;
    if (which == 0) {
      hipLaunchKernelGGL((k_project<B, EnsRun>), dim3(nblk), dim3(B), 0, s, R, (const double*)p.M, p.Mr,
                         p.flags, p.P);
      launch_planes<EM, 1, FT, EnsRun>(s, R64, p.nblk64, p.Mr, vp, p.flags, (const float*)nullptr, p.L,
                                       p.cnt, p.P);
      hipLaunchKernelGGL((k_close<B, EM, FT, EnsRun>), dim3(nblk), dim3(B), 0, s, R, p.Mr, F, vp, p.flags,
                         p.P);
    } else if (which == 1) {
      hipLaunchKernelGGL((ke_update<B, FT>), dim3(nblk), dim3(B), 0, s, p.Mr, F, vp, p.M, p.R, T, p.P);
    } else {
      hipLaunchKernelGGL((k_project<B, EnsRun>), dim3(nblk), dim3(B), 0, s, R, (const double*)p.M, p.Mr,
                         (uint32_t*)nullptr, p.P);
      launch_planes<EM, 2, FT, EnsRun>(s, R64, p.nblk64, p.Mr, (FT*)nullptr, (uint32_t*)nullptr,
                                       (const float*)nullptr, p.L, p.cnt, p.P);
      hipLaunchKernelGGL((k_relax<B, MIXED, EnsRun>), dim3(nblk), dim3(B), 0, s, R, p.M,
                         (const double*)p.Mr, p.P);
    }
  };
  if (b == 64) cells(std::integral_constant<int, 64>{});
  else if (b == 128) cells(std::integral_constant<int, 128>{});
  else cells(std::integral_constant<int, 256>{});
}

// per-precision entry points (one translation unit each)
void launch_fp64(int which, int b, unsigned nblk, const Blk* T, const EnsPtrs& p, hipStream_t s);
void launch_mixed(int which, int b, unsigned nblk, const Blk* T, const EnsPtrs& p, hipStream_t s);
void launch_newton(int which, int b, unsigned nblk, const Blk* T, const EnsPtrs& p, hipStream_t s);

}  // namespace hyq_ens
