// HIP kernels and the C ABI of libhyqmom_hip.so (declared in include/hyqmom.h).
//
// Device layout: the state is 35 structure-of-arrays moment planes of N = Nx*Ny*Nz
// doubles, cell index i + Nx*(j + Ny*k) -- the reference's own (Nx,Ny,Nz,35) Julia layout,
// so host upload/download is a straight copy.  One step is a chain of launches on the context
// stream, none of which waits on the host (hyq_step_kernels.h holds the cell kernels):
//   k_step_begin  : active = (t < tmax); nn += active; the step's counters to 0   (1 thread)
//   pass 1        : k_project, k_planes (fast modes: k_solve), k_hard, k_close: projection,
//                   x/y/z wave speeds, closure + fluxes, 1D speeds; writes Mr, Fx/Fy/Fz,
//                   vp, flags; wave max |vp| -> atomic max
//   k_dt          : dt = min(CFL*min(dx,dy,dz)/vmax, min(dtmax,Kn), tmax-t); t += dt
//   k_update      : per cell: x/y/z HLL updates with the reference's boundary rules,
//                   combined as Mx+My+Mz-2M
//   pass 2        : k_project, k_planes (k_solve), k_hard, k_relax: projection, x/y wave-speed
//                   corrections, projection, BGK
#include <hip/hip_runtime.h>

#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "../../include/hyqmom.h"
#include "hyq_hostcopy.h"
#include "hyq_step_kernels.h"
#include "hyq_update.h"

using namespace hyq;

extern "C" int hyq_mlp_infer_async(hyq_mlp* m, const float* X, int64_t n, float* P,
                                   hipStream_t stream);
extern "C" int hyq_mlp_infer_masked_async(hyq_mlp* m, const float* X, int64_t n, float* P,
                                          hipStream_t stream);
extern "C" int hyq_mlp_infer_bf16_masked_async(hyq_mlp* m, const short* Xb, int64_t n, float* P,
                                               hipStream_t stream);
extern "C" int hyq_mlp_infer_bf16_segments_async(hyq_mlp* m, const short* Xb, const uint32_t* idx,
                                                 const uint32_t* seg, int64_t nseg, int32_t seg_rows,
                                                 float* P, hipStream_t stream);
extern "C" const float* hyq_mlp_input_norm(hyq_mlp* m);

namespace {

thread_local std::string g_err;

int fail(int code, const char* what, hipError_t e = hipSuccess) {
  g_err = what;
  if (e != hipSuccess) {
    g_err += ": ";
    g_err += hipGetErrorString(e);
  }
  return code;
}
#define HIPCHK(x, msg)                                   \
  do {                                                   \
    hipError_t _e = (x);                                 \
    if (_e != hipSuccess) return fail(HYQ_EHIP, msg, _e); \
  } while (0)

constexpr int kBlock = 128;
constexpr int kNev = 5;  // timing events per step
constexpr const char* kNonfiniteMsg =
    "non-finite Jacobian in the z wave-speed solve (eigenvalues6z_hyperbolic_3D.jl:108,121 throws)";

struct DevScalars {  // device-resident step scalars
  double t, dt, tmax, active;
  unsigned long long vmax_bits;
  long long nn, nnmax;
  unsigned long long err;  // bit 0: a non-finite z Jacobian (where the reference throws)
  StepCounts cnt;
};

// The one run of a context, or a batch (sc null: no step scalars).
struct Solo {
  static constexpr bool kRoundFast = true, kWide = true;
  DevScalars* sc;
  long long N;
  int flag2D, positivity;
  double Ma, Kn;
  __device__ __forceinline__ CellCtx entry(const Lists&, unsigned) const { return all(); }
  __device__ __forceinline__ CellCtx all() const {
    CellCtx x;
    x.run = -1;
    x.active = sc == nullptr || sc->active != 0.0;
    x.in = false;
    x.c = 0;
    x.flag2D = flag2D;
    x.positivity = positivity;
    x.Ma = Ma;
    x.Kn = Kn;
    x.dt = sc != nullptr ? sc->dt : 0.0;
    x.vmax = sc != nullptr ? &sc->vmax_bits : nullptr;
    x.err = sc != nullptr ? &sc->err : nullptr;
    return x;
  }
  __device__ __forceinline__ CellCtx cell(unsigned block, int threads, unsigned t) const {
    CellCtx x = all();
    x.c = (long long)block * threads + t;
    x.in = x.c < N;
    return x;
  }
};

// ---- dt (simulation_runner.jl:402-433, :496) -------------------------------------------
__global__ void k_step_begin(DevScalars* sc) {
  const bool act = (sc->t < sc->tmax) && (sc->nn < sc->nnmax);
  sc->active = act ? 1.0 : 0.0;
  if (act) sc->nn += 1;
  sc->vmax_bits = 0ull;
  clear_counts(&sc->cnt);
}
__global__ void k_dt(DevScalars* sc, double CFL, double hmin, double dtmax, double Kn) {
  if (sc->active == 0.0) return;
  const double vmax = __longlong_as_double((long long)sc->vmax_bits);
  double dt = jmin(CFL * hmin / vmax, jmin(dtmax, Kn));
  dt = jmin(dt, sc->tmax - sc->t);
  sc->dt = dt;
  sc->t += dt;
}

// ---- HLL update (the line logic is in hyq_update.h) ----------------------------------
// FT = double: FP64 fluxes and arithmetic; FT = float: the mixed-precision difference form.
constexpr int kUpdBlock = 256;  // 128: 2-3% slower; 64: 5-9%; 512: 3% (120x120x60)
HD inline unsigned update_grid(long long n) { return (unsigned)((n + kUpdBlock - 1) / kUpdBlock); }
// A thread updates 35 moments one after the other, each a round trip to memory.  A grid too
// small to fill the chip spreads them over kUpdSplit threads instead (blockIdx.y), which
// repeat the face data: a launch takes 34 -> 9.4 us at 20x20x1, 36 -> 11 us at 37x29x17
// (mixed).  With more blocks than CUs the repeats cost as much as the waves give: 48.1 us
// whole, 49.3 us split at 61x53x37 (468 blocks).
constexpr int kUpdSplit = 7;
constexpr unsigned kUpdSplitBelow = 256;  // blocks
template <typename FT, bool SPLIT>
__global__ __launch_bounds__(kUpdBlock) void k_update(const double* __restrict__ Mr,
                                                   const FT* __restrict__ F,
                                                   const FT* __restrict__ vp,
                                                   double* __restrict__ Mout, const DevScalars* sc,
                                                   int Nx, int Ny, int Nz, double dx, double dy,
                                                   double dz) {
  if (sc->active == 0.0) return;
  const long long N = (long long)Nx * Ny * Nz;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const int i = (int)(c % Nx);
  const int j = (int)((c / Nx) % Ny);
  const int k = (int)(c / ((long long)Nx * Ny));
  const double dt = sc->dt;
  constexpr int kPer = SPLIT ? 35 / kUpdSplit : 35;
  const int n0 = SPLIT ? (int)blockIdx.y * kPer : 0;
  update_cell<FT>(Mr, F, vp, Mout, c, i, j, k, Nx, Ny, Nz, N, dt / dx, dt / dy, dt / dz, n0, n0 + kPer);
}

// ---- batch kernels ---------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void k_closure_batch(const double* __restrict__ M, long long N,
                                                          double Ma, int flag2D, double* Mr,
                                                          double* Fx, double* Fy, double* Fz,
                                                          uint32_t* flags) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double m[35], mr[35];
#pragma unroll
  for (int n = 0; n < 35; ++n) m[n] = M[(size_t)n * N + c];
  uint32_t fl = 0;
  if (Fx != nullptr && Fy != nullptr && Fz != nullptr) {
    flux_closure35<true, double, false>(m, flag2D, Ma, mr, Fx + c, Fy + c, Fz + c, (size_t)N, fl);
  } else {
    flux_closure35<false, double, false>(m, flag2D, Ma, mr, nullptr, nullptr, nullptr, 0, fl);
  }
  if (Mr)
#pragma unroll
    for (int n = 0; n < 35; ++n) Mr[(size_t)n * N + c] = mr[n];
  if (flags) flags[c] = fl;
}

// Moments5_3D of n independent cells: M [35][n] in, M5, C5, S5 [21][n] out.
__global__ __launch_bounds__(kBlock) void k_moments5_batch(const double* __restrict__ M,
                                                           long long N, double* __restrict__ M5,
                                                           double* __restrict__ C5,
                                                           double* __restrict__ S5) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double m[35];
#pragma unroll
  for (int n = 0; n < 35; ++n) m[n] = M[(size_t)n * N + c];
  moments5_cell(m, M5 + c, C5 + c, S5 + c, (size_t)N);
}

__global__ __launch_bounds__(kBlock) void k_collision_batch(const double* __restrict__ M,
                                                            long long N, double dt, double Kn,
                                                            int positivity, double* Mo) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double m[35], o[35];
#pragma unroll
  for (int n = 0; n < 35; ++n) m[n] = M[(size_t)n * N + c];
  collision_cell(m, dt, Kn, positivity != 0, o);
#pragma unroll
  for (int n = 0; n < 35; ++n) Mo[(size_t)n * N + c] = o[n];
}

// closure_and_eigenvalues speeds of n 5-moment sets ([5][n]).
__global__ __launch_bounds__(kBlock) void k_closure1d_batch(const double* __restrict__ m5,
                                                            long long N, double* vmin,
                                                            double* vmax) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double a, b;
  closure1d_speeds(m5[c], m5[N + c], m5[2 * N + c], m5[3 * N + c], m5[4 * N + c], a, b);
  vmin[c] = a;
  vmax[c] = b;
}

// pas_HLL on L independent lines of np cells (cell s of line l at l*np + s), FP64: the
// x-direction part of the step's update (hyq_update.h) on its own.
__global__ __launch_bounds__(kBlock) void k_hll_lines(const double* __restrict__ M,
                                                      const double* __restrict__ F,
                                                      const double* __restrict__ vmin,
                                                      const double* __restrict__ vmax,
                                                      long long N, int np, double dtdx,
                                                      double* __restrict__ out) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const int s = (int)(c % np);
  const UpdDir<double> d = upd_dir(vmin + c, vmax + c, s, np, 1);
  const long long l0 = c - s;  // the line's first cell: offsets within the line
  const UpdOff o = upd_off<double, double>(d, (unsigned)s);
  for (int n = 0; n < 35; ++n)
    out[(size_t)n * N + c] =
        upd_value(d, upd_load(o, M + (size_t)n * N + l0, F + (size_t)n * N + l0), dtdx);
}

// eigvals of jacobian6 for a 15-moment slice (jacobian6.jl argument order), sorted by real
// part; computed on the standardized plane and mapped back.
__global__ __launch_bounds__(kBlock) void k_eig6_batch(const double* __restrict__ m15, long long N,
                                                       double* wr_out, double* wi_out) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double r[15];
#pragma unroll
  for (int t = 0; t < 15; ++t) r[t] = m15[(size_t)t * N + c];
  // raw plane moments R[i][j] = m_ij / m00 (i: flux direction)
  double R[5][5];
#pragma unroll
  for (int a = 0; a < 5; ++a)
#pragma unroll
    for (int b = 0; b < 5; ++b) R[a][b] = 0.0;
  const double i0 = 1.0 / r[0];
  R[0][0] = 1.0; R[0][1] = r[1] * i0; R[0][2] = r[2] * i0; R[0][3] = r[3] * i0; R[0][4] = r[4] * i0;
  R[1][0] = r[5] * i0; R[1][1] = r[6] * i0; R[1][2] = r[7] * i0; R[1][3] = r[8] * i0;
  R[2][0] = r[9] * i0; R[2][1] = r[10] * i0; R[2][2] = r[11] * i0; R[3][0] = r[12] * i0;
  R[3][1] = r[13] * i0; R[4][0] = r[14] * i0;
  // embed as a 3D packed array with the third axis empty and shift to central moments
  double cc[35];
#pragma unroll
  for (int t = 0; t < 35; ++t) cc[t] = 0.0;
#pragma unroll
  for (int a = 0; a < 5; ++a)
#pragma unroll
    for (int b = 0; a + b < 5; ++b) cc[tpos(a, b, 0)] = R[a][b];
  const double a = R[1][0], b = R[0][1];
  taylor_shift<0, 4>(cc, -a);
  taylor_shift<1, 4>(cc, -b);
  Plane p = plane<0, 1>(cc, a, b, 0.0);
  double H[36];
  jacobian_std(p, H);
  double wr[6], wi[6];
  bool fin = p.ok;
#pragma unroll
  for (int t = 0; t < 36; ++t) fin = fin && (fabs(H[t]) < 1e300);
  if (fin) {
    balance_n<6>(H);
    hessenberg_n<6>(H);
    fin = hqr_n<6>(H, wr, wi);
  }
  for (int t = 0; t < 6; ++t) {
    if (!fin) { wr[t] = NAN; wi[t] = NAN; }
    else { wr[t] = p.a + p.sig * wr[t]; wi[t] = p.sig * wi[t]; }
  }
  // insertion sort by real part
  for (int x = 1; x < 6; ++x)
    for (int y = x; y > 0 && wr[y] < wr[y - 1]; --y) {
      double tt = wr[y]; wr[y] = wr[y - 1]; wr[y - 1] = tt;
      tt = wi[y]; wi[y] = wi[y - 1]; wi[y - 1] = tt;
    }
  for (int t = 0; t < 6; ++t) {
    wr_out[(size_t)t * N + c] = wr[t];
    wi_out[(size_t)t * N + c] = wi[t];
  }
}

// ---- learned warm start: plane features and the split pass 1 -------------------------
// The five distinct plane Jacobians of a cell, in warm-start slot order: UV, UW, VU, VW, WU.
// Feature row of a plane: its 15 standardized moments in jacobian6.jl argument order
// (S00 S01 S02 S03 S04 S10 S11 S12 S13 S20 S21 S22 S30 S31 S40), padded to 16.
__device__ void plane_feature(const Plane& p, float* x) {
  x[0] = 1.f; x[1] = 0.f; x[2] = 1.f; x[3] = (float)p.S03; x[4] = (float)p.S04;
  x[5] = 0.f; x[6] = (float)p.S11; x[7] = (float)p.S12; x[8] = (float)p.S13;
  x[9] = 1.f; x[10] = (float)p.S21; x[11] = (float)p.S22; x[12] = (float)p.S30;
  x[13] = (float)p.S31; x[14] = (float)p.S40;
  // column 15 is not a network input (normalization zeroes it): it marks the planes the
  // step's masked inference must evaluate (the others take the Gaussian seed)
  x[15] = plane_near_gaussian(p) ? 0.f : 1.f;
}
__device__ void cell_planes(const double* M, Plane pl[5]) {
  double c[35], M000, um, vm, wm;
  raw_to_central4(M, c, M000, um, vm, wm);
  pl[0] = plane<0, 1>(c, um, vm, wm);
  pl[1] = plane<0, 2>(c, um, vm, wm);
  pl[2] = plane<1, 0>(c, um, vm, wm);
  pl[3] = plane<1, 2>(c, um, vm, wm);
  pl[4] = plane<2, 0>(c, um, vm, wm);
}
// Features (and, with L != null, labels from the full FP64 solve: standardized lmin, lmax and
// a validity mask -- finite and real) of the five planes of n cells; sample = plane*n + cell.
__global__ __launch_bounds__(kBlock) void k_plane_dataset(const double* __restrict__ M, long long n,
                                                          float* __restrict__ X, float* L,
                                                          uint8_t* valid) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= n) return;
  double m[35];
#pragma unroll
  for (int t = 0; t < 35; ++t) m[t] = M[(size_t)t * n + c];
  Plane pl[5];
  cell_planes(m, pl);
  for (int q = 0; q < 5; ++q) {
    float x[16];
    plane_feature(pl[q], x);
    x[15] = 0.f;
    float4* dst = reinterpret_cast<float4*>(X + ((size_t)q * n + c) * 16);
#pragma unroll
    for (int t = 0; t < 4; ++t) dst[t] = make_float4(x[4 * t], x[4 * t + 1], x[4 * t + 2], x[4 * t + 3]);
    if (L) {
      uint32_t fl = 0;
      Plane ps = pl[q];
      ps.a = 0.0;
      ps.sig = 1.0;  // standardized eigenvalues
      const EigRes r = plane_eigs(ps, fl);
      L[((size_t)q * n + c) * 2] = (float)r.vmin;
      L[((size_t)q * n + c) * 2 + 1] = (float)r.vmax;
      valid[(size_t)q * n + c] = (r.ok && !r.cplx) ? 1 : 0;
    }
  }
}
// The learned mode's projection (k_project) with the network's work: a plane whose standardized
// moments are within kNetTol of a Gaussian's takes the Gaussian's extreme eigenvalues,
// -sqrt(3), +sqrt(3), as its seeds (written to P directly; NaN for a plane that is not finite); the others are handed to the network as compacted
// rows, normalized with `norm` (16 means, 16 standard deviations) and rounded to bf16 as the
// network's first layer takes them (the same FP32 operations and rounding as its own
// normalization; column 15 is 1).  Each wave owns a segment of kSegRows rows of Xb, one row
// per lane and plane: its rows, plane by plane in lane order, go to the front of its
// segment with their plane indices q N + c in idx, and the wave writes its row count to
// seg[wave].  No atomics: the network's kernel reads each segment's count.
constexpr unsigned kSegRows = 320;  // 64 lanes x 5 planes
__device__ __forceinline__ short to_bf16(float f) { return __builtin_bit_cast(short, (__bf16)f); }
__global__ __launch_bounds__(kBlock, kProjWaves) void k_project_feat(
    const double* __restrict__ M, double* __restrict__ A, short* __restrict__ Xb,
    unsigned* __restrict__ idx, unsigned* __restrict__ seg, float* __restrict__ P,
    uint32_t* __restrict__ flags, DevScalars* sc, long long N, int flag2D, double Ma,
    const float* __restrict__ norm) {
  if (sc->active == 0.0) return;
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;  // whole waves past N never run; the last wave's lane 0 is inside
  double m[35], a[35];
#pragma unroll
  for (int t = 0; t < 35; ++t) m[t] = HYQ_LOAD_STREAM(&M[(size_t)t * N + c]);
  uint32_t fl = 0;
  pass1a_cell(m, flag2D, Ma, a, fl);
#pragma unroll
  for (int t = 0; t < 35; ++t) HYQ_STORE_STREAM(&A[(size_t)t * N + c], a[t]);
  flags[c] = fl;
  Plane pl[5];
  cell_planes(a, pl);
  const unsigned lane = threadIdx.x & 63;
  const long long wave = c / 64;
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned used = 0u;  // rows of the earlier planes (the same on every lane)
  for (int q = 0; q < 5; ++q) {
    const bool need = pl[q].ok && !(plane_gauss_dev(pl[q]) < kNetTol);
    const unsigned long long want = __ballot(need);  // the wave's active lanes
    if (need) {
      const size_t row = (size_t)wave * kSegRows + used + (unsigned)__popcll(want & below);
      float x[16];
      plane_feature(pl[q], x);
      typedef short s8v __attribute__((ext_vector_type(8)));
      s8v h[2];
#pragma unroll
      for (int t = 0; t < 16; ++t) {
        const float v = t < 15 ? (x[t] - norm[t]) / norm[16 + t] : 1.0f;
        h[t / 8][t % 8] = to_bf16(v);
      }
      s8v* dst = reinterpret_cast<s8v*>(Xb + row * 16);
      dst[0] = h[0];
      dst[1] = h[1];
      idx[row] = (unsigned)((long long)q * N + c);
    } else {
      const float g = pl[q].ok ? 1.7320508075688772f : NAN;
      P[((size_t)q * N + c) * 2] = -g;
      P[((size_t)q * N + c) * 2 + 1] = g;
    }
    used += (unsigned)__popcll(want);
  }
  if (lane == 0) seg[wave] = used;
}

// ---- snapshot fields ----------------------------------------------------------------
// compute_central_field / compute_standardized_field (src/utils/compute_standardized_field.jl:
// 16-62): M2CS4_35 (src/moments/M2CS4_35.jl) per cell.  STD = 0: the central moments C4
// (c000 = 1, first order 0); STD = 1: the standardized S4, C4[ijk] / (s_x^i s_y^j s_z^k)
// with s = sqrt(max(C2, eps)) per axis, 1 for the order-0 and pure second-order entries, 0
// for the first order.  Out: [35][N] planes.
template <int STD>
__global__ __launch_bounds__(kBlock) void k_snapshot_field(const double* __restrict__ M,
                                                           long long N, double* __restrict__ out) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  double m[35], cm[35];
#pragma unroll
  for (int n = 0; n < 35; ++n) m[n] = M[(size_t)n * N + c];
  double M000, u, v, w;
  raw_to_central4(m, cm, M000, u, v, w);
  const double sx = sqrt(jmax(cm[tpos(2, 0, 0)], EPS));
  const double sy = sqrt(jmax(cm[tpos(0, 2, 0)], EPS));
  const double sz = sqrt(jmax(cm[tpos(0, 0, 2)], EPS));
#pragma unroll
  for (int n = 0; n < 35; ++n) {
    const int i = e35().e[n][0], j = e35().e[n][1], k = e35().e[n][2];
    const double cv = cm[T35(n)];
    double r = cv;
    if (STD) {
      const int o = i + j + k;
      if (o == 0) r = 1.0;
      else if (o == 1) r = 0.0;
      else if (o == 2 && (i == 2 || j == 2 || k == 2)) r = 1.0;
      else {
        double d = 1.0;
        for (int t = 0; t < i; ++t) d *= sx;
        for (int t = 0; t < j; ++t) d *= sy;
        for (int t = 0; t < k; ++t) d *= sz;
        r = cv / d;
      }
    }
    out[(size_t)n * N + c] = r;
  }
}

// ---- runner diagnostics -------------------------------------------------------------
// Symmetry test of simulation_runner.jl:565-628 on the k = 1 slice: the diagonal cells
// (d, d), d < Nd = min(Nx, Ny), against their mirrors (Nd-1-d, Nd-1-d) for the first five
// moments, differences for moments 1, 3, 5 and sums for 2, 4 (as the reference pairs them);
// per moment max(Diff) / (|Diff|_2 + 1), and the largest magnitude of the five.  One block.
__global__ __launch_bounds__(256) void k_symmetry(const double* __restrict__ M, long long N,
                                                  int Nx, int Ny, double* __restrict__ out) {
  __shared__ double smax[5][256], ssq[5][256];
  const int tid = threadIdx.x;
  const int nd = Nx < Ny ? Nx : Ny;
  double mx[5], sq[5];
#pragma unroll
  for (int n = 0; n < 5; ++n) {
    mx[n] = -INFINITY;
    sq[n] = 0.0;
  }
  for (int d = tid; d < nd; d += 256) {
    const long long a = d + (long long)Nx * d, b = (nd - 1 - d) + (long long)Nx * (nd - 1 - d);
#pragma unroll
    for (int n = 0; n < 5; ++n) {
      const double va = M[(size_t)n * N + a], vb = M[(size_t)n * N + b];
      const double df = (n & 1) ? va + vb : va - vb;
      mx[n] = df > mx[n] ? df : mx[n];
      sq[n] += df * df;
    }
  }
#pragma unroll
  for (int n = 0; n < 5; ++n) {
    smax[n][tid] = mx[n];
    ssq[n][tid] = sq[n];
  }
  __syncthreads();
  for (int h = 128; h > 0; h >>= 1) {
    if (tid < h) {
#pragma unroll
      for (int n = 0; n < 5; ++n) {
        smax[n][tid] = smax[n][tid + h] > smax[n][tid] ? smax[n][tid + h] : smax[n][tid];
        ssq[n][tid] += ssq[n][tid + h];
      }
    }
    __syncthreads();
  }
  if (tid == 0) {
    double r = 0.0;
    for (int n = 0; n < 5; ++n) {
      const double v = smax[n][0] / (sqrt(ssq[n][0]) + 1.0);
      out[n] = v;
      r = fabs(v) > r ? fabs(v) : r;
    }
    out[5] = r;
  }
}

// First-step diagnostics of simulation_runner.jl:404-494 on the last step's wave speeds
// vp [6][N] (x min, x max, y min, y max, z min, z max): bits[0..2] the largest |speed| per
// direction (as ordered bits of non-negative doubles; a NaN speed ranks above every number,
// as the reference's maximum propagates it), bits[4] the largest |speed| over the cells
// without a NaN speed, then the cell that reaches it first in the reference's search order
// (k, then i, then j; its `>` test never takes a NaN cell): bits[3] its key
// (k Nx + i) Ny + j, minimum over the cells that reach bits[4].
template <typename FT>
__global__ __launch_bounds__(kBlock) void k_vmax_dirs(const FT* __restrict__ vp, long long N,
                                                      unsigned long long* __restrict__ bits) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  unsigned long long b[3] = {0ull, 0ull, 0ull}, fin = 0ull;
  if (c < N) {
    bool nan = false;
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const double lo = fabs((double)vp[(size_t)(2 * d) * N + c]);
      const double hi = fabs((double)vp[(size_t)(2 * d + 1) * N + c]);
      const bool dn = lo != lo || hi != hi;
      nan = nan || dn;
      b[d] = dn ? 0x7FF8000000000000ull : __double_as_longlong(hi > lo ? hi : lo);
    }
    if (!nan) {
      fin = b[0] > b[1] ? b[0] : b[1];
      fin = b[2] > fin ? b[2] : fin;
    }
  }
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const unsigned long long w = wave_max_u64(b[d]);
    if ((threadIdx.x & 63) == 0) atomicMax(&bits[d], w);
  }
  const unsigned long long wf = wave_max_u64(fin);
  if ((threadIdx.x & 63) == 0) atomicMax(&bits[4], wf);
}
template <typename FT>
__global__ __launch_bounds__(kBlock) void k_vmax_worst(const FT* __restrict__ vp, long long N,
                                                       int Nx, int Ny,
                                                       unsigned long long* __restrict__ bits) {
  const long long c = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (c >= N) return;
  const unsigned long long g = bits[4];
  unsigned long long m = 0ull;
#pragma unroll
  for (int t = 0; t < 6; ++t) {
    const double v = fabs((double)vp[(size_t)t * N + c]);
    if (v != v) return;
    const unsigned long long vb = __double_as_longlong(v);
    m = vb > m ? vb : m;
  }
  if (m != g) return;
  const long long i = c % Nx, j = (c / Nx) % Ny, k = c / ((long long)Nx * Ny);
  atomicMin(&bits[3], (unsigned long long)((k * Nx + i) * Ny + j));
}

unsigned grid_for(long long n) { return (unsigned)((n + kBlock - 1) / kBlock); }

}  // namespace

// ---------------------------------------------------------------------------------------
// Context
// Steps that hyq_run queues before it reads the device scalars back: a run stops within one
// chunk of reaching tmax, however large nnmax is.  A queued step past the end is a chain of
// empty launches, 45 us.  So a call that leaves the end to tmax (nnmax further away than a
// chunk) starts with kFirst steps, and then queues no more than the last dt makes of the
// time that is left: 4 steps to tmax at 20x20x1 FP64 3.2 -> 1.1 ms.
constexpr int kChunk = 64, kFirst = 16;

struct hyq_ctx {
  hyq_params p;
  long long N;
  double dx, dy, dz;
  hipStream_t stream;
  double* M;       // [35][N]
  double* Mr;      // [35][N]
  void* F;         // [105][N] double (FP64) or float (mixed)
  void* vp;        // [6][N]
  uint32_t* flags; // [N]
  DevScalars* sc;
  hipEvent_t ev[kNev * kChunk];  // per step: pass 1 | dt | update | pass 2 (a ring of kChunk steps)
  double ms_pass1, ms_update, ms_pass2;
  long long timed_steps;
  hyq_mlp* mlp;  // learned mode: warm-start network (not owned)
  float* X;        // learned mode: the network's input rows, a segment of kSegRows rows of
                   // 16 bf16 per wave of 64 cells
  unsigned* Xidx;  // [segments x kSegRows] plane index q N + c of each row
  unsigned* Xseg;  // [ceil(N / 64)] rows in each wave's segment
  float* P;        // [5N][2] seeds of each plane: the network's predictions or the Gaussian's
  Lists L;         // the entries of a pass, in F, which is free then
  double* diag;            // [8] results of the diagnostics
  HostCopy* copy;          // the state's copies from and to the host
};

extern "C" {

const char* hyq_last_error(void) { return g_err.c_str(); }
const char* hyq_version(void) { return "hyqmom-mi355x 0.2 (gfx950)"; }

int hyq_create(const hyq_params* params, hyq_ctx** out) {
  if (!params || !out) return fail(HYQ_EINVAL, "null argument");
  const hyq_params& p = *params;
  if (p.Nmom != 35) return fail(HYQ_EINVAL, "Nmom must be 35");
  if (p.Nx < 1 || p.Ny < 1 || p.Nz < 1) return fail(HYQ_EINVAL, "grid sizes must be >= 1");
  if ((long long)p.Nx * p.Ny * p.Nz >= kMaxUpdateCells)
    return fail(HYQ_EINVAL, "more than 2^29 - 1 cells");
  if (p.precision < HYQ_PREC_FP64 || p.precision > HYQ_PREC_MIXED_NEWTON)
    return fail(HYQ_EINVAL, "unknown precision mode");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(HYQ_ENODEV, "no HIP device");
  hyq_ctx* c = new hyq_ctx();
  std::memset(c, 0, sizeof(*c));
  c->p = p;
  c->N = (long long)p.Nx * p.Ny * p.Nz;
  c->dx = (p.xmax - p.xmin) / p.Nx;  // simulation_runner.jl:133-139
  c->dy = (p.ymax - p.ymin) / p.Ny;
  c->dz = (p.zmax - p.zmin) / p.Nz;
  const size_t fsz = p.precision == HYQ_PREC_FP64 ? sizeof(double) : sizeof(float);
  hipError_t e;
  if ((e = hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking)) != hipSuccess) {
    delete c;
    return fail(HYQ_EHIP, "hipStreamCreate", e);
  }
  bool ok = hipMalloc(&c->M, sizeof(double) * 35 * c->N) == hipSuccess &&
            hipMalloc(&c->Mr, sizeof(double) * 35 * c->N) == hipSuccess &&
            hipMalloc(&c->F, fsz * 105 * c->N) == hipSuccess &&
            hipMalloc(&c->vp, fsz * 6 * c->N) == hipSuccess &&
            hipMalloc(&c->flags, sizeof(uint32_t) * c->N) == hipSuccess &&
            hipMalloc(&c->sc, sizeof(DevScalars)) == hipSuccess &&
            hipMalloc(&c->diag, sizeof(double) * 8) == hipSuccess;
  if (ok && p.precision == HYQ_PREC_MIXED_LEARNED)
    ok = hipMalloc(&c->X, sizeof(short) * 16 * kSegRows * ((c->N + 63) / 64)) == hipSuccess &&
         hipMalloc(&c->Xidx, sizeof(unsigned) * kSegRows * ((c->N + 63) / 64)) == hipSuccess &&
         hipMalloc(&c->Xseg, sizeof(unsigned) * ((c->N + 63) / 64)) == hipSuccess &&
         hipMalloc(&c->P, sizeof(float) * 2 * 5 * c->N) == hipSuccess &&
         // no rows until a step's projection has listed some: the network's kernel then
         // reads counts of 0 (it runs, as every kernel of the step, also in a step that has
         // nothing left to do).  On the steps' own stream, which does not wait for the null
         // stream, where a fill may outlast its call
         hipMemsetAsync(c->Xseg, 0, sizeof(unsigned) * ((c->N + 63) / 64), c->stream) == hipSuccess &&
         hipStreamSynchronize(c->stream) == hipSuccess;
  if (ok) c->L = carve_lists(c->F, c->N);
  if (ok) ok = (c->copy = HostCopy::create(sizeof(double) * 35 * c->N)) != nullptr;
  if (!ok) {
    hyq_destroy(c);
    return fail(HYQ_ENOMEM, "device allocation failed");
  }
  for (int i = 0; i < kNev * kChunk; ++i) {
    if ((e = hipEventCreate(&c->ev[i])) != hipSuccess) {
      hyq_destroy(c);
      return fail(HYQ_EHIP, "hipEventCreate", e);
    }
  }
  *out = c;
  return HYQ_OK;
}

int hyq_destroy(hyq_ctx* c) {
  if (!c) return HYQ_OK;
  if (c->stream) hipStreamSynchronize(c->stream);
  hipFree(c->M);
  hipFree(c->Mr);
  hipFree(c->F);
  hipFree(c->vp);
  hipFree(c->flags);
  hipFree(c->sc);
  hipFree(c->diag);
  hipFree(c->X);
  hipFree(c->Xidx);
  hipFree(c->Xseg);
  hipFree(c->P);
  delete c->copy;
  for (int i = 0; i < kNev * kChunk; ++i)
    if (c->ev[i]) hipEventDestroy(c->ev[i]);
  if (c->stream) hipStreamDestroy(c->stream);
  delete c;
  return HYQ_OK;
}

int hyq_set_state(hyq_ctx* c, const double* M) {
  if (!c || !M) return fail(HYQ_EINVAL, "null argument");
  HIPCHK(c->copy->to_device(c->M, M, sizeof(double) * 35 * c->N, c->stream), "set_state copy");
  return HYQ_OK;
}

int hyq_get_state(hyq_ctx* c, double* M) {
  if (!c || !M) return fail(HYQ_EINVAL, "null argument");
  HIPCHK(c->copy->to_host(M, c->M, sizeof(double) * 35 * c->N, c->stream), "get_state copy");
  return HYQ_OK;
}

}  // extern "C"

// One step on the context stream; ev (or null): kNev events bracketing its parts.  FT: the
// fluxes' and speeds' type (float: the mixed modes); EM: 1 for the fast modes.
template <typename FT, int EM>
static int enqueue_step_t(hyq_ctx* c, hipEvent_t* ev) {
  constexpr bool kMixed = sizeof(FT) == 4;
  const hyq_params& p = c->p;
  const unsigned g = grid_for(c->N), g64 = (unsigned)((c->N + 63) / 64);
  const double hmin = jmin(jmin(c->dx, c->dy), c->dz);
  const Solo R{c->sc, c->N, p.flag2D, p.positivity, p.Ma, p.Kn};
  FT* F = (FT*)c->F;
  FT* vp = (FT*)c->vp;
  hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(1), 0, c->stream, c->sc);
  if (ev) hipEventRecord(ev[0], c->stream);
  const bool learned = p.precision == HYQ_PREC_MIXED_LEARNED && c->mlp != nullptr;
  if (learned) {
    // the network's input rows and warm starts with the projection
    hipLaunchKernelGGL(k_project_feat, dim3(g), dim3(kBlock), 0, c->stream, c->M, c->Mr,
                       reinterpret_cast<short*>(c->X), c->Xidx, c->Xseg, c->P, c->flags, c->sc,
                       c->N, p.flag2D, p.Ma, hyq_mlp_input_norm(c->mlp));
    const int rc = hyq_mlp_infer_bf16_segments_async(
        c->mlp, reinterpret_cast<const short*>(c->X), c->Xidx, c->Xseg, (c->N + 63) / 64,
        (int32_t)kSegRows, c->P, c->stream);
    if (rc) return rc;
  } else {
    hipLaunchKernelGGL((k_project<kBlock, Solo>), dim3(g), dim3(kBlock), 0, c->stream, R, c->M, c->Mr,
                       c->flags, c->N);
  }
  launch_planes<EM, 1, FT, Solo>(c->stream, R, g64, c->Mr, vp, c->flags,
                                 learned ? (const float*)c->P : (const float*)nullptr, c->L,
                                 &c->sc->cnt, c->N);
  hipLaunchKernelGGL((k_close<kBlock, EM, FT, Solo>), dim3(g), dim3(kBlock), 0, c->stream, R, c->Mr, F,
                     vp, c->flags, c->N);
  if (ev) hipEventRecord(ev[1], c->stream);
  hipLaunchKernelGGL(k_dt, dim3(1), dim3(1), 0, c->stream, c->sc, p.CFL, hmin, p.dtmax, p.Kn);
  if (ev) hipEventRecord(ev[2], c->stream);
  const unsigned ub = update_grid(c->N);
  if (ub < kUpdSplitBelow)
    hipLaunchKernelGGL((k_update<FT, true>), dim3(ub, kUpdSplit), dim3(kUpdBlock), 0, c->stream, c->Mr,
                       (const FT*)F, (const FT*)vp, c->M, c->sc, p.Nx, p.Ny, p.Nz, c->dx, c->dy, c->dz);
  else
    hipLaunchKernelGGL((k_update<FT, false>), dim3(ub), dim3(kUpdBlock), 0, c->stream, c->Mr,
                       (const FT*)F, (const FT*)vp, c->M, c->sc, p.Nx, p.Ny, p.Nz, c->dx, c->dy, c->dz);
  if (ev) hipEventRecord(ev[3], c->stream);
  hipLaunchKernelGGL((k_project<kBlock, Solo>), dim3(g), dim3(kBlock), 0, c->stream, R,
                     (const double*)c->M, c->Mr, (uint32_t*)nullptr, c->N);
  launch_planes<EM, 2, FT, Solo>(c->stream, R, g64, c->Mr, (FT*)nullptr, (uint32_t*)nullptr,
                                 (const float*)nullptr, c->L, &c->sc->cnt, c->N);
  hipLaunchKernelGGL((k_relax<kBlock, kMixed, Solo>), dim3(g), dim3(kBlock), 0, c->stream, R, c->M,
                     (const double*)c->Mr, c->N);
  if (ev) hipEventRecord(ev[4], c->stream);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(HYQ_EHIP, "kernel launch", e);
  return HYQ_OK;
}
static int enqueue_step(hyq_ctx* c, hipEvent_t* ev) {
  if (c->p.precision == HYQ_PREC_FP64) return enqueue_step_t<double, 0>(c, ev);
  if (c->p.precision == HYQ_PREC_MIXED) return enqueue_step_t<float, 0>(c, ev);
  return enqueue_step_t<float, 1>(c, ev);
}

extern "C" {

static int load_scalars(hyq_ctx* c, double t, long long nn, double tmax, long long nnmax) {
  DevScalars s;
  std::memset(&s, 0, sizeof(s));
  s.t = t;
  s.tmax = tmax;
  s.nn = nn;
  s.nnmax = nnmax;
  HIPCHK(hipMemcpyAsync(c->sc, &s, sizeof(s), hipMemcpyHostToDevice, c->stream), "scalars");
  return HYQ_OK;
}

static int accumulate_times(hyq_ctx* c, hipEvent_t* ev) {
  float a = 0, b = 0, d = 0;
  HIPCHK(hipEventElapsedTime(&a, ev[0], ev[1]), "event time");
  HIPCHK(hipEventElapsedTime(&b, ev[2], ev[3]), "event time");
  HIPCHK(hipEventElapsedTime(&d, ev[3], ev[4]), "event time");
  c->ms_pass1 += a;
  c->ms_update += b;
  c->ms_pass2 += d;
  c->timed_steps += 1;
  return HYQ_OK;
}

int hyq_step(hyq_ctx* c, double* t_inout, double* dt_out, int64_t* nn_inout) {
  if (!c || !t_inout || !nn_inout) return fail(HYQ_EINVAL, "null argument");
  // one pass of the loop body; a no-op if t >= tmax (the caller owns the loop condition)
  int rc = load_scalars(c, *t_inout, *nn_inout, c->p.tmax, (long long)*nn_inout + 1);
  if (rc) return rc;
  rc = enqueue_step(c, c->ev);
  if (rc) {
    hipStreamSynchronize(c->stream);
    return rc;
  }
  DevScalars s;
  HIPCHK(hipMemcpyAsync(&s, c->sc, sizeof(s), hipMemcpyDeviceToHost, c->stream), "scalars back");
  HIPCHK(hipStreamSynchronize(c->stream), "step sync");
  if (s.active != 0.0) {
    rc = accumulate_times(c, c->ev);
    if (rc) return rc;
  }
  *t_inout = s.t;
  if (dt_out) *dt_out = s.active != 0.0 ? s.dt : 0.0;
  *nn_inout = s.nn;
  if (s.err) return fail(HYQ_ENONFINITE, kNonfiniteMsg);
  return HYQ_OK;
}

int hyq_run(hyq_ctx* c, double tmax, int64_t nnmax, double* t_inout, int64_t* nn_inout) {
  if (!c || !t_inout || !nn_inout) return fail(HYQ_EINVAL, "null argument");
  int rc = load_scalars(c, *t_inout, *nn_inout, tmax, nnmax);
  if (rc) return rc;
  // Steps are queued in chunks of kChunk; a step after t >= tmax (or nn >= nnmax) is a no-op
  // on the device.  After each chunk the scalars come back, and the run ends once a chunk
  // left it inactive, or on an error.  HIP events from a ring of kChunk steps bracket pass 1,
  // the update and pass 2 of every step.
  long long nn0 = *nn_inout;
  DevScalars s;
  std::memset(&s, 0, sizeof(s));
  s.t = *t_inout;
  s.nn = nn0;
  bool more = s.t < tmax && s.nn < (long long)nnmax;
  double steps = (long long)nnmax - s.nn > kChunk ? kFirst : kChunk;  // to tmax, as far as known
  while (more) {
    const long long left = (long long)nnmax - s.nn;
    int todo = (int)(left < kChunk ? left : kChunk);
    if (steps < todo) todo = (int)steps;
    for (int q = 0; q < todo && rc == HYQ_OK; ++q) rc = enqueue_step(c, &c->ev[kNev * q]);
    if (rc) {
      hipStreamSynchronize(c->stream);
      return rc;
    }
    HIPCHK(hipMemcpyAsync(&s, c->sc, sizeof(s), hipMemcpyDeviceToHost, c->stream), "scalars back");
    HIPCHK(hipStreamSynchronize(c->stream), "run sync");
    const long long ran = s.nn - nn0;  // active steps of this chunk (they come first)
    for (long long q = 0; q < ran && rc == HYQ_OK; ++q) rc = accumulate_times(c, &c->ev[kNev * q]);
    if (rc) return rc;
    nn0 = s.nn;
    if (s.err) break;
    more = s.active != 0.0 && s.t < tmax && s.nn < (long long)nnmax;
    steps = (tmax - s.t) / s.dt + 1.0;
    if (!(steps >= 1.0)) steps = kChunk;  // a dt that is zero or not a number
  }
  *t_inout = s.t;
  *nn_inout = s.nn;
  if (s.err) return fail(HYQ_ENONFINITE, kNonfiniteMsg);
  return HYQ_OK;
}

int hyq_get_wave_speeds(hyq_ctx* c, double* vp) {
  if (!c || !vp) return fail(HYQ_EINVAL, "null argument");
  if (c->p.precision == HYQ_PREC_FP64) {
    HIPCHK(hipMemcpy(vp, c->vp, sizeof(double) * 6 * c->N, hipMemcpyDeviceToHost), "vp copy");
  } else {
    float* tmp = new float[6 * c->N];
    const hipError_t e = hipMemcpy(tmp, c->vp, sizeof(float) * 6 * c->N, hipMemcpyDeviceToHost);
    if (e == hipSuccess)
      for (long long i = 0; i < 6 * c->N; ++i) vp[i] = tmp[i];
    delete[] tmp;
    HIPCHK(e, "vp copy");
  }
  return HYQ_OK;
}

int hyq_snapshot_fields(hyq_ctx* c, double* C, double* S) {
  if (!c) return fail(HYQ_EINVAL, "null argument");
  // Mr is free between steps (each step's pass 1 rewrites it before reading it)
  const unsigned g = grid_for(c->N);
  for (int which = 0; which < 2; ++which) {
    double* dst = which == 0 ? C : S;
    if (!dst) continue;
    if (which == 0)
      hipLaunchKernelGGL(k_snapshot_field<0>, dim3(g), dim3(kBlock), 0, c->stream,
                         (const double*)c->M, c->N, c->Mr);
    else
      hipLaunchKernelGGL(k_snapshot_field<1>, dim3(g), dim3(kBlock), 0, c->stream,
                         (const double*)c->M, c->N, c->Mr);
    HIPCHK(hipGetLastError(), "snapshot field launch");
    HIPCHK(c->copy->to_host(dst, c->Mr, sizeof(double) * 35 * c->N, c->stream), "snapshot field copy");
  }
  return HYQ_OK;
}

int hyq_symmetry_maxdiff(hyq_ctx* c, double* maxdiff, double* per_moment) {
  if (!c || !maxdiff) return fail(HYQ_EINVAL, "null argument");
  double h[6];
  hipLaunchKernelGGL(k_symmetry, dim3(1), dim3(256), 0, c->stream, (const double*)c->M, c->N,
                     c->p.Nx, c->p.Ny, c->diag);
  HIPCHK(hipGetLastError(), "symmetry launch");
  HIPCHK(hipMemcpyAsync(h, c->diag, sizeof(h), hipMemcpyDeviceToHost, c->stream), "symmetry copy");
  HIPCHK(hipStreamSynchronize(c->stream), "symmetry sync");
  *maxdiff = h[5];
  if (per_moment)
    for (int n = 0; n < 5; ++n) per_moment[n] = h[n];
  return HYQ_OK;
}

int hyq_vmax_breakdown(hyq_ctx* c, double* vdir, int64_t* worst) {
  if (!c || !vdir) return fail(HYQ_EINVAL, "null argument");
  unsigned long long h[5] = {0ull, 0ull, 0ull, ~0ull, 0ull};
  unsigned long long* d = reinterpret_cast<unsigned long long*>(c->diag);
  HIPCHK(hipMemcpyAsync(d, h, sizeof(h), hipMemcpyHostToDevice, c->stream), "vmax init");
  const unsigned g = grid_for(c->N);
  if (c->p.precision == HYQ_PREC_FP64) {
    hipLaunchKernelGGL(k_vmax_dirs<double>, dim3(g), dim3(kBlock), 0, c->stream,
                       (const double*)c->vp, c->N, d);
    hipLaunchKernelGGL(k_vmax_worst<double>, dim3(g), dim3(kBlock), 0, c->stream,
                       (const double*)c->vp, c->N, c->p.Nx, c->p.Ny, d);
  } else {
    hipLaunchKernelGGL(k_vmax_dirs<float>, dim3(g), dim3(kBlock), 0, c->stream,
                       (const float*)c->vp, c->N, d);
    hipLaunchKernelGGL(k_vmax_worst<float>, dim3(g), dim3(kBlock), 0, c->stream,
                       (const float*)c->vp, c->N, c->p.Nx, c->p.Ny, d);
  }
  HIPCHK(hipGetLastError(), "vmax launch");
  HIPCHK(hipMemcpyAsync(h, d, sizeof(h), hipMemcpyDeviceToHost, c->stream), "vmax copy");
  HIPCHK(hipStreamSynchronize(c->stream), "vmax sync");
  for (int k = 0; k < 3; ++k) {
    double v;
    std::memcpy(&v, &h[k], sizeof(v));
    vdir[k] = v;
  }
  if (worst && h[3] == ~0ull) {  // every cell has a NaN speed
    worst[0] = worst[1] = worst[2] = -1;
  } else if (worst) {
    const long long key = (long long)h[3], Nx = c->p.Nx, Ny = c->p.Ny;
    worst[0] = (key / Ny) % Nx;      // i
    worst[1] = key % Ny;             // j
    worst[2] = key / (Ny * Nx);      // k
  }
  return HYQ_OK;
}

int hyq_get_flags(hyq_ctx* c, uint32_t* flags) {
  if (!c || !flags) return fail(HYQ_EINVAL, "null argument");
  HIPCHK(hipMemcpy(flags, c->flags, sizeof(uint32_t) * c->N, hipMemcpyDeviceToHost), "flags copy");
  return HYQ_OK;
}

int hyq_kernel_times(hyq_ctx* c, double* ms_pass1, double* ms_update, double* ms_pass2,
                     int64_t* nsteps) {
  if (!c) return fail(HYQ_EINVAL, "null argument");
  const double n = c->timed_steps > 0 ? (double)c->timed_steps : 1.0;
  if (ms_pass1) *ms_pass1 = c->ms_pass1 / n;
  if (ms_update) *ms_update = c->ms_update / n;
  if (ms_pass2) *ms_pass2 = c->ms_pass2 / n;
  if (nsteps) *nsteps = c->timed_steps;
  return HYQ_OK;
}

int hyq_deferred_cells(hyq_ctx* c, int64_t* pass1, int64_t* pass2) {
  if (!c) return fail(HYQ_EINVAL, "null argument");
  DevScalars s;
  HIPCHK(hipMemcpyAsync(&s, c->sc, sizeof(s), hipMemcpyDeviceToHost, c->stream), "scalars back");
  HIPCHK(hipStreamSynchronize(c->stream), "sync");
  const StepCounts& n = s.cnt;
  if (pass1) *pass1 = (int64_t)n.nhard[0] + (int64_t)n.nslot[0] - (int64_t)n.ncplx[0];
  if (pass2) *pass2 = (int64_t)n.nhard[1] + (int64_t)n.nslot[1] - (int64_t)n.ncplx[1];
  return HYQ_OK;
}

int hyq_fast_path_counts(hyq_ctx* c, int64_t* counts) {
  if (!c || !counts) return fail(HYQ_EINVAL, "null argument");
  DevScalars s;
  HIPCHK(hipMemcpyAsync(&s, c->sc, sizeof(s), hipMemcpyDeviceToHost, c->stream), "scalars back");
  HIPCHK(hipStreamSynchronize(c->stream), "sync");
  const StepCounts& n = s.cnt;
  const unsigned v[8] = {n.nslot[0], n.npend[0], n.ncplx[0], n.nhard[0] - n.ncplx[0],
                         n.nslot[1], n.npend[1], n.ncplx[1], n.nhard[1] - n.ncplx[1]};
  for (int k = 0; k < 8; ++k) counts[k] = (int64_t)v[k];
  return HYQ_OK;
}

int hyq_reset_kernel_times(hyq_ctx* c) {
  if (!c) return fail(HYQ_EINVAL, "null argument");
  c->ms_pass1 = c->ms_update = c->ms_pass2 = 0.0;
  c->timed_steps = 0;
  return HYQ_OK;
}

int hyq_closure_batch(const double* M, int64_t n, double Ma, int32_t flag2D, double* Mr,
                      double* Fx, double* Fy, double* Fz, uint32_t* flags) {
  if (!M || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_closure_batch, dim3(grid_for(n)), dim3(kBlock), 0, 0, M, (long long)n, Ma,
                     flag2D, Mr, Fx, Fy, Fz, flags);
  HIPCHK(hipGetLastError(), "closure launch");
  HIPCHK(hipDeviceSynchronize(), "closure sync");
  return HYQ_OK;
}

int hyq_moments5_batch(const double* M, int64_t n, double* M5, double* C5, double* S5) {
  if (!M || !M5 || !C5 || !S5 || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_moments5_batch, dim3(grid_for(n)), dim3(kBlock), 0, 0, M, (long long)n, M5,
                     C5, S5);
  HIPCHK(hipGetLastError(), "moments5 launch");
  HIPCHK(hipDeviceSynchronize(), "moments5 sync");
  return HYQ_OK;
}

static int batch_args(const double* M, int64_t n, int32_t precision, const double* Mr,
                      const double* Fx, const double* Fy, const double* Fz, const double* vp,
                      const uint32_t* flags) {
  if (!M || !Mr || !Fx || !Fy || !Fz || !vp || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (precision != HYQ_PREC_FP64 && precision != HYQ_PREC_MIXED_NEWTON)
    return fail(HYQ_EINVAL, "batch wave speeds: precision must be FP64 or MIXED_NEWTON");
  if (precision == HYQ_PREC_MIXED_NEWTON && !flags)
    return fail(HYQ_EINVAL, "the fast batch needs the flags output");
  if (n > 0x7FFFFFFFLL / 5) return fail(HYQ_EINVAL, "batch too large");
  // the three flux outputs must be one [105][n] block for the pass-1 kernels
  if (n > 0 && (Fy != Fx + (size_t)35 * n || Fz != Fx + (size_t)70 * n))
    return fail(HYQ_EINVAL, "Fx, Fy, Fz must be consecutive [35][n] blocks");
  return HYQ_OK;
}

}  // extern "C"

// Scratch of a batch of n cells: the flux output, which k_close alone writes, holds the
// z-path states [35][n], the counters, the entries' lists, and the flags when the caller
// wants none.  The counters take 64-bit atomics: they sit on a double's boundary, ahead of
// the 32-bit lists, whose length may be odd.
struct BatchCounts {
  StepCounts step;
  unsigned long long wide[kWideRounds + 1];
};
constexpr size_t kCountDoubles = sizeof(BatchCounts) / sizeof(double);
static_assert(kCountDoubles * sizeof(double) == sizeof(BatchCounts), "whole doubles");
static_assert(35 * sizeof(double) + sizeof(BatchCounts) + kListBytes + sizeof(uint32_t) <= 105 * sizeof(double),
              "a batch's scratch fits the fluxes");
// The counters start at zero, on the stream of the kernels that count.
__global__ void k_batch_begin(BatchCounts* n) {
  clear_counts(&n->step);
  for (int r = 0; r <= kWideRounds; ++r) n->wide[r] = 0ull;
}
// Batches from this size on take their entries through a launch per phase, 13 launches for one.
// The number of entries, which decides what is faster, is known on the device only; with few
// of them the launches cost 45 us.  us, k_hard / wide, by cells:
//                  131072       160000       199999       262144       400000       1000000
//   mixtures FP64  2008 / 2258  2643 / 2637  3649 / 3192  3677 / 3780  5920 / 5347  13713 / 11836
//            fast  1676 / 1776  2362 / 2144  2545 / 2634  3100 / 2814  4688 / 4176  11107 / 9278
//   jets     FP64   487 / 521    662 / 701    822 / 869    828 / 866   1215 / 1253   2568 / 2594
//            fast   218 / 261    266 / 301    323 / 373    338 / 372    452 / 497     959 / 957
constexpr long long kWideCells = 200000;
static_assert(35 * sizeof(double) + sizeof(BatchCounts) / 1000 + kListBytes + sizeof(uint32_t) + kWideBytes <=
                  105 * sizeof(double), "a large batch's scratch fits the fluxes");
// Pass 1 of the step on a batch (FP64 outputs), no allocation.
template <int EM>
static void enqueue_batch(const double* M, long long n, double Ma, int flag2D, int positivity,
                          double* Mr, double* F, double* vp, uint32_t* flags) {
  const Solo R{nullptr, n, flag2D, positivity, Ma, 0.0};
  BatchCounts* cnt = reinterpret_cast<BatchCounts*>(F + (size_t)35 * n);
  const Lists L = carve_lists(F, n, kCountDoubles);
  uint32_t* fl = L.item + 5 * (size_t)n;
  const WideLists W{fl + (size_t)n,     fl + 2 * (size_t)n, fl + 3 * (size_t)n,
                    fl + 4 * (size_t)n, fl + 5 * (size_t)n, cnt->wide};
  if (flags) fl = flags;
  const unsigned g = grid_for(n);
  hipLaunchKernelGGL((k_project<kBlock, Solo>), dim3(g), dim3(kBlock), 0, 0, R, M, Mr, fl, n);
  hipLaunchKernelGGL(k_batch_begin, dim3(1), dim3(1), 0, 0, cnt);
  launch_planes<EM, 1, double, Solo>(0, R, (unsigned)((n + 63) / 64), Mr, vp, fl, (const float*)nullptr,
                                     L, &cnt->step, n, n >= kWideCells ? &W : nullptr);
  hipLaunchKernelGGL((k_close<kBlock, EM, double, Solo>), dim3(g), dim3(kBlock), 0, 0, R, Mr, F, vp,
                     flags, n);
}

extern "C" {

int hyq_wavespeed_batch(const double* M, int64_t n, double Ma, int32_t flag2D,
                        int32_t positivity, int32_t precision, double* Mr, double* Fx,
                        double* Fy, double* Fz, double* vp, uint32_t* flags) {
  const int rc = batch_args(M, n, precision, Mr, Fx, Fy, Fz, vp, flags);
  if (rc) return rc;
  if (n == 0) return HYQ_OK;
  if (precision == HYQ_PREC_FP64) enqueue_batch<0>(M, n, Ma, flag2D, positivity, Mr, Fx, vp, flags);
  else enqueue_batch<1>(M, n, Ma, flag2D, positivity, Mr, Fx, vp, flags);
  HIPCHK(hipGetLastError(), "batch launch");
  HIPCHK(hipDeviceSynchronize(), "batch sync");
  return HYQ_OK;
}

constexpr long long kNoAllocMaxCells = 1LL << 16;
int hyq_wavespeed_batch_noalloc(const double* M, int64_t n, double Ma, int32_t flag2D,
                                int32_t positivity, int32_t precision, double* Mr, double* Fx,
                                double* Fy, double* Fz, double* vp, uint32_t* flags) {
  const int rc = batch_args(M, n, precision, Mr, Fx, Fy, Fz, vp, flags);
  if (rc) return rc;
  if (n > kNoAllocMaxCells)
    return fail(HYQ_EINVAL, "hyq_wavespeed_batch_noalloc: at most 65536 cells per call");
  return hyq_wavespeed_batch(M, n, Ma, flag2D, positivity, precision, Mr, Fx, Fy, Fz, vp, flags);
}

int hyq_eig6_batch(const double* m15, int64_t n, double* wr, double* wi) {
  if (!m15 || !wr || !wi || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_eig6_batch, dim3(grid_for(n)), dim3(kBlock), 0, 0, m15, (long long)n, wr, wi);
  HIPCHK(hipGetLastError(), "eig6 launch");
  HIPCHK(hipDeviceSynchronize(), "eig6 sync");
  return HYQ_OK;
}

int hyq_set_mlp(hyq_ctx* c, hyq_mlp* mlp) {
  if (!c) return fail(HYQ_EINVAL, "null argument");
  if (mlp && c->p.precision != HYQ_PREC_MIXED_LEARNED)
    return fail(HYQ_EINVAL, "a warm-start network needs precision HYQ_PREC_MIXED_LEARNED");
  c->mlp = mlp;
  return HYQ_OK;
}

int hyq_plane_dataset(const double* M, int64_t n, float* X, float* L, uint8_t* valid) {
  if (!M || !X || n < 0 || ((L == nullptr) != (valid == nullptr)))
    return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_plane_dataset, dim3(grid_for(n)), dim3(kBlock), 0, 0, M, (long long)n, X, L,
                     valid);
  HIPCHK(hipGetLastError(), "dataset launch");
  HIPCHK(hipDeviceSynchronize(), "dataset sync");
  return HYQ_OK;
}

int hyq_closure1d_batch(const double* m5, int64_t n, double* vmin, double* vmax) {
  if (!m5 || !vmin || !vmax || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_closure1d_batch, dim3(grid_for(n)), dim3(kBlock), 0, 0, m5, (long long)n,
                     vmin, vmax);
  HIPCHK(hipGetLastError(), "closure1d launch");
  HIPCHK(hipDeviceSynchronize(), "closure1d sync");
  return HYQ_OK;
}

int hyq_hll_lines(const double* M, const double* F, const double* vmin, const double* vmax,
                  int64_t nlines, int32_t np, double dt, double dx, double* Mout) {
  if (!M || !F || !vmin || !vmax || !Mout || nlines < 0 || np < 1 || !(dx > 0))
    return fail(HYQ_EINVAL, "bad argument");
  if (np >= kMaxUpdateCells) return fail(HYQ_EINVAL, "line longer than 2^29 - 1 cells");
  const long long n = (long long)nlines * np;
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_hll_lines, dim3(grid_for(n)), dim3(kBlock), 0, 0, M, F, vmin, vmax, n,
                     (int)np, dt / dx, Mout);
  HIPCHK(hipGetLastError(), "hll launch");
  HIPCHK(hipDeviceSynchronize(), "hll sync");
  return HYQ_OK;
}

int hyq_collision_batch(const double* M, int64_t n, double dt, double Kn, int32_t positivity,
                        double* Mout) {
  if (!M || !Mout || n < 0) return fail(HYQ_EINVAL, "bad argument");
  if (n == 0) return HYQ_OK;
  hipLaunchKernelGGL(k_collision_batch, dim3(grid_for(n)), dim3(kBlock), 0, 0, M, (long long)n, dt,
                     Kn, positivity, Mout);
  HIPCHK(hipGetLastError(), "collision launch");
  HIPCHK(hipDeviceSynchronize(), "collision sync");
  return HYQ_OK;
}

}  // extern "C"
