// Device code of the step's cell kernels, shared by the single run, the batches
// (hyq_kernels.hip) and the ensemble (hyq_ensemble_kernels.h).  A kernel takes a `Run` that says
// which cell a thread has and the parameters and step scalars of that cell's run.
//
// Pass 1 is project -> planes [-> solve] -> hard -> close, pass 2 project -> planes
// [-> solve] -> hard -> relax; the brackets are the fast modes' (EM = 1).
//   project  the realizability projection of every cell, to A
//   planes   the plane Jacobians of A: one wave per plane, one lane per cell
//   solve    the planes the fast solve left open: block test, then the QR
//   hard     the cells the others did not finish: eigenvalue corrections, z-path
//            clamp and re-projection
//   close    closure and fluxes of A, 1D speeds
//   relax    projection and BGK of A
// The one-kernel-per-pass form this replaces kept every path of a cell in one kernel: 0.6 to
// 1.1 MB of code against an instruction cache of 64 KB shared by two CUs, with 1 KB of
// scratch per lane.  These kernels are 8 to 109 KB each.  Those that project have 240 B of
// scratch for the realizability edge branch; the two-wave forms for long lists spill beyond
// that (k_hard 496 and 320 B, k_wide_close 272, k_wide_solve 448 with EM 1), the others do not.  Per step (pass 1 + pass 2, one kernel per pass -> this
// form): 20x20x10 FP64 389 + 267 -> 150 + 143 us; 37x29x17 mixed 468 + 274 -> 260 + 185;
// 120x120x60 FP64 1557 + 1082 -> 1336 + 964, learned 1830 -> 1306 in all.  What is left is the
// latency of the serial root iterations (at 1 to 4 waves a SIMD) and, on small grids, of one
// wave through each kernel.
#pragma once
#include <hip/hip_runtime.h>

#include "hyq_planes.h"

namespace hyq {

// Counters of one step, per pass: cells that left `planes` (entries, low word of nlist) and
// their open planes (items, high word: one atomic hands out both); then, for the fast
// modes' diagnostics, cells on the full path, cells with open planes only, those planes,
// and cells an open plane sent to the full path.
struct StepCounts {
  unsigned long long nlist[2];
  unsigned nhard[2], nslot[2], npend[2], ncplx[2];
};
HD void clear_counts(StepCounts* n) { *n = StepCounts{}; }

// The entries: cells with a plane that is open, complex or not finite, or a z path that
// clamps or re-projects.  They live in the flux buffer, which is free between projection and
// k_close (and in pass 2), so that no mode allocates for them.  cap: the plane stride.
struct Lists {
  double* v;       // [10][cap] the planes' extremes, v[2q], v[2q + 1]
  double* S;       // [35][cap] the state before a z re-projection
  int* cell;       // [cap]
  int* run;        // [cap] ensemble: the entry's run (else unused)
  uint32_t* info;  // [5][cap] what is known of each plane (plane_decide)
  uint32_t* item;  // [5 cap] open planes: 5 entry + q
};
constexpr size_t kListBytes = 10 * 8 + (1 + 1 + 5 + 5) * 4;  // per cell, without S
static_assert(35 * sizeof(double) + kListBytes <= 105 * sizeof(float), "the lists fit the FP32 fluxes");
// Lists for cap cells in F: S, then `skip` doubles the caller has other use for, the rest.
inline Lists carve_lists(void* F, long long cap, size_t skip = 0) {
  Lists L;
  L.S = static_cast<double*>(F);
  L.v = L.S + 35 * (size_t)cap + skip;
  L.cell = reinterpret_cast<int*>(L.v + 10 * (size_t)cap);
  L.run = L.cell + cap;
  L.info = reinterpret_cast<uint32_t*>(L.run + cap);
  L.item = L.info + 5 * (size_t)cap;
  return L;
}
constexpr uint32_t kEntryHard = 1u << 31;  // in info of plane 0: on the full path from the start
constexpr uint32_t kEntryOpen = 7u << 28;  // in info of plane 0: open planes it had
constexpr uint32_t kPlExtra = 0xFF00u;     // iterations of a fast solve that left the plane open
constexpr int kPlExtraShift = 8;

struct CellCtx {
  bool active, in;  // active: the same for the whole block
  long long c;
  int run;  // -1: there is one
  int flag2D, positivity;
  double Ma, Kn, dt;
  unsigned long long *vmax, *err;  // null: not wanted (batches)
};

// The wave maximum |vp| in two parts: the 6x6 speeds' where they are found (k_planes, k_hard),
// in FP64 before they are rounded to FT, and the 1D speeds' in k_close.  The maximum over both
// kinds is that over the combined speeds.  The single run's fast modes take the maximum of the
// combined speeds from the rounded 6x6 ones instead (Run::kRoundFast), all in k_close.
template <int EM, typename Run>
constexpr bool split_max() {
  return EM == 0 || !Run::kRoundFast;
}
__device__ __forceinline__ unsigned long long wave_max_u64(unsigned long long v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long w = __shfl_xor(v, o);
    v = w > v ? w : v;
  }
  return v;
}
// Raises *m to v.  The plain read first (it may be stale, but *m only grows) spares most of
// the atomics, which all meet on one address across the XCDs.
__device__ __forceinline__ void raise_max(unsigned long long* m, unsigned long long v) {
  if (v > __hip_atomic_load(m, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP)) atomicMax(m, v);
}
__device__ __forceinline__ unsigned long long abs_bits(double v) {
  return __double_as_longlong(fabs(v));  // |v| >= 0: bit order = value order; NaN sorts above +Inf
}

// The z path's clamp or re-projection (eigenvalues6z_hyperbolic_3D.jl:27-104) of a state
// whose density and second moments are m0 .. : 0 none, 1 clamp, 2 re-projection (bits).
HD int z_special(bool positivity, double m0, double m1, double m2, double m5, double m9, double m15,
                 double m19) {
  if (!positivity) return 0;
  int r = 0;
  if (m0 <= 0.0) {
    r = 1;
    m0 = jmax(m0, 1e-14);
  }
  if (m0 > 1e-15) {
    const double vx = m2 / m0 - (m1 / m0) * (m1 / m0);
    const double vy = m9 / m0 - (m5 / m0) * (m5 / m0);
    const double vz = m19 / m0 - (m15 / m0) * (m15 / m0);
    if (vx < 0.0 || vy < 0.0 || vz < 0.0) r |= 2;
  }
  return r;
}

// ---- planes: the plane Jacobians of every cell -----------------------------------------------
// Sorts out the cells of a wave after their planes (info in si, extremes in sv, per lane):
// those whose planes are all real write their speeds (pass 1; min and max over each
// direction's two planes), the others become entries.  zs: the z path clamps or re-projects.
template <int EM, int PASS, bool SPLITMAX, typename FT>
__device__ __forceinline__ void sort_out(const CellCtx& x, int lane, bool zs, const double (*sv)[64],
                                         const uint32_t (*si)[64], FT* __restrict__ vp,
                                         uint32_t* __restrict__ flags, const Lists& L,
                                         StepCounts* cnt, long long N) {
  constexpr int NP = PASS == 1 ? 5 : 4;
  uint32_t in[NP];
  bool real = !zs, full = zs, cplx = false;
  unsigned nopen = 0u;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    in[p] = si[p][lane];
    const uint32_t st = in[p] & kPlState;
    real = real && st == kPlReal;
    full = full || st == kPlComplex || st == kPlNotFinite;
    cplx = cplx || st == kPlComplex;
    nopen += st == kPlOpen ? 1u : 0u;
  }
  // (pass 2: a plane that is not finite takes no correction)
  const bool ent = x.in && !real && !(PASS == 2 && EM == 0 && !cplx);
  if (PASS == 1) {
    unsigned long long vb = 0;
    if (x.in && !ent) {
      double v[10], v6[6];
      uint32_t its = 0u;
#pragma unroll
      for (int p = 0; p < 5; ++p) {
        v[2 * p] = sv[2 * p][lane];
        v[2 * p + 1] = sv[2 * p + 1][lane];
        its += in[p] >> kPlIterShift;
      }
      combine_planes(v, v6);
#pragma unroll
      for (int d = 0; d < 6; ++d) {
        vp[(size_t)d * N + x.c] = (FT)v6[d];
        const unsigned long long b = abs_bits(v6[d]);
        vb = b > vb ? b : vb;
      }
      if (EM == 1) flags[x.c] = (flags[x.c] & 0xFFFFu) | ((its < 0xFFFu ? its : 0xFFFu) << 16);
    }
    if (SPLITMAX && x.vmax != nullptr) {
      vb = wave_max_u64(vb);
      if (lane == 0) raise_max(x.vmax, vb);
    }
  }
  const unsigned long long em = __ballot(ent);
  if (em == 0ull) return;
  const unsigned long long below = (1ull << lane) - 1ull;
  unsigned long long om[NP];
  unsigned nitem = 0u;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    om[p] = EM == 1 ? __ballot(ent && (in[p] & kPlState) == kPlOpen) : 0ull;
    nitem += (unsigned)__popcll(om[p]);
  }
  unsigned long long base = 0ull;
  if (lane == 0)
    base = atomicAdd(&cnt->nlist[PASS - 1],
                     (unsigned long long)__popcll(em) | ((unsigned long long)nitem << 32));
  const unsigned e0 = __builtin_amdgcn_readfirstlane((unsigned)base);
  unsigned i0 = __builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
  if (!ent) return;
  const unsigned e = e0 + (unsigned)__popcll(em & below);
  L.cell[e] = (int)x.c;
  if (x.run >= 0) L.run[e] = x.run;
#pragma unroll
  for (int p = 0; p < NP; ++p) {
    uint32_t f = in[p];
    if (EM == 1 && (f & kPlState) == kPlOpen) {
      L.item[i0 + (unsigned)__popcll(om[p] & below)] = 5u * e + (unsigned)p;
      f = ((f >> kPlIterShift) << kPlExtraShift) & kPlExtra;
    }
    if (p == 0) f |= (full ? kEntryHard : 0u) | (nopen << 28);
    L.info[(size_t)p * N + e] = f;
    i0 += (unsigned)__popcll(om[p]);
    if (PASS == 1) {
      L.v[(size_t)(2 * p) * N + e] = sv[2 * p][lane];
      L.v[(size_t)(2 * p + 1) * N + e] = sv[2 * p + 1][lane];
    }
  }
}

// Two shapes, with the same values.  One copy of the plane solve serves all planes, with a
// plane's 15 moments in registers instead of a cell's 35.
//   SPREAD: a block per 64 cells, wave q solves plane q (UV, UW, VU, VW, WU; pass 2 the
//     first four) of them from LDS, then wave 0 sorts out the cells.  For grids that do not
//     fill the chip: a cell's planes are solved side by side.
//   else: a wave per 64 cells solves its planes in turn.  For grids that do: no wave waits
//     for another (with five waves to a block the other form keeps 1.1 waves per SIMD of the
//     two that fit).
// EM 1: P the network's seeds, or null.
//
// kManyComplex: lanes.  8, 16 and 32 take the same time; 1: a 120x120x60 step on jets 3% more, 100000 jets
// cells as a batch 482 -> 512 us; never: 100000 mixture cells 1831 -> 2092 us, 1000000 11.8
// -> 13.1 ms.
constexpr int kManyComplex = 16;
template <int EM>
constexpr int kPlaneWaves = EM == 0 ? 2 : 4;  // waves per SIMD
template <bool SPREAD, int PASS>
constexpr int kPlaneThreads = SPREAD && PASS == 1 ? 320 : 256;
template <bool SPREAD, int EM, int PASS, typename FT, typename Run>
__global__ __launch_bounds__((kPlaneThreads<SPREAD, PASS>), kPlaneWaves<EM>) void k_planes(
    Run R, const double* __restrict__ A, FT* __restrict__ vp, uint32_t* __restrict__ flags,
    const float* __restrict__ P, Lists L, StepCounts* cnt, long long N, unsigned nblk) {
  constexpr int NP = PASS == 1 ? 5 : 4, kGroups = SPREAD ? 1 : 4;
  __shared__ double sm[SPREAD ? 35 : 1][64];
  __shared__ double sv[kGroups][PASS == 1 ? 10 : 1][64];
  __shared__ uint32_t si[kGroups][NP][64];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const unsigned blk = SPREAD ? blockIdx.x : blockIdx.x * 4u + (unsigned)w;
  if (blk >= nblk) return;  // not SPREAD: no barrier follows
  const CellCtx x = R.cell(blk, 64, lane);
  if (!x.active) return;
  if (SPREAD) {
    if (x.in)
      for (int t = w; t < 35; t += NP) sm[t][lane] = A[(size_t)t * N + x.c];
    __syncthreads();
  }
  const int g = SPREAD ? 0 : w;
  // a byte offset within a plane: the planes' bases are uniform, so a load needs one address
  // register (64-bit addresses, hoisted out of the loop over the planes, took 70 and spilled)
  const unsigned c8 = (unsigned)x.c * 8u;
  // EM 0, planes in turn: a cell with a complex pair in UV or UW is corrected before its other
  // planes count, so it leaves them open; where that is much of a wave, every cell does and
  // becomes an entry (k_hard solves open planes, one per lane).
  bool skip = false;
  uint32_t prev = kPlReal;
#pragma unroll 1
  for (int q = SPREAD ? w : 0; q < (SPREAD ? w + 1 : NP); ++q) {
    if (!SPREAD && EM == 0 && PASS == 1 && q == kVU) {
      skip = x.in && prev == kPlComplex;
      if (__popcll(__ballot(skip)) >= kManyComplex) skip = true;
    }
    unsigned o8 = c8;
    if (!SPREAD) asm volatile("" : "+v"(o8));  // keeps the addresses out of the loop's invariants
    uint32_t info = skip ? kPlOpen : kPlReal;
    if (x.in && !skip) {
      constexpr SetT T = plane_sets();
      double m[15];
      auto load = [&](const int* at) {
#pragma unroll
        for (int t = 0; t < 15; ++t)
          m[t] = SPREAD ? sm[SPREAD ? at[t] : 0][lane] : at_byte(A + (size_t)at[t] * N, o8);
      };
      switch (plane_set(q)) {
        case 0: load(T.m[0]); break;
        case 1: load(T.m[1]); break;
        default: load(T.m[2]);
      }
      float w0 = NAN, w1 = NAN;
      if (EM == 1 && PASS == 1 && P != nullptr) {
        const float2 s = reinterpret_cast<const float2*>(P)[(size_t)q * N + x.c];
        w0 = s.x;
        w1 = s.y;
      }
      double v0, v1;
      info = plane_decide<EM, false, PASS == 1>(plane_of_set(m, plane_swapped(q)), w0, w1, false, v0, v1);
      if (PASS == 1) {
        sv[g][2 * q][lane] = v0;
        sv[g][2 * q + 1][lane] = v1;
      }
    }
    if (!SPREAD && EM == 0 && PASS == 1 && (info & kPlState) == kPlComplex) prev = kPlComplex;
    si[g][q][lane] = info;
  }
  if (SPREAD) {
    __syncthreads();
    if (w != 0) return;
  }
  bool zs = false;
  if (PASS == 1 && x.in) {
    auto at = [&](int t) { return SPREAD ? sm[SPREAD ? t : 0][lane] : at_byte(A + (size_t)t * N, c8); };
    zs = z_special(x.positivity != 0, at(0), at(1), at(2), at(5), at(9), at(15), at(19)) != 0;
  }
  sort_out<EM, PASS, split_max<EM, Run>(), FT>(x, lane, zs, sv[g], si[g], vp, flags, L, cnt, N);
}

// The 15 moments of plane q (not the same on every lane) of cell c.
__device__ __forceinline__ void load_plane_set(const double* A, long long N, long long c, int q,
                                               double* m) {
  constexpr SetT T = plane_sets();
  const int s = plane_set(q);
#pragma unroll
  for (int t = 0; t < 15; ++t) {
    const int n = s == 0 ? T.m[0][t] : (s == 1 ? T.m[1][t] : T.m[2][t]);
    m[t] = A[(size_t)n * N + c];
  }
}

// Spread of a list of n entries over every wave of the grid: each wave takes `per`
// consecutive entries (per = ceil(n / waves), at most 64) on its first `per` lanes, and the
// grid strides by waves * per.  Few entries per wave keep the union of their branch paths,
// which a wave executes, short; these entries are the rare, branch-heavy ones.
struct ListSpread {
  unsigned n, per, wave, lane, stride;
  __device__ explicit ListSpread(unsigned n_) : n(n_) {
    const unsigned waves = gridDim.x * (blockDim.x / 64);
    per = (n + waves - 1) / waves;
    per = per < 1 ? 1 : (per > 64 ? 64 : per);
    wave = blockIdx.x * (blockDim.x / 64) + threadIdx.x / 64;
    lane = threadIdx.x & 63;
    stride = waves * per;
  }
  __device__ unsigned first() const { return wave * per + lane; }
  __device__ bool mine(unsigned i) const { return lane < per && i < n; }
};

// The open planes, one per lane: the fast solve with the 2x2 block test of a nearly double
// pair, the QR where that does not decide.
constexpr int kSolveWaves = 1;
constexpr unsigned kSolveBlocks = 256 * 4 * kSolveWaves / 2;
template <int PASS>
__global__ __launch_bounds__(128, kSolveWaves) void k_solve(const double* __restrict__ A,
                                                            const float* __restrict__ P, Lists L,
                                                            const StepCounts* cnt, long long N) {
  const ListSpread ls((unsigned)(cnt->nlist[PASS - 1] >> 32));
  for (unsigned i = ls.first(); i < ls.n; i += ls.stride) {
    if (!ls.mine(i)) continue;
    const unsigned it = L.item[i], e = it / 5u;
    const int q = (int)(it % 5u);
    const long long c = L.cell[e];
    float w0 = NAN, w1 = NAN;
    if (PASS == 1 && P != nullptr) {
      const float2 w = reinterpret_cast<const float2*>(P)[(size_t)q * N + c];
      w0 = w.x;
      w1 = w.y;
    }
    double m[15], v0, v1;
    load_plane_set(A, N, c, q, m);
    const uint32_t f =
        plane_decide<1, true, PASS == 1>(plane_of_set(m, plane_swapped(q)), w0, w1, false, v0, v1);
    const size_t at = (size_t)q * N + e;
    L.info[at] = (L.info[at] & (kPlExtra | kEntryHard | kEntryOpen)) | f;
    if (PASS == 1) {
      L.v[(size_t)(2 * q) * N + e] = v0;
      L.v[(size_t)(2 * q + 1) * N + e] = v1;
    }
  }
}

// ---- hard: the entries ------------------------------------------------------------------------
// Those whose planes turned out real write their speeds; the others go through the
// corrections of eig6_axis (x, y) and eig6_z in rounds: a correction changes the cell's state
// in A, and the planes the rest of the path needs are then solved again on it, one (entry,
// plane) per lane.  A cell whose axis needs no correction keeps its planes' decisions for the
// next (the state did not change), so most entries take one round: one closure and one plane
// solve, where solving each axis in turn took three solves and up to three closures one
// after the other.  The same functions on the same values as pass1_cell and pass2_cell, so
// the same bits.
//
// An entry's progress: the axis it is at, and what it waits for.
constexpr uint32_t kStAxis = 3u, kStFin = 16u, kStZChk = 32u, kStSpec = 64u, kStDone = 128u;
// A round's work for an entry: a closure (op: the planes to correct, or a plain
// re-projection; kFromS: of the state saved before the z clamp or re-projection), then the
// planes to solve (bit q), of which `last` for their values after the correction.
constexpr uint32_t kC01 = 1u, kC02 = 2u, kC12 = 4u, kFromS = 8u, kProj = 16u;
struct Work {
  uint32_t op, solve, last;
};
constexpr uint32_t kPlInfo = 0x0FFFFFFFu;  // info without the entry's bits

template <int PASS>
__device__ __forceinline__ EigRes entry_plane(const Lists& L, long long N, unsigned e, int q, bool fin) {
  return plane_result(L.info[(size_t)q * N + e], PASS == 1 ? L.v[(size_t)(2 * q) * N + e] : 0.0,
                      PASS == 1 ? L.v[(size_t)(2 * q + 1) * N + e] : 0.0, fin);
}

// EM 1, first of all: an entry that had open planes only, all of them real now, is finished
// as `planes` would have done.  Counts the diagnostics into stat[4] (may be null): on the full
// path from the start, open planes only, those planes, sent to the full path by one.
template <int PASS, typename FT>
__device__ __forceinline__ bool entry_real(unsigned e, long long c, FT* vp, uint32_t* flags, const Lists& L,
                                           long long N, unsigned long long* vmax, unsigned* stat) {
  const uint32_t i0 = L.info[e];
  if (i0 & kEntryHard) {
    if (stat) atomicAdd(&stat[0], 1u);
    return false;
  }
  if (stat) {
    atomicAdd(&stat[1], 1u);
    atomicAdd(&stat[2], (i0 & kEntryOpen) >> 28);
  }
  bool real = true;
  uint32_t f = PASS == 1 ? flags[c] & 0xFFFFu : 0u;
  double v[10], v6[6];
#pragma unroll
  for (int q = 0; q < (PASS == 1 ? 5 : 4); ++q) {
    const uint32_t i = L.info[(size_t)q * N + e];
    real = real && (i & kPlState) == kPlReal;
    f = plane_flags(f, (i & kPlInfo) + (((i & kPlExtra) >> kPlExtraShift) << kPlIterShift), false);
    if (PASS == 1) {
      v[2 * q] = L.v[(size_t)(2 * q) * N + e];
      v[2 * q + 1] = L.v[(size_t)(2 * q + 1) * N + e];
    }
  }
  if (!real) {
    if (stat) atomicAdd(&stat[3], 1u);
    return false;
  }
  if (PASS == 1) {
    combine_planes(v, v6);
    unsigned long long vb = 0;
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      vp[(size_t)d * N + c] = (FT)v6[d];
      const unsigned long long b = abs_bits(v6[d]);
      vb = b > vb ? b : vb;
    }
    flags[c] = f;
    if (vmax != nullptr) raise_max(vmax, vb);
  }
  return true;
}

// Takes entry e as far as it gets without new solves; returns the work it then waits for, or
// sets kStDone.  ahead: after a correction of x or y, WU is solved along with the planes
// that are needed in any case, a round less and often for nothing: for k_hard, whose rounds
// are latency (20000 mixture cells in the fast mode 1078 -> 895 us, 30000 1113 -> 850).
template <int EM, int PASS, typename FT, typename Run>
__device__ __forceinline__ Work advance(const Run& R, unsigned e, long long c, double* A, FT* vp,
                                        uint32_t* flags, const Lists& L, long long N, bool ahead,
                                        uint32_t& st, uint32_t& fl) {
  Work w{0u, 0u, 0u};
  auto info = [&](int q) { return L.info[(size_t)q * N + e] & kPlInfo; };
  auto is_open = [&](int q) { return (L.info[(size_t)q * N + e] & kPlState) == kPlOpen; };
  auto speeds = [&](int d, double lo, double hi) {  // direction d's extremes
    vp[(size_t)(2 * d) * N + c] = (FT)lo;
    vp[(size_t)(2 * d + 1) * N + c] = (FT)hi;
    unsigned long long* vmax = split_max<EM, Run>() ? R.entry(L, e).vmax : nullptr;
    if (vmax != nullptr) {
      const unsigned long long b0 = abs_bits(lo), b1 = abs_bits(hi);
      raise_max(vmax, b0 > b1 ? b0 : b1);
    }
  };
  while (!(st & kStDone) && !w.op && !w.solve) {
    const int ax = (int)(st & kStAxis);
    const bool fin = (st & kStFin) != 0u;
    if (ax < 2) {
      const int qa = ax == 0 ? kUV : kVU, qb = ax == 0 ? kUW : kVW;
      if (!fin && (is_open(qa) || is_open(qb))) {
        w.solve = (1u << qa) | (1u << qb);
        break;
      }
      if (PASS == 1) fl = plane_flags(plane_flags(fl, info(qa), fin), info(qb), fin);
      const EigRes ra = entry_plane<PASS>(L, N, e, qa, fin), rb = entry_plane<PASS>(L, N, e, qb, fin);
      if (!fin && (ra.cplx || rb.cplx)) {
        fl |= ax == 0 ? F_ECX : F_ECY;
        w.op = (ra.cplx ? kC01 : 0u) | (rb.cplx ? (ax == 0 ? kC02 : kC12) : 0u);
        if (PASS == 1) {
          w.last = (1u << qa) | (1u << qb);
          w.solve = w.last | (ax == 0 ? (1u << kVU) | (1u << kVW) : 0u);
          if (ahead) w.solve |= 1u << kWU;
          else L.info[(size_t)kWU * N + e] = kPlOpen;
          st |= kStFin;
        } else {  // only the corrections matter, not the speeds
          if (ax == 0) w.solve = (1u << kVU) | (1u << kVW);
          ++st;
        }
        break;
      }
      if (PASS == 1) {
        double lo, hi;
        combine_guarded(ra, rb, lo, hi);
        speeds(ax, lo, hi);
      }
      st = (st & ~kStFin) + 1u;
    } else if (PASS == 2) {
      st |= kStDone;
    } else if (!(st & kStZChk)) {
      st |= kStZChk;
      double m[7];
      const int at[7] = {0, 1, 2, 5, 9, 15, 19};
#pragma unroll
      for (int t = 0; t < 7; ++t) m[t] = A[(size_t)at[t] * N + c];
      const int z = z_special(R.entry(L, e).positivity != 0, m[0], m[1], m[2], m[3], m[4], m[5], m[6]);
      if (z) {
        st |= kStSpec;
        for (int t = 0; t < 35; ++t) L.S[(size_t)t * N + e] = A[(size_t)t * N + c];
        if (z & 1) {
          A[c] = jmax(m[0], 1e-14);
          fl |= F_RHO;
        }
        if (z & 2) {
          fl |= F_ZNEG;
          w.op = kProj | kFromS;
        }
        w.solve = (1u << kWU) | (1u << kVW);
      } else {
        w.solve = (is_open(kWU) ? 1u << kWU : 0u) | (is_open(kVW) ? 1u << kVW : 0u);
      }
    } else {
      fl = plane_flags(plane_flags(fl, info(kWU), fin), info(kVW), fin);
      const EigRes ra = entry_plane<PASS>(L, N, e, kWU, fin), rb = entry_plane<PASS>(L, N, e, kVW, fin);
      if (!fin && (!ra.ok || !rb.ok)) fl |= F_NONFIN;  // the reference's eigvals throws here
      if (!fin && (ra.cplx || rb.cplx)) {
        fl |= F_ECZ;
        w.op = (ra.cplx ? kC02 : 0u) | (rb.cplx ? kC12 : 0u) | ((st & kStSpec) ? kFromS : 0u);
        w.last = w.solve = (1u << kWU) | (1u << kVW);
        st |= kStFin;
        break;
      }
      speeds(2, jmin(ra.vmin, rb.vmin), jmax(ra.vmax, rb.vmax));
      flags[c] = fl;
      st |= kStDone;
    }
  }
  return w;
}

// The closure of a round for entry e: A becomes the corrected (or re-projected) state.
// Returns its flags.
__device__ __forceinline__ uint32_t apply_op(const CellCtx& x, uint32_t op, unsigned e, long long c,
                                             double* A, const Lists& L, long long N) {
  const double* src = (op & kFromS) ? L.S + e : A + c;
  double m[35], b[35];
#pragma unroll
  for (int t = 0; t < 35; ++t) m[t] = src[(size_t)t * N];
  if (!(op & kProj)) {  // axis_correct
    double cc[35], cn[35], M000, um, vm, wm;
    raw_to_central4(m, cc, M000, um, vm, wm);
#pragma unroll
    for (int t = 0; t < 35; ++t) cn[t] = cc[t];
    if (op & kC01) correct_plane<0, 1>(cc, cn);
    if (op & kC02) correct_plane<0, 2>(cc, cn);
    if (op & kC12) correct_plane<1, 2>(cc, cn);
    central_to_raw<4>(cn, M000, um, vm, wm);
    pack35(cn, m);
  }
  uint32_t f = 0u;
  flux_closure35<false, double>(m, x.flag2D, x.Ma, b, nullptr, nullptr, nullptr, 0, f);
#pragma unroll
  for (int t = 0; t < 35; ++t) A[(size_t)t * N + c] = b[t];
  return f;
}

// The solve of plane q of entry e on its current state.
template <int EM, int PASS>
__device__ __forceinline__ void solve_item(unsigned e, int q, bool fin, long long c, const double* A,
                                           const float* P, const Lists& L, long long N) {
  float w0 = NAN, w1 = NAN;
  if (EM == 1 && PASS == 1 && P != nullptr) {
    const float2 s = reinterpret_cast<const float2*>(P)[(size_t)q * N + c];
    w0 = s.x;
    w1 = s.y;
  }
  double m[15], v0, v1;
  load_plane_set(A, N, c, q, m);
  L.info[(size_t)q * N + e] = plane_decide<EM, true, PASS == 1>(plane_of_set(m, plane_swapped(q)), w0, w1,
                                                                fin, v0, v1);
  if (PASS == 1) {
    L.v[(size_t)(2 * q) * N + e] = v0;
    L.v[(size_t)(2 * q + 1) * N + e] = v1;
  }
}

// In one launch, for lists that are short or of unknown length (a step's): a block takes up
// to kHardThreads entries through all their rounds, with the rounds' lists in LDS.  One wave
// per SIMD (WAVES = 1): the time of a short list is the latency of one closure and one solve,
// which is shortest with the whole register file.  With EM 0 a list of more than
// kHardEntries, which would take several turns of that form, goes to one of two waves per
// SIMD (496 B of scratch): a step's first pass on mixtures, us for the step, one wave / two,
// 61x53x37 2627 / 2195, 120x120x60 15750 / 13360; 100000 mixture cells as a batch 2475 /
// 1965.  The length is known on the device only, so both are launched, each for its range
// [lo, hi); the idle one costs 3 us.  With EM 1 the second form needs 832 B of scratch and
// costs 12 us also when idle, 1.5% of a 120x120x60 step that has no such list.
constexpr int kHardThreads = 256;
constexpr unsigned kHardBlocks = 256;  // one per CU
constexpr unsigned kHardEntries = kHardBlocks * kHardThreads;
template <int EM, int PASS, int WAVES, typename FT, typename Run>
__global__ __launch_bounds__(kHardThreads, WAVES) void k_hard(Run R, double* A, FT* vp, uint32_t* flags,
                                                              const float* P, Lists L, StepCounts* cnt,
                                                              long long N, unsigned lo, unsigned hi) {
  const unsigned n = (unsigned)cnt->nlist[PASS - 1];
  if (n < lo || n >= hi) return;
  unsigned per = (n + gridDim.x - 1) / gridDim.x;
  per = per < 1 ? 1 : (per > kHardThreads ? kHardThreads : per);
  // s_item: final solves from the front, the others from the back
  __shared__ unsigned s_nop, s_nitem, s_nother, s_stat[4];
  __shared__ uint32_t s_op[kHardThreads], s_fl[kHardThreads], s_item[5 * kHardThreads];
  const unsigned tid = threadIdx.x;
  // work k of a round goes to lane k / waves of wave k % waves: short lists use every SIMD
  const unsigned slot = (tid & 63u) * (kHardThreads / 64) + (tid >> 6);
  constexpr uint32_t kFin = 1u << 16;  // s_item: 8 owner + plane; s_op: op << 16 | owner
  if (tid < 4) s_stat[tid] = 0u;
  __syncthreads();
  // An entry's context (R.entry) is read where it is used, not kept: the ensemble's holds
  // pointers of each lane's run, and kept through the rounds they were spilled under a
  // branch's execution mask, for some of the lanes only.
  for (unsigned first = blockIdx.x * per; first < n; first += gridDim.x * per) {
    const bool mine = tid < per && first + tid < n;
    const unsigned e = first + tid;
    const long long c = mine ? L.cell[e] : 0;
    uint32_t fl = PASS == 1 && mine ? flags[c] & 0xFFFFu : 0u;
    uint32_t st = mine ? 0u : kStDone;
    if (EM == 1 && mine &&
        entry_real<PASS, FT>(e, c, vp, flags, L, N, split_max<EM, Run>() ? R.entry(L, e).vmax : nullptr, s_stat))
      st = kStDone;
    if (tid == 0) s_nop = s_nitem = s_nother = 0u;
    __syncthreads();
    for (;;) {
      const Work w = advance<EM, PASS, FT, Run>(R, e, c, A, vp, flags, L, N, true, st, fl);
      if (w.op) {
        s_op[atomicAdd(&s_nop, 1u)] = tid | (w.op << 16);
        s_fl[tid] = 0u;
      }
      if (w.solve) {
        const uint32_t front = EM == 1 ? w.solve & w.last : w.solve, back = w.solve & ~front;
        unsigned at = front ? atomicAdd(&s_nitem, (unsigned)__popc(front)) : 0u;
        unsigned bt = back ? 5u * kHardThreads - 1u - atomicAdd(&s_nother, (unsigned)__popc(back)) : 0u;
#pragma unroll
        for (int q = 0; q < 5; ++q) {
          const uint32_t it = tid * 8u + (unsigned)q + ((w.last & (1u << q)) ? kFin : 0u);
          if (front & (1u << q)) s_item[at++] = it;
          if (back & (1u << q)) s_item[bt--] = it;
        }
      }
      __syncthreads();
      const unsigned nop = s_nop, nitem = s_nitem, nother = s_nother;
      if (nop + nitem + nother == 0u) break;  // the same on every thread
      if (slot < nop) {
        const unsigned o = s_op[slot] & 0xFFFFu, oe = first + o;
        s_fl[o] = apply_op(R.entry(L, oe), s_op[slot] >> 16, oe, L.cell[oe], A, L, N);
      }
      __syncthreads();
      // Item k: below nitem the front's, from sep on the back's.  EM 1: a final solve mostly
      // takes the QR and the others mostly do not, and a wave runs the paths of all its
      // lanes one after the other, so no wave gets both kinds (mixture cells, 30000 as a batch 893 ->
      // 845 us, 100000 1900 -> 1630; a 120x120x60 step on them 15240 -> 13720).
      unsigned k = slot, end = nitem + nother, sep = nitem;
      if (EM == 1 && nitem != 0u && nother != 0u) {
        if (nitem <= kHardThreads / 2 && nother <= kHardThreads / 2) {  // two waves each
          k = (tid & 63u) * 2u + ((tid >> 6) & 1u);
          if (tid < kHardThreads / 2) end = nitem;
          else k += nitem;
        } else {  // the back's from the next whole wave on
          sep = (nitem + 63u) & ~63u;
          k = tid;
          end = sep + nother;
        }
      }
      for (; k < end; k += kHardThreads) {
        if (k >= nitem && k < sep) continue;
        const uint32_t it = s_item[k < nitem ? k : 5u * kHardThreads - 1u - (k - sep)];
        const unsigned oe = first + ((it & 0xFFFFu) >> 3);
        solve_item<EM, PASS>(oe, (int)(it & 7u), (it & kFin) != 0u, L.cell[oe], A, P, L, N);
      }
      __syncthreads();
      if (w.op) fl |= s_fl[tid];
      if (tid == 0) s_nop = s_nitem = s_nother = 0u;
      __syncthreads();
    }
    __syncthreads();
  }
  if (EM == 1 && tid == 0) {
    if (s_stat[0] + s_stat[3]) atomicAdd(&cnt->nhard[PASS - 1], s_stat[0] + s_stat[3]);
    if (s_stat[1]) {
      atomicAdd(&cnt->nslot[PASS - 1], s_stat[1]);
      atomicAdd(&cnt->npend[PASS - 1], s_stat[2]);
      if (s_stat[3]) atomicAdd(&cnt->ncplx[PASS - 1], s_stat[3]);
    }
  }
}

// The same in a launch per phase, for a large batch whose entries may be most of its cells:
// each phase runs on a dense list over the whole chip, at the two waves per SIMD its own
// registers allow.  Pass 1 only.
struct WideLists {
  uint32_t *st, *fl;      // [cap] an entry's progress and flags
  uint32_t *ope, *opb;    // [cap] the round's closures: entry, op
  uint32_t* item;         // [5 cap] the round's solves: 5 entry + q, top bit: final
  unsigned long long* n;  // [kWideRounds] closures (low word) and solves (high) of each round
};
constexpr int kWideRounds = 4;  // x, y, the z re-projection or WU, z
constexpr size_t kWideBytes = (2 + 2 + 5) * 4;
template <int EM, typename Run>
__global__ __launch_bounds__(256) void k_wide_advance(Run R, int round, double* A, double* vp,
                                                      uint32_t* flags, Lists L, WideLists W,
                                                      const StepCounts* cnt, long long N) {
  const unsigned n = (unsigned)cnt->nlist[0];
  const int lane = threadIdx.x & 63;
  const unsigned long long below = (1ull << lane) - 1ull;
  // whole waves stay in the loop: the ballots below need every lane
  for (unsigned e0 = (blockIdx.x * 256u + threadIdx.x) & ~63u; e0 < n; e0 += gridDim.x * 256u) {
    const unsigned e = e0 + (unsigned)lane;
    const bool in = e < n;
    Work w{0u, 0u, 0u};
    if (in) {
      const long long c = L.cell[e];
      uint32_t st = round == 0 ? 0u : W.st[e], fl = round == 0 ? flags[c] & 0xFFFFu : W.fl[e];
      if (EM == 1 && round == 0 && entry_real<1, double>(e, c, vp, flags, L, N, R.entry(L, e).vmax, nullptr))
        st = kStDone;
      if (!(st & kStDone) || round == 0) {
        w = advance<EM, 1, double, Run>(R, e, c, A, vp, flags, L, N, false, st, fl);
        W.st[e] = st;
        W.fl[e] = fl;
      }
    }
    const unsigned long long om = __ballot(w.op != 0u);
    unsigned nitem = 0u;
    unsigned long long im[5];
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      im[q] = __ballot((w.solve >> q) & 1u);
      nitem += (unsigned)__popcll(im[q]);
    }
    if (nitem == 0u) continue;  // a closure always comes with solves
    unsigned long long base = 0ull;
    if (lane == 0)
      base = atomicAdd(&W.n[round], (unsigned long long)__popcll(om) | ((unsigned long long)nitem << 32));
    const unsigned o0 = __builtin_amdgcn_readfirstlane((unsigned)base);
    unsigned i0 = __builtin_amdgcn_readfirstlane((unsigned)(base >> 32));
    if (w.op) {
      const unsigned o = o0 + (unsigned)__popcll(om & below);
      W.ope[o] = e;
      W.opb[o] = w.op;
    }
#pragma unroll
    for (int q = 0; q < 5; ++q) {
      if ((w.solve >> q) & 1u)
        W.item[i0 + (unsigned)__popcll(im[q] & below)] =
            (5u * e + (unsigned)q) | (((w.last >> q) & 1u) << 31);
      i0 += (unsigned)__popcll(im[q]);
    }
  }
}
template <typename Run>
__global__ __launch_bounds__(128, 2) void k_wide_close(Run R, int round, double* A, Lists L, WideLists W,
                                                       long long N) {
  const unsigned n = (unsigned)W.n[round];
  for (unsigned k = blockIdx.x * 128u + threadIdx.x; k < n; k += gridDim.x * 128u) {
    const unsigned e = W.ope[k];
    W.fl[e] |= apply_op(R.entry(L, e), W.opb[k], e, L.cell[e], A, L, N);
  }
}
template <int EM>
__global__ __launch_bounds__(128, 2) void k_wide_solve(int round, const double* A, Lists L, WideLists W,
                                                       long long N) {
  const unsigned n = (unsigned)(W.n[round] >> 32);
  for (unsigned k = blockIdx.x * 128u + threadIdx.x; k < n; k += gridDim.x * 128u) {
    const uint32_t it = W.item[k], f = it & 0x7FFFFFFFu;
    solve_item<EM, 1>(f / 5u, (int)(f % 5u), (it >> 31) != 0u, L.cell[f / 5u], A, nullptr, L, N);
  }
}

// ---- the kernels of every cell ---------------------------------------------------------------
// The closure kernels need 310 to 400 registers: one wave per SIMD holds them without scratch.
constexpr int kProjWaves = 2, kCloseWaves = 1;

// The projection of every cell to A, and its flags (flags may be null).
template <int B, typename Run>
__global__ __launch_bounds__(B, kProjWaves) void k_project(Run R, const double* __restrict__ M,
                                                           double* __restrict__ A,
                                                           uint32_t* __restrict__ flags, long long N) {
  const CellCtx x = R.cell(blockIdx.x, B, threadIdx.x);
  if (!x.active || !x.in) return;
  double m[35], a[35];
#pragma unroll
  for (int t = 0; t < 35; ++t) m[t] = HYQ_LOAD_STREAM(&M[(size_t)t * N + x.c]);
  uint32_t fl = 0;
  pass1a_cell(m, x.flag2D, x.Ma, a, fl);
#pragma unroll
  for (int t = 0; t < 35; ++t) HYQ_STORE_STREAM(&A[(size_t)t * N + x.c], a[t]);
  if (flags != nullptr) flags[x.c] = fl;
}

// Pass 1's closure and fluxes of every cell, after the entries: A (the projected state, or a
// corrected one) to its closure Mr in place, the fluxes, the 1D speeds of Mr combined with
// the 6x6 speeds in vp (min and max commute with rounding to FT, so combining the rounded
// ones gives the same FT speeds), the flags (may be null), the wave maximum |vp| (its part of
// the 1D speeds, with split_max).
template <int B, int EM, typename FT, typename Run>
__global__ __launch_bounds__(B, kCloseWaves) void k_close(Run R, double* __restrict__ AMr,
                                                         FT* __restrict__ F, FT* __restrict__ vp,
                                                         uint32_t* __restrict__ flags, long long N) {
  const CellCtx x = R.cell(blockIdx.x, B, threadIdx.x);
  if (!x.active) return;
  unsigned long long vb = 0;
  if (x.in) {
    const long long c = x.c;
    double a[35], mr[35], s1[6], v6[6], vd[6];
#pragma unroll
    for (int t = 0; t < 35; ++t) a[t] = HYQ_LOAD_STREAM(&AMr[(size_t)t * N + c]);
    uint32_t fl = flags != nullptr ? flags[c] : 0u;
    flux_closure35<true, FT>(a, x.flag2D, x.Ma, mr, F + c, F + (size_t)35 * N + c,
                             F + (size_t)70 * N + c, (size_t)N, fl);
    closure1d_all(mr, s1);
#pragma unroll
    for (int d = 0; d < 6; ++d) v6[d] = (double)vp[(size_t)d * N + c];
    combine_vp(s1, v6, vd);
#pragma unroll
    for (int d = 0; d < 6; ++d) {
      vp[(size_t)d * N + c] = (FT)vd[d];
      const unsigned long long b = abs_bits(split_max<EM, Run>() ? s1[d] : vd[d]);
      vb = b > vb ? b : vb;
    }
#pragma unroll
    for (int t = 0; t < 35; ++t) HYQ_STORE_STREAM(&AMr[(size_t)t * N + c], mr[t]);
    if (flags != nullptr) flags[c] = fl;
    if ((fl & F_NONFIN) && x.err != nullptr) atomicOr(x.err, 1ull);
  }
  if (x.vmax != nullptr) {
    vb = wave_max_u64(vb);
    if ((threadIdx.x & 63) == 0) raise_max(x.vmax, vb);
  }
}

// Pass 2's projection and BGK of every cell, after the entries: A to M.
template <int B, bool MIXED, typename Run>
__global__ __launch_bounds__(B, kProjWaves) void k_relax(Run R, double* __restrict__ M,
                                                         const double* __restrict__ A, long long N) {
  const CellCtx x = R.cell(blockIdx.x, B, threadIdx.x);
  if (!x.active || !x.in) return;
  double a[35], o[35];
#pragma unroll
  for (int n = 0; n < 35; ++n) a[n] = A[(size_t)n * N + x.c];
  uint32_t fl = 0;
  pass2_relax<MIXED>(a, x.flag2D, x.Ma, x.positivity != 0, x.dt, x.Kn, o, fl);
#pragma unroll
  for (int n = 0; n < 35; ++n) M[(size_t)n * N + x.c] = o[n];
}

// Below so many blocks of 64 cells the planes of a cell are spread over waves.  The pass, in us,
// spread / in turn, by blocks:
//                  286          1025         1404         2052         4096        13500
//   FP64   pass 2  180 / 304    245 / 320    279 / 351    338 / 396    535 / 554   979 / 964
//   fast   pass 1  123 / 145    174 / 177    202 / 202    243 / 236    370 / 323
//          pass 2  112 / 119    122 / 130    133 / 138    169 / 171    233 / 228
// (Pass 1 spreads over five waves a block, of which fewer fit than of pass 2's four.)
// FP64 pass 1, from as many blocks as there are SIMDs on in turn, on jets at Ma 0.7 and 1.5 and as
// a batch of mixture cells:
//          708          927          1000         1051         1131         1214         1422
//   0.7    419 / 477    466 / 522    474 / 490    517 / 511    544 / 558    572 / 537    628 / 580
//   1.5    412 / 469    478 / 519    472 / 479    513 / 499    550 / 537    579 / 540    638 / 581
//   batch 1390 / 1240  1570 / 1345  1605 / 1370  1670 / 1405  1820 / 1715  2020 / 1728  2153 / 1736
template <int EM, int PASS>
constexpr unsigned kSpreadBelow = PASS == 1 ? (EM == 0 ? 1024 : 1280) : (EM == 0 ? 4096 : 2048);
// Launches of one pass after its projection (pass 1 up to k_hard, pass 2 up to k_hard).
template <int EM, int PASS, typename FT, typename Run>
void launch_planes(hipStream_t s, const Run& R, unsigned blocks64, double* A, FT* vp, uint32_t* flags,
                   const float* P, const Lists& L, StepCounts* cnt, long long N,
                   const WideLists* W = nullptr) {
  if (blocks64 < kSpreadBelow<EM, PASS>)
    hipLaunchKernelGGL((k_planes<true, EM, PASS, FT, Run>), dim3(blocks64),
                       dim3(kPlaneThreads<true, PASS>), 0, s, R, (const double*)A, vp, flags, P, L, cnt,
                       N, blocks64);
  else
    hipLaunchKernelGGL((k_planes<false, EM, PASS, FT, Run>), dim3((blocks64 + 3) / 4),
                       dim3(kPlaneThreads<false, PASS>), 0, s, R, (const double*)A, vp, flags, P, L,
                       cnt, N, blocks64);
  if (EM == 1)
    hipLaunchKernelGGL(k_solve<PASS>, dim3(kSolveBlocks), dim3(128), 0, s, (const double*)A, P, L,
                       (const StepCounts*)cnt, N);
  if (W == nullptr) {
    const bool both = EM == 0 && N > kHardEntries;
    hipLaunchKernelGGL((k_hard<EM, PASS, 1, FT, Run>), dim3(kHardBlocks), dim3(kHardThreads), 0, s, R, A,
                       vp, flags, P, L, cnt, N, 0u, both ? kHardEntries + 1u : ~0u);
    if constexpr (EM == 0)
      if (both)
        hipLaunchKernelGGL((k_hard<EM, PASS, 2, FT, Run>), dim3(2 * kHardBlocks), dim3(kHardThreads), 0, s,
                           R, A, vp, flags, P, L, cnt, N, kHardEntries + 1u, ~0u);
    return;
  }
  if constexpr (PASS == 1 && sizeof(FT) == 8 && Run::kWide)
    for (int r = 0; r <= kWideRounds; ++r) {
      hipLaunchKernelGGL((k_wide_advance<EM, Run>), dim3(1024), dim3(256), 0, s, R, r, A, vp, flags, L, *W,
                         (const StepCounts*)cnt, N);
      if (r == kWideRounds) break;
      hipLaunchKernelGGL(k_wide_close<Run>, dim3(1024), dim3(128), 0, s, R, r, A, L, *W, N);
      hipLaunchKernelGGL(k_wide_solve<EM>, dim3(1024), dim3(128), 0, s, r, (const double*)A, L, *W, N);
    }
}

}  // namespace hyq
