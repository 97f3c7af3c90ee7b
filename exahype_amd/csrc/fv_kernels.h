// Finite-volume kernels for gfx950: Godunov (2D/3D), MUSCL-Hancock (3D),
// Rusanov flux, FV CFL time step, ghost-layer filling of periodic patch grids.
//
// Device layout of a patch: structure of arrays over the patch including
// its ghost layers, [patch][v][cell], cell = (k*S + j)*S + i (3D) or j*S + i
// (2D), S = patch + 2*ghost.  Godunov is written in gather form: one thread
// per interior cell evaluates the Rusanov fluxes of its 2*DIM faces and
// applies them in the reference's order (x-, x+, y-, y+, z-, z+), so each
// cell's accumulation matches the reference's face loops
// (kernels/finitevolumes/godunov/c/{2d,3d}/godunov.cpph).  MUSCL-Hancock
// (kernels/finitevolumes/musclhancock/c/3d/musclhancock.cpph) forms every flux
// once and adds up a cell's fluxes in another order, before its state: a few
// roundings apart.
#pragma once
#include "common.h"
#include "pde_euler.h"

namespace exa {
namespace fv {

constexpr int V = 5;

struct PatchGeom {
  int P, G, S, dim;
  __host__ __device__ int ncells_box() const { return dim == 3 ? S * S * S : S * S; }
  __host__ __device__ int stride(int d) const { return d == 0 ? 1 : (d == 1 ? S : S * S); }
};

// rusanov<useNCP=false,useFlux=true>, kernels/finitevolumes/riemannsolvers/c/rusanov.cpph:24-156
template <class PDE>
__device__ inline double rusanov(const double* qL, const double* qR, int d, double gamma, double* f) {
  const double sL = PDE::max_abs_eigenvalue(qL, d, gamma);
  const double sR = PDE::max_abs_eigenvalue(qR, d, gamma);
  double s_max = -1.0;
  s_max = sL < s_max ? s_max : sL;
  s_max = sR < s_max ? s_max : sR;
  double FL[V], FR[V];
  PDE::flux_dir(qL, d, FL, gamma);
  PDE::flux_dir(qR, d, FR, gamma);
#pragma unroll
  for (int i = 0; i < V; ++i) {
    f[i] = 0.5 * s_max * (qL[i] - qR[i]);
    f[i] += 0.5 * (FL[i] + FR[i]);
  }
  return s_max;
}

__device__ inline void load_q(const double* base, int nbox, int cell, double* q) {
#pragma unroll
  for (int v = 0; v < V; ++v) q[v] = base[v * nbox + cell];
}

__device__ inline void interior_coords(const PatchGeom& g, int c, int& i, int& j, int& k) {
  i = c % g.P + g.G;
  j = (c / g.P) % g.P + g.G;
  k = g.dim == 3 ? c / (g.P * g.P) + g.G : 0;
}

__device__ inline int box_index(const PatchGeom& g, int i, int j, int k) {
  return g.dim == 3 ? (k * g.S + j) * g.S + i : j * g.S + i;
}

// Admissible time step of faces (or subcells) with wave speeds s: the smallest
// exa_dt_sane(cfl_h / s), with one division for the largest speed instead of
// one a face.
struct FaceSpeeds {
  double hi = 0.0;
  bool bad = false;
  // a face with wave speed s, if `face`
  __device__ inline void add(bool face, double s, double cfl_h) {
    hi = face && s > hi ? s : hi;
    if (face && !(s > 1.0e-290 && s <= 1.7976931348623157e308)) bad = bad || exa_dt_sane(cfl_h / s) == 0.0;
  }
  __device__ inline double candidate(double cfl_h) const {
    return bad ? 0.0 : (hi > 0.0 ? exa_dt_sane(cfl_h / hi) : 1.0e300);
  }
};

// Wave speeds of a state in every direction, for the CFL time step (as k_fv_stable_dt).
template <int DIM, class PDE>
__device__ inline void add_state(FaceSpeeds* speeds, bool subcell, const double* q, const double* cfl_h, double gamma) {
#pragma unroll
  for (int d = 0; d < DIM; ++d) speeds[d].add(subcell, PDE::max_abs_eigenvalue(q, d, gamma), cfl_h[d]);
}
template <int DIM>
__device__ inline double admissible(const FaceSpeeds* speeds, const double* cfl_h) {
  double dtm = 1.0e300;
#pragma unroll
  for (int d = 0; d < DIM; ++d) {
    const double cand = speeds[d].candidate(cfl_h[d]);
    dtm = cand < dtm ? cand : dtm;
  }
  return dtm;
}

// A grid's minimum over its workgroups, kept in SLOTS words a cache line apart:
// the workgroups that start together all find the word of a single minimum
// still high and each take their turn at it, 12 ns one after the other (81 x 81
// patches of 10^2, two minima: k_godunov 48.9 -> 45 us).
constexpr int MIN_SLOTS = 64, MIN_STRIDE = 16;
constexpr int MIN_WORDS = MIN_SLOTS * MIN_STRIDE;

// The workgroup's smallest value: as its patch's, and into the grid's slots.
__device__ inline void put_minimum(double v, double* red, double* dt_patch, unsigned long long* slots) {
  v = block_min(v, red);
  if (threadIdx.x == 0) {
    if (dt_patch) dt_patch[blockIdx.x] = v;
    if (slots) atomic_min_pos_double(slots + blockIdx.x % MIN_SLOTS * MIN_STRIDE, v);
  }
}

// One wave: the slots' minimum, and the slots cleared for the next step.
__device__ inline double take_minimum(unsigned long long* slots) {
  unsigned long long* w = slots + threadIdx.x % MIN_SLOTS * MIN_STRIDE;
  const double v = __longlong_as_double((long long)*w);
  *w = (unsigned long long)__double_as_longlong(1.0e300);
  return wave_min(v);
}

// Godunov update of patches p0 .. p0 + np - 1: luh_new(interior) = luh + flux
// differences, and the patch-boundary face updates of the first ghost layer by
// the subcells beside it, which have just formed those fluxes (the reference's
// face loops run over both patch-boundary faces of every line: -= at the lower
// ghost, += at the upper one).  Also the admissible dt of the face wave speeds,
// min CFL/DIM * h / s_max (godunov.cpph:33-143), as a global minimum or, one
// patch in one workgroup, in dt_patch; next_slots: the CFL time step of the new
// states too (null: not asked for), which are at hand here.
// One subcell a thread, the patches' subcells end to end: a 10^2 patch fills 39
// of 100 lanes of a workgroup of its own.  Bound by the latency of its loads;
// 81 x 81 patches of 10^2: 45 us, with a workgroup a patch, the ghost
// layers' fluxes formed again and a pass of its own for the time step 72.
template <int DIM, class PDE>
__global__ __launch_bounds__(256) void k_godunov(const double* __restrict__ luh, double* __restrict__ luh_new,
                                                 double* __restrict__ dt_patch, unsigned long long* adm_slots,
                                                 unsigned long long* next_slots, PatchGeom g, int p0, int np, double dx0,
                                                 double dx1, double dx2, const double* __restrict__ dtp, double gamma,
                                                 double cfl) {
  __shared__ double red[8];
  const double dt = *dtp;
  const int nbox = g.ncells_box();
  const double h[3] = {dx0 / g.P, dx1 / g.P, dx2 / g.P};
  const unsigned ninterior = DIM == 3 ? g.P * g.P * g.P : g.P * g.P;
  const double cfl_h[3] = {cfl / DIM * h[0], cfl / DIM * h[1], cfl / DIM * h[2]};
  FaceSpeeds speeds[DIM], next[DIM];
  for (unsigned it = blockIdx.x * blockDim.x + threadIdx.x; it < np * ninterior; it += gridDim.x * blockDim.x) {
    const double* u = luh + (size_t)(p0 + it / ninterior) * V * nbox;
    double* un = luh_new + (size_t)(p0 + it / ninterior) * V * nbox;
    int ijk[3];
    interior_coords(g, it % ninterior, ijk[0], ijk[1], ijk[2]);
    const int idx = box_index(g, ijk[0], ijk[1], ijk[2]);
    double q[V], acc[V], qn[V], f[V];
    load_q(u, nbox, idx, q);
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = q[v];
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const double fac = dt / h[d];
      const int o = g.stride(d);
      load_q(u, nbox, idx - o, qn);
      speeds[d].add(true, rusanov<PDE>(qn, q, d, gamma, f), cfl_h[d]);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] += fac * f[v];
      if (ijk[d] == g.G)
#pragma unroll
        for (int v = 0; v < V; ++v) un[v * nbox + idx - o] = un[v * nbox + idx - o] - fac * f[v];
      load_q(u, nbox, idx + o, qn);
      speeds[d].add(true, rusanov<PDE>(q, qn, d, gamma, f), cfl_h[d]);
#pragma unroll
      for (int v = 0; v < V; ++v) acc[v] -= fac * f[v];
      if (ijk[d] == g.G + g.P - 1)
#pragma unroll
        for (int v = 0; v < V; ++v) un[v * nbox + idx + o] = un[v * nbox + idx + o] + fac * f[v];
    }
#pragma unroll
    for (int v = 0; v < V; ++v) un[v * nbox + idx] = acc[v];
    if (next_slots) add_state<DIM, PDE>(next, true, acc, cfl_h, gamma);
  }
  put_minimum(admissible<DIM>(speeds, cfl_h), red, dt_patch, adm_slots);
  if (next_slots) put_minimum(admissible<DIM>(next, cfl_h), red, nullptr, next_slots);
}

__device__ inline double minmod(double a, double b) {
  const double m = fabs(a) < fabs(b) ? a : b;
  return a * b < 0.0 ? 0.0 : m;
}

// A value is formed here, and not at its first use.
__device__ inline void fv_pin(double& x) { asm volatile("" : "+v"(x)); }

// The same value in every lane, held in scalar registers.
__device__ inline double wave_uniform(double x) {
  const long long b = __double_as_longlong(x);
  const unsigned lo = __builtin_amdgcn_readfirstlane((int)b), hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
  return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// MUSCL-Hancock (kernels/finitevolumes/musclhancock/c/3d/musclhancock.cpph:
// 27-309), one workgroup per patch, which walks along z.  A thread owns a
// column (x, y) of the interior or of the first ghost layer beside it and per
// plane
//   -  forms its slopes, the half-step evolution (:62-213; ghosts keep their
//      unevolved states) and its six face states, once;
//   -  exchanges the lower x and y states through the LDS, forms the fluxes of
//      its upper x and y faces, exchanges those; the z states and fluxes stay
//      with it from plane to plane (:215-281).
// The first ghost layer receives the patch-boundary face updates as in the
// reference.  The planes above are loaded while a plane is worked on.
//
// Bound by vector FP64 (the ALUs are busy for 77 % of a launch at 11^3): 1155
// instructions a plane and wave (15 divisions, 6 square roots), two barriers
// between at most five waves.  36 KB of LDS at 11^3 let four workgroups share a compute unit, and
// cover each other's waits, if 168 registers hold a thread: values that wait
// longest stay in the LDS or are loaded again, since a spilled register's
// reload also waits for every load in flight (24 spills: 344 us; 2 are left).
// 12 x 13 x 14 patches of 11^3: 232 us, 254 with the new states' time step (a
// pass of its own: 41).  Forming the states of each subcell
// and face where they are used, every state four times: 527; one thread per
// two subcells, a patch's states in the LDS at once, one workgroup per compute
// unit: 400.
template <int PC>
struct MusclForm {
  static constexpr int S = PC + 4, T = PC + 2;
  static constexpr int NT = round_up64(T * T);
  static constexpr size_t LDS = sizeof(double) * V * (S * S + 4 * T * T);
};

// One patch: u (with its ghost layers) -> un (interior and the first ghost
// layer's face updates); sm: MusclForm<PC>::LDS bytes.  Returns the thread's
// part of the admissible time step; NEXT: adds the new states' speeds to next[3].
template <class PDE, int PC, bool NEXT>
__device__ __forceinline__ double muscl_patch(const double* __restrict__ u, double* __restrict__ un, double* sm,
                                              double dx0, double dx1, double dx2, double dt, double gamma,
                                              double cfl, FaceSpeeds* next = nullptr, const double* next_h = nullptr) {
  constexpr int S = PC + 4, T = PC + 2, PL = S * S, nbox = S * PL, TT = T * T;
  const double h[3] = {dx0 / PC, dx1 / PC, dx2 / PC};
  const double fac[3] = {wave_uniform(dt / h[0]), wave_uniform(dt / h[1]), wave_uniform(dt / h[2])};
  const double cfl_h[3] = {wave_uniform(cfl / 3 * h[0]), wave_uniform(cfl / 3 * h[1]), wave_uniform(cfl / 3 * h[2])};
  double* sP = sm;            // [v][y][x]: the plane
  double* sS = sP + V * PL;   // [d][v][column]: lower face states
  double* sF = sS + 2 * V * TT;  // [d][v][column]: fluxes of the upper faces
  // threads beyond the columns repeat column 0, a corner: same values, same places
  const unsigned t = threadIdx.x < TT ? threadIdx.x : 0;
  const bool column = threadIdx.x < TT;
  const unsigned x = t % T + 1, y = t / T + 1, col = y * S + x;
  const bool ix = column && x > 1 && x < PC + 2, iy = column && y > 1 && y < PC + 2;
  const bool inner = ix && iy, kept = ix || iy;  // not the four corners
  const bool up0 = iy && x < PC + 2, up1 = ix && y < PC + 2;  // a face above
  // the columns beside this one; where there is no face, any column that has
  // none above it (its flux is zero)
  const bool lo0 = iy && x > 1, lo1 = ix && y > 1;
  auto above = [&](unsigned t, int d) { return d == 0 ? (up0 ? t + 1 : t) : (up1 ? t + T : t); };
  auto below = [&](unsigned t, int d) { return d == 0 ? (lo0 ? t - 1 : 0) : (lo1 ? t - T : 0); };
  // the column again, so that the places derived from it are formed where they
  // are used: a spilled one's reload waits for every load in flight
  auto here = [&] {
    unsigned c = t;
    asm volatile("" : "+v"(c));
    return c;
  };
  // the second ghost layer beside the faces: one node of the plane a thread
  const bool rim = threadIdx.x < 4 * PC;
  const unsigned side = threadIdx.x / PC, k = threadIdx.x % PC + 2;
  const unsigned rc = !rim ? 0 : (side < 2 ? k * S + (side ? S - 1 : 0) : (side == 3 ? S - 1 : 0) * S + k);

  double qm[V], q[V], qp[V], wz[V], acc[V], r[V];
  // node c of plane z: uniform bases and one 32-bit lane offset, formed in place
  // (left alone, the loop keeps a pointer per array and variable in registers)
  auto offset = [](unsigned z, unsigned c) {
    unsigned o = 8 * (z * PL + c);
    asm volatile("" : "+v"(o));
    return o;
  };
  auto load_node = [&](const double* a, unsigned z, unsigned c, double* w) {
    const unsigned o = offset(z, c);
#pragma unroll
    for (int v = 0; v < V; ++v)
      w[v] = *reinterpret_cast<const double*>(reinterpret_cast<const char*>(a + v * nbox) + o);
  };
  auto store_node = [&](unsigned z, const double* w) {
    const unsigned o = offset(z, col);
#pragma unroll
    for (int v = 0; v < V; ++v) *reinterpret_cast<double*>(reinterpret_cast<char*>(un + v * nbox) + o) = w[v];
  };
  auto put_plane = [&](const double* own) {
#pragma unroll
    for (int v = 0; v < V; ++v) sP[v * PL + col] = own[v];
#pragma unroll
    for (int v = 0; v < V; ++v) sP[v * PL + rc] = r[v];
  };
  FaceSpeeds speeds[3];
  // the upper face of the plane below, whose update it completes
  auto z_face = [&](const double* w, double* f) {
    speeds[2].add(inner, rusanov<PDE>(wz, w, 2, gamma, f), cfl_h[2]);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      f[v] = inner ? fac[2] * f[v] : 0.0;
      acc[v] -= f[v];
    }
  };
  load_node(u, 0, col, r);
  load_node(u, 1, col, qm);
  load_node(u, 2, col, q);
  load_node(u, 3, col, qp);
  load_node(un, 1, col, acc);
#pragma unroll
  for (int v = 0; v < V; ++v) wz[v] = qm[v] + 0.5 * minmod(q[v] - qm[v], qm[v] - r[v]);
  // between the planes the sum and the upper z state wait in this thread's own
  // places of sS, free until the lower states are written there: 20 registers
  // less where most are in use, which is what lets three waves a SIMD run
  auto park = [&] {
    const unsigned t = here();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      sS[v * TT + t] = acc[v];
      sS[(V + v) * TT + t] = wz[v];
    }
    asm volatile("" ::: "memory");  // not kept in registers all the same
  };
  auto unpark = [&] {
    const unsigned t = here();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      acc[v] = sS[v * TT + t];
      wz[v] = sS[(V + v) * TT + t];
    }
  };
  load_node(u, 2, rc, r);
  put_plane(q);
  park();
  __syncthreads();
#pragma unroll 1
  for (int z = 2; z < PC + 2; ++z) {
    double e[V], hs[3][V], f[V], w[V];
#pragma unroll
    for (int v = 0; v < V; ++v) e[v] = 0.0;
#pragma unroll
    for (int i = 0; i < 3; ++i) {
      const int d = (i + 2) % 3, o = d == 0 ? 1 : S;
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const double a = d == 2 ? qm[v] : sP[v * PL + col - o], b = d == 2 ? qp[v] : sP[v * PL + col + o];
        hs[d][v] = 0.5 * minmod(b - q[v], q[v] - a);
        w[v] = q[v] - hs[d][v];
      }
      PDE::flux_dir(w, d, f, gamma);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        e[v] += 0.5 * fac[d] * f[v];
        w[v] = q[v] + hs[d][v];
        fv_pin(e[v]);
      }
      PDE::flux_dir(w, d, f, gamma);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        e[v] -= 0.5 * fac[d] * f[v];
        fv_pin(e[v]);
      }
    }
    unpark();
    const unsigned c = here();
#pragma unroll
    for (int v = 0; v < V; ++v) {
      e[v] = inner ? q[v] + e[v] : q[v];  // evolved centre
      sS[v * TT + c] = e[v] - hs[0][v];
      sS[(V + v) * TT + c] = e[v] - hs[1][v];
      w[v] = e[v] - hs[2][v];
#pragma unroll
      for (int d = 0; d < 3; ++d) {
        hs[d][v] = e[v] + hs[d][v];  // upper face states
        fv_pin(hs[d][v]);
      }
    }
    z_face(w, f);
    if (z > 2 ? kept : inner) store_node(z - 1, acc);
    if (NEXT) add_state<3, PDE>(next, inner && z > 2, acc, next_h, gamma);
#pragma unroll
    for (int v = 0; v < V; ++v) wz[v] = hs[2][v];
    __builtin_amdgcn_sched_barrier(0);
    // used at the end of the plane only: what a ghost's update is added to, and
    // the planes above (the next one's values again: not kept through the slopes)
    double old[V], qn[V];
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] = f[v];
    load_node(un, z, inner ? 0 : col, old);
    load_node(u, z + 1, rc, r);
    load_node(u, z + 1, col, qp);
    load_node(u, z + 2, col, qn);
    __syncthreads();
#pragma unroll
    for (int d = 0; d < 2; ++d) {
      const bool face = d == 0 ? up0 : up1;
#pragma unroll
      for (int v = 0; v < V; ++v) w[v] = sS[(d * V + v) * TT + above(c, d)];
      speeds[d].add(face, rusanov<PDE>(hs[d], w, d, gamma, f), cfl_h[d]);
#pragma unroll
      for (int v = 0; v < V; ++v) {
        f[v] = face ? fac[d] * f[v] : 0.0;
        acc[v] -= f[v];
        sF[(d * V + v) * TT + c] = f[v];
        fv_pin(acc[v]);
      }
    }
    put_plane(qp);
    __syncthreads();
    const unsigned b0 = below(c, 0), b1 = below(c, 1);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      acc[v] += sF[v * TT + b0];
      acc[v] += sF[(V + v) * TT + b1];
      acc[v] += inner ? q[v] : old[v];
      qm[v] = q[v];
      q[v] = qp[v];
      qp[v] = qn[v];
    }
    park();
  }
  unpark();
  double f[V], w[V];
#pragma unroll
  for (int v = 0; v < V; ++v) w[v] = q[v] - 0.5 * minmod(qp[v] - q[v], q[v] - qm[v]);
  z_face(w, f);
  if (kept) store_node(PC + 1, acc);
  if (NEXT) add_state<3, PDE>(next, inner, acc, next_h, gamma);
  if (inner) {
    load_node(un, PC + 2, col, acc);
#pragma unroll
    for (int v = 0; v < V; ++v) acc[v] += f[v];
    store_node(PC + 2, acc);
  }
  return admissible<3>(speeds, cfl_h);
}

// next_slots: the CFL time step (factor next_cfl) of the new states, or null.
template <class PDE, int PC>
__global__ __launch_bounds__(MusclForm<PC>::NT) __attribute__((amdgpu_waves_per_eu(3))) void k_muscl(
    const double* __restrict__ luh, double* __restrict__ luh_new, double* __restrict__ dt_patch,
    unsigned long long* adm_slots, unsigned long long* next_slots, double dx0, double dx1, double dx2,
    const double* __restrict__ dtp, double gamma, double cfl, double next_cfl) {
  extern __shared__ double sm[];
  __shared__ double red[8];
  constexpr int nbox = (PC + 4) * (PC + 4) * (PC + 4);
  const double next_h[3] = {wave_uniform(next_cfl / 3 * (dx0 / PC)), wave_uniform(next_cfl / 3 * (dx1 / PC)),
                            wave_uniform(next_cfl / 3 * (dx2 / PC))};
  FaceSpeeds next[3];
  const double dtm =
      muscl_patch<PDE, PC, true>(luh + (size_t)blockIdx.x * V * nbox, luh_new + (size_t)blockIdx.x * V * nbox, sm, dx0,
                                 dx1, dx2, *dtp, gamma, cfl, next, next_h);
  put_minimum(dtm, red, dt_patch, adm_slots);
  if (next_slots) put_minimum(admissible<3>(next, next_h), red, nullptr, next_slots);
}

// FV CFL time step of every patch (commons.cpph:26-67 2D, :410-463 3D).
template <int DIM, class PDE>
__global__ __launch_bounds__(256) void k_fv_stable_dt(const double* __restrict__ luh, double* __restrict__ dt_patch,
                                                      unsigned long long* dt_min, PatchGeom g, double dx0,
                                                      double dx1, double dx2, double gamma, double cfl) {
  __shared__ double red[8];
  const int nbox = g.ncells_box();
  const double* u = luh + (size_t)blockIdx.x * V * nbox;
  const double dxs[3] = {dx0, dx1, dx2};
  const int ninterior = DIM == 3 ? g.P * g.P * g.P : g.P * g.P;
  double dtm = 1.0e300;
  for (int c = threadIdx.x; c < ninterior; c += blockDim.x) {
    int i, j, k;
    interior_coords(g, c, i, j, k);
    double q[V];
    load_q(u, nbox, box_index(g, i, j, k), q);
#pragma unroll
    for (int d = 0; d < DIM; ++d) {
      const double s = PDE::max_abs_eigenvalue(q, d, gamma);
      const double cand = exa_dt_sane(cfl / DIM * (dxs[d] / g.P) / s);
      dtm = cand < dtm ? cand : dtm;
    }
  }
  dtm = block_min(dtm, red);
  if (threadIdx.x == 0) {
    if (dt_patch) dt_patch[blockIdx.x] = dtm;
    if (dt_min) atomic_min_pos_double(dt_min, dtm);
  }
}

// ---------------------------------------------------------------------------
// Boundary hooks of a patch (commons.cpph 2D :99-403, 3D :503-982).  Face
// blocks hold (layer k, slower transverse a, faster transverse b): 3D
// idx_bnd_x(P,P,G), idx_bnd_y(P,G,P), idx_bnd_z(G,P,P); 2D idx_bnd_x(P,G),
// idx_bnd_y(G,P).
__host__ __device__ inline int fv_bnd(int dim, int d, int P, int G, int k, int a, int b) {
  if (dim == 2) return d == 0 ? b * G + k : k * P + b;
  if (d == 0) return (a * P + b) * G + k;
  if (d == 1) return (a * G + k) * P + b;
  return (k * P + a) * P + b;
}

// the transverse axes of direction d: o1 faster, o2 slower (2 = none in 2D)
__host__ __device__ inline void fv_axes(int dim, int d, int& o1, int& o2) {
  o1 = dim == 2 ? 1 - d : (d == 0 ? 1 : 0);
  o2 = dim == 2 ? 2 : (d == 2 ? 1 : 2);
}

// Layer of the patch that boundaryLayerExtraction puts at layer k of the
// face block (side 1: patchEnd-G+k; side 0: patchBegin+k, but the 3D y and
// z faces read patchBegin for every k, commons.cpph:561, :591).
__host__ __device__ inline int fv_extract_layer(int dim, int d, int side, int P, int G, int k) {
  return side ? P + k : (dim == 3 && d > 0 ? G : G + k);
}

// boundaryValues of the Euler FV solvers at an outside subcell centre:
// outflow copies, a reflecting wall negates the normal momentum, exact data
// give the state of bc.exact at (x, t).
__device__ inline void fv_boundary_values(const exa_bc& bc, const double x[3], double t, int d, double gamma,
                                          const double (&qin)[V], double (&qout)[V]) {
  if (bc.kind == EXA_BC_EXACT) {
    exa_ic_point(bc.exact, gamma, x, t, qout);
    return;
  }
#pragma unroll
  for (int v = 0; v < V; ++v) qout[v] = qin[v];
  if (bc.kind == EXA_BC_REFLECTING) qout[1 + d] = -qin[1 + d];
}

// The outside subcell centre of boundaryConditions for layer k (0 the
// outermost) at transverse (a, b) of face (d, side) of a cell.
__device__ inline void fv_outside_centre(int dim, int d, int side, int P, int G, int k, int a, int b,
                                         const double c[3], const double h[3], double x[3]) {
  int o1, o2;
  fv_axes(dim, d, o1, o2);
  const int K = G - k - 1;  // mirror
  x[0] = x[1] = x[2] = 0.0;
  x[d] = side ? c[d] + 0.5 * h[d] * (1.0 + k * 1.0 / (2.0 * P)) : c[d] - 0.5 * h[d] * (1.0 + K * 1.0 / (2.0 * P));
  const double qa = (2.0 * a + 1.0) / (2.0 * P), qb = (2.0 * b + 1.0) / (2.0 * P);
  if (dim == 3) x[o2] = c[o2] + h[o2] * (qa - 0.5);
  // the 3D x+ face scales its y coordinate by size[2] (commons.cpph:780)
  x[o1] = c[o1] + h[(dim == 3 && d == 0 && side) ? 2 : o1] * (qb - 0.5);
}

// Domain boundaries of a grid: the boundary values, the cell geometry of
// every patch and the device-held time stamp of the step.
struct FvBoundary {
  exa_bc bc;
  double off[3], h[3];
  int nx, ny;
  const double* time;
  double gamma;
};

// Layer kk and transverse place t of a face's item; on the x faces the layers
// come first: they lie beside each other in memory.
__device__ inline void fv_ghost_place(const PatchGeom& g, int trans, int d, int r, int& kk, int& t) {
  kk = d == 0 ? r % g.G : r / trans;
  t = d == 0 ? r / g.G : r % trans;
}

// Face ghost layers of patches p0 .. p0 + np - 1 from the neighbours' interiors
// (ghostLayerFilling, commons.cpph:337-402, :876-982).  nbr[(2*d + side)*npatch
// + p]: neighbour of patch p on side (0: -, 1: +) of direction d, < 0 where a
// closed axis leaves none.
// The patches' places end to end, B of them a thread with all their loads in
// flight before the first store.  Bound by memory lines in 3D: the x layers
// touch most lines of a patch and of its x neighbours for two values each
// (12 x 13 x 14 patches of 11^3: 119 us, 840 MB of lines), by launch and
// latency in 2D (81 x 81 patches of 10^2: 19 us).
template <int DIM>
__global__ __launch_bounds__(256) void k_fv_ghosts(double* __restrict__ luh, const int* __restrict__ nbr, PatchGeom g,
                                                   int npatch, int p0, int np) {
  constexpr int B = DIM == 3 ? 4 : 1;
  const int nbox = g.ncells_box();
  const int trans = DIM == 3 ? g.P * g.P : g.P;
  const unsigned per_side = g.G * trans, total = 2 * DIM * per_side;
  double w[B][V];
  double* dst[B];
#pragma unroll
  for (int b = 0; b < B; ++b) {
    const unsigned it = (blockIdx.x * B + b) * 256 + threadIdx.x, i = it < np * total ? it : 0;
    const int p = p0 + i / total, ds = i % total / per_side, d = ds / 2, side = ds % 2;
    int kk, t, o1, o2, c[3];
    fv_ghost_place(g, trans, d, i % per_side, kk, t);
    fv_axes(DIM, d, o1, o2);
    c[o1] = t % g.P + g.G;
    c[o2] = DIM == 3 ? t / g.P + g.G : 0;
    c[d] = side ? g.G + g.P + kk : kk;
    const int q = nbr[ds * npatch + p];
    dst[b] = it < np * total && q >= 0 ? luh + (size_t)p * V * nbox + box_index(g, c[0], c[1], c[2]) : nullptr;
    c[d] = side ? g.G + kk : g.P + kk;
    load_q(luh + (size_t)(q >= 0 ? q : p) * V * nbox, nbox, box_index(g, c[0], c[1], c[2]), w[b]);
  }
#pragma unroll
  for (int b = 0; b < B; ++b)
    if (dst[b]) {
#pragma unroll
      for (int v = 0; v < V; ++v) dst[b][v * nbox] = w[b][v];
    }
}

// Those without a neighbour, as mergeWithBoundaryData fills them
// (E/solvers/FiniteVolumesSolver.cpp:689-728): the mirrored layer of the
// boundary-layer extraction through boundaryValues.  One workgroup per patch,
// launched where an axis is closed; kept apart because the analytical boundary
// values take 157 registers in 2D and 168 in 3D (the copy alone 22 and 58).
template <int DIM>
__global__ __launch_bounds__(256) void k_fv_boundary(double* __restrict__ luh, const int* __restrict__ nbr,
                                                     PatchGeom g, int npatch, FvBoundary fb) {
  const int p = blockIdx.x;
  const int nbox = g.ncells_box();
  const int trans = DIM == 3 ? g.P * g.P : g.P;
  double* me = luh + (size_t)p * V * nbox;
  for (int ds = 0; ds < 2 * DIM; ++ds) {
    if (nbr[ds * npatch + p] >= 0) continue;
    const int d = ds / 2, side = ds % 2;
    for (int r = threadIdx.x; r < g.G * trans; r += blockDim.x) {
      int kk, t, o1, o2, ci[3], ni[3];
      fv_ghost_place(g, trans, d, r, kk, t);
      const int ta = DIM == 3 ? t / g.P : 0, tb = t % g.P;  // transverse interior indices
      fv_axes(DIM, d, o1, o2);
      ci[o1] = ni[o1] = tb + g.G;
      ci[o2] = ni[o2] = DIM == 3 ? ta + g.G : 0;
      ci[d] = side ? g.G + g.P + kk : kk;
      const int K = g.G - kk - 1;
      ni[d] = fv_extract_layer(DIM, d, side, g.P, g.G, K);
      const int px = p % fb.nx, py = (p / fb.nx) % fb.ny, pz = p / (fb.nx * fb.ny);
      const double c[3] = {fb.off[0] + (px + 0.5) * fb.h[0], fb.off[1] + (py + 0.5) * fb.h[1],
                           DIM == 3 ? fb.off[2] + (pz + 0.5) * fb.h[2] : 0.0};
      double x[3], qin[V], qout[V];
      fv_outside_centre(DIM, d, side, g.P, g.G, kk, ta, tb, c, fb.h, x);
      load_q(me, nbox, box_index(g, ni[0], ni[1], ni[2]), qin);
      fv_boundary_values(fb.bc, x, *fb.time, d, fb.gamma, qin, qout);
      const int cidx = box_index(g, ci[0], ci[1], ci[2]);
#pragma unroll
      for (int v = 0; v < V; ++v) me[v * nbox + cidx] = qout[v];
    }
  }
}

// The per-patch hooks on one patch in the reference layout (node-major,
// nd values per subcell), one thread per (layer, transverse) entry:
// op 0 boundaryLayerExtraction (dst = luhbnd, src = luh), 1
// ghostLayerFillingAtBoundary (dst = luh, src = luhbnd), 2 ghostLayerFilling
// (dst = luh, src = the neighbour's luh), 3 boundaryConditions (dst =
// stateOut, src = stateIn; face d, side given by faceIndex).
struct FvHookArgs {
  int op, dim, d, side, P, G, nd;
  exa_bc bc;
  double c[3], h[3], t, gamma;
};

static __global__ __launch_bounds__(256) void k_fv_patch_hook(double* __restrict__ dst, const double* __restrict__ src,
                                                       FvHookArgs A) {
  const int dim = A.dim, P = A.P, G = A.G, S = P + 2 * G, d = A.d, side = A.side, nd = A.nd;
  const int na = dim == 3 ? P : 1;
  const int total = na * P * G;
  int o1, o2;
  fv_axes(dim, d, o1, o2);
  for (int it = blockIdx.x * blockDim.x + threadIdx.x; it < total; it += gridDim.x * blockDim.x) {
    const int k = it % G, b = (it / G) % P, a = it / (G * P);
    int x[3] = {0, 0, 0};
    x[o1] = G + b;
    if (dim == 3) x[o2] = G + a;
    auto cell = [&](int layer) {
      int y[3] = {x[0], x[1], x[2]};
      y[d] = layer;
      return dim == 3 ? ((size_t)y[2] * S + y[1]) * S + y[0] : (size_t)y[1] * S + y[0];
    };
    const size_t bk = (size_t)fv_bnd(dim, d, P, G, k, a, b);
    if (A.op == 0) {
      const size_t s = cell(fv_extract_layer(dim, d, side, P, G, k));
      for (int v = 0; v < nd; ++v) dst[bk * nd + v] = src[s * nd + v];
    } else if (A.op == 1) {
      const size_t o = cell(side ? G + P + k : k);
      for (int v = 0; v < nd; ++v) dst[o * nd + v] = src[bk * nd + v];
    } else if (A.op == 2) {
      const size_t o = cell(side ? G + P + k : k), s = cell(side ? G + k : P + k);
      for (int v = 0; v < nd; ++v) dst[o * nd + v] = src[s * nd + v];
    } else {
      const size_t bK = (size_t)fv_bnd(dim, d, P, G, G - k - 1, a, b);
      double xo[3], qin[V], qout[V];
      fv_outside_centre(dim, d, side, P, G, k, a, b, A.c, A.h, xo);
#pragma unroll
      for (int v = 0; v < V; ++v) qin[v] = src[bK * nd + v];
      fv_boundary_values(A.bc, xo, A.t, d, A.gamma, qin, qout);
#pragma unroll
      for (int v = 0; v < V; ++v) dst[bk * nd + v] = qout[v];
      for (int v = V; v < nd; ++v) dst[bk * nd + v] = src[bK * nd + v];
    }
  }
}

// Initial conditions at the subcell centres (commons.cpph:69-97).
template <int DIM>
__global__ __launch_bounds__(256) void k_fv_initial_conditions(double* __restrict__ luh, exa_ic ic, double gamma,
                                                               PatchGeom g, int nx, int ny, double ox, double oy,
                                                               double oz, double dx0, double dx1, double dx2) {
  const int p = blockIdx.x;
  const int nbox = g.ncells_box();
  const int px = p % nx, py = (p / nx) % ny, pz = p / (nx * ny);
  const double cx = ox + (px + 0.5) * dx0, cy = oy + (py + 0.5) * dx1, cz = oz + (pz + 0.5) * dx2;
  const int ninterior = DIM == 3 ? g.P * g.P * g.P : g.P * g.P;
  for (int c = threadIdx.x; c < ninterior; c += blockDim.x) {
    int i, j, k;
    interior_coords(g, c, i, j, k);
    const double qr = (2.0 * (i - g.G) + 1.0) / (2.0 * g.P);
    const double qs = (2.0 * (j - g.G) + 1.0) / (2.0 * g.P);
    const double qt = (2.0 * (k - g.G) + 1.0) / (2.0 * g.P);
    double X[3] = {cx + dx0 * (qr - 0.5), cy + dx1 * (qs - 0.5), DIM == 3 ? cz + dx2 * (qt - 0.5) : 0.0};
    double Q[V];
    exa_ic_point(ic, gamma, X, 0.0, Q);
    const int idx = box_index(g, i, j, k);
#pragma unroll
    for (int v = 0; v < V; ++v) luh[(size_t)p * V * nbox + v * nbox + idx] = Q[v];
  }
}

}  // namespace fv
}  // namespace exa
