// Space-time predictor of the Euler equations at orders 1..8, FP64 and mixed
// precision (the default form): Picard iteration, time averages, volume
// integral and face extrapolation of one cell per workgroup.  Same scheme as
// k_predictor (spaceTimePredictorNonlinear.cpph:43-577,
// volumeIntegralNonlinear.cpph:26-125).
//
// What bounds it: LDS traffic (60 words per node and slice) and vector FP64
// together, behind the latency of two barriers per slice, so the registers --
// hence the resident waves -- and the number of slices decide.  Against the
// other forms it takes one slice instead of B in the first sweep (HistTables
// a, b), half the products of the spatial contraction (ev, od), no pencil
// constants (the scale is applied once per node), and fewer registers (pin,
// park): at N = 5 168 in FP64 and 158 with FP32 sweeps, three waves per SIMD,
// instead of 255 and 239.  ms per launch (FP64 / FP32 sweeps, vortex grid;
// before: the fastest of the other forms):
//   N = 1  45^3   0.42 -> 0.23     0.45 -> 0.23
//   N = 2  45^3   0.72 -> 0.48     0.68 -> 0.40
//   N = 3  45^3   1.23 -> 0.81     1.07 -> 0.66
//   N = 4  45^3   2.84 -> 1.78     2.50 -> 1.51
//   N = 5  45^3   6.05 -> 4.07     5.69 -> 3.50
//   N = 6  27^3   3.86 -> 2.26     3.48 -> 1.94
//   N = 7  27^3   8.71 -> 3.36     7.41 -> 2.91
//   N = 8  18^3   4.57 -> 2.66     4.11 -> 1.46
#pragma once
#include "aderdg_kernels.h"

// Products and sums are fused within an expression only, so that every
// instance of a function below rounds alike: a uniform cell of the mixed
// variant takes the FP64 predictor's steps bit for bit.
#pragma clang fp contract(on)

namespace exa {

// Tables derived from the DG operators, per order.
// a, b: the first sweep.  Starting from data constant in time every level has
// the same flux, so the first iterate is q1[t] = a[t] u + b[t] L with
// a = iK1 F0, b = iK1 w, L = -dt sum_d D_d F_d(u).
// ev, od: the halves of Kxi.  The nodes are symmetric, Kxi[B-1-n][B-1-l] =
// -Kxi[n][l], so a pencil f splits into e[l] = sum_n (f[n] - f[B-1-n]) ev[n][l]
// and o[l] = sum_n (f[n] + f[B-1-n]) od[n][l] with (f Kxi)[l] = e + o and
// (f Kxi)[B-1-l] = e - o: half the products and half the table.  A middle
// node (odd B) enters od once, a middle output is ev alone.
constexpr int EXA_NH = EXA_NB / 2;
template <typename T>
struct HistTables {
  T a[EXA_NB], b[EXA_NB];
  T ev[EXA_NH][EXA_NH], od[EXA_NH][EXA_NH];
};
static __constant__ HistTables<double> c_ht[EXA_MAX_ORDER + 1];
static __constant__ HistTables<float> c_htf[EXA_MAX_ORDER + 1];

inline void fill_hist_tables(const DGTables* tab, HistTables<double>* ht) {
  for (int N = 1; N <= EXA_MAX_ORDER; ++N) {
    const int B = N + 1;
    for (int t = 0; t < B; ++t)
      for (int k = 0; k < B; ++k) {
        ht[N].a[t] += tab[N].iK1[t][k] * tab[N].F0[k];
        ht[N].b[t] += tab[N].iK1[t][k] * tab[N].w[k];
      }
    for (int n = 0; n < (B + 1) / 2; ++n)
      for (int l = 0; l < (B + 1) / 2; ++l) {
        const double p = tab[N].Kxi[n][l], q = tab[N].Kxi[n][B - 1 - l];
        ht[N].ev[n][l] = 0.5 * (p + q);
        ht[N].od[n][l] = 0.5 * (p - q);
      }
  }
}

template <typename T>
__device__ __forceinline__ const HistTables<T>& hist_tables(int N) {
  if constexpr (std::is_same<T, double>::value)
    return c_ht[N];
  else
    return c_htf[N];
}

template <int N>
struct HistOrd {
  // one flux slice in the direction layouts (the averages reuse it) and two
  // residual sums
  static constexpr int SLICE = 3 * V * Ord<N>::BLK + 32;
  // Time levels of a sweep's input iterate that wait in the LDS for the
  // residual and the flux averages: FP64 sweeps (doubles), and the one FP64
  // sweep after FP32 sweeps (floats).  Never more than the LDS holds beside the
  // slices of the workgroups that the registers admit; ms per launch with none
  // / these / as many as that (meshes as above):
  //           FP64                            FP32 sweeps
  //   N = 4   1.81 / none / 1.86 (2)          1.52 / none / 1.52 (4)
  //   N = 5   5.06 / 4.05 (2, the most)       3.93 / 3.47 (4) / 3.49 (5)
  //   N = 6   2.25 / none / 2.46 (7)          2.35 / 1.93 (5, the most)
  //   N = 7   3.36 / 3.34 (4, the most)       2.79 / 2.90 (8, the most)
  //   N = 8   2.96 / 2.66 (2, the most)       1.66 / 1.45 (4) / 1.44 (5)
  static constexpr int PARK64 = N == 5 ? 2 : N == 7 ? 4 : N == 8 ? 2 : 0;
  static constexpr int PARKMX = N == 5 ? 4 : N == 6 ? 5 : N == 7 ? 8 : N == 8 ? 4 : 0;
  // Waves per SIMD.  N = 5, ms at 45^3 with 2 / 3 / 4: FP64 5.1 / 4.2 / 7.4
  // (spills), mixed 4.5 / 3.65 / 3.8.  N = 6 is six waves per workgroup, of
  // which two fit only at 4 per SIMD: FP64 spills too much there (2.3 / - / 3.9
  // at 27^3), mixed 164 bytes a lane (2.1 / 2.1 / 1.9).  N = 7: 3.4 / 4.7 and
  // 2.9 / 3.5.
  // N = 3 (one wave per cell): 0.88 / 0.81 / 0.81 and 0.78 / 0.68 / 0.66.
  static constexpr int WPE64 = N <= 3 ? 4 : N == 6 || N == 7 ? 2 : 3;
  static constexpr int WPEMX = N == 7 ? 2 : N <= 3 || N == 6 ? 4 : 3;
  static constexpr int lds_doubles(bool fp64_sweeps, bool one_sweep) {
    const int p = fp64_sweeps ? PARK64 * V * Ord<N>::B3 : 0;
    const int q = one_sweep ? (PARKMX * V * Ord<N>::B3 + 1) / 2 : 0;
    return SLICE + (p > q ? p : q);
  }
};

// Keeps a value where it is computed: without it the time contraction's sums,
// not needed before the end of the sweep, sink there, and the terms of every
// slice are held in their place (N = 5 in FP64, nothing parked, two waves per
// SIMD: 243 registers for 190; with two levels parked 174).
template <typename T>
__device__ __forceinline__ void pin(T& x) {
  asm volatile("" : "+v"(x));
}
// A zero the compiler cannot see through: a table or memory read indexed with
// it is issued there and not hoisted to where its registers would be held for
// long.
__device__ __forceinline__ int opaque_zero() {
  int z;
  asm volatile("s_mov_b32 %0, 0" : "=s"(z));
  return z;
}

// One pencil of a slice contracted in place with Kxi (TRANSPOSED: with
// Kxi^T, the volume integral, whose halves are the transposed other ones).
template <int N, typename T, bool TRANSPOSED>
__device__ __forceinline__ void hist_contract_pencil(T* pf) {
  constexpr int B = Ord<N>::B, H = B / 2, M = B % 2;
  const HistTables<T>& K = hist_tables<T>(N);
  T d[H + M], s[H + M];
#pragma unroll
  for (int n = 0; n < H; ++n) {
    const T p = pf[n], q = pf[B - 1 - n];
    d[n] = p - q;
    s[n] = p + q;
  }
  if (M) s[H] = pf[H];
#pragma unroll
  for (int l = 0; l < H + M; ++l) {
    T e = T(0), o = T(0);
#pragma unroll
    for (int n = 0; n < H; ++n) e += d[n] * (TRANSPOSED ? K.od[l][n] : K.ev[n][l]);
    if (l < H) {
#pragma unroll
      for (int n = 0; n < H + M; ++n) o += s[n] * (TRANSPOSED ? K.ev[l][n] : K.od[n][l]);
      pf[l] = e + o;
      pf[B - 1 - l] = e - o;
    } else {
      pf[l] = e;
    }
  }
}

// The node a thread owns and what it needs in every slice.
struct HistNode {
  int s, ox, oy, oz;  // node index and its offsets in the direction layouts
  bool act;
  int rot;  // the wave that takes the first items of a phase P
};

// EulerPDE::flux with the momentum products that two directions share formed once.
template <typename T>
__device__ __forceinline__ void hist_flux(const T* Q, T (&F)[3][V], T gamma) {
  const T irho = T(1.0) / Q[0];
  const T p = (gamma - T(1)) * (Q[4] - T(0.5) * (Q[1] * Q[1] + Q[2] * Q[2] + Q[3] * Q[3]) * irho);
  const T h = Q[4] + p;
  const T u[3] = {irho * Q[1], irho * Q[2], irho * Q[3]};
  const T xy = u[0] * Q[2], xz = u[0] * Q[3], yz = u[1] * Q[3];
  F[0][0] = Q[1];
  F[0][1] = u[0] * Q[1] + p;
  F[0][2] = xy;
  F[0][3] = xz;
  F[0][4] = u[0] * h;
  F[1][0] = Q[2];
  F[1][1] = xy;
  F[1][2] = u[1] * Q[2] + p;
  F[1][3] = yz;
  F[1][4] = u[1] * h;
  F[2][0] = Q[3];
  F[2][1] = xz;
  F[2][2] = yz;
  F[2][3] = u[2] * Q[3] + p;
  F[2][4] = u[2] * h;
}

// Phase F: the flux of Q at the node, stored in the direction layouts.
template <int N, typename T>
__device__ __forceinline__ void hist_store_flux(const T* Q, T* sF, const HistNode& n, T gamma) {
  constexpr int BLK = Ord<N>::BLK;
  if (n.act) {
    T F[3][V];
    hist_flux<T>(Q, F, gamma);
#pragma unroll
    for (int v = 0; v < V; ++v) sF[(0 * V + v) * BLK + n.ox] = F[0][v];
#pragma unroll
    for (int v = 0; v < V; ++v) sF[(1 * V + v) * BLK + n.oy] = F[1][v];
#pragma unroll
    for (int v = 0; v < V; ++v) sF[(2 * V + v) * BLK + n.oz] = F[2][v];
  }
}

// Phase P: the 3 V B^2 pencils of the slice.
template <int N, typename T>
__device__ __forceinline__ void hist_contract(T* sF, int s, int rot) {
  using O = Ord<N>;
  constexpr int B2 = O::B2, PS = O::PS, BLK = O::BLK;
  constexpr int NITEMS = 3 * V * B2;
  const int s1 = s + rot * 64;
#pragma unroll 1
  for (int i = s1 < O::NT ? s1 : s1 - O::NT; i < NITEMS; i += O::NT) {
    const int dv = i / B2, ab = i - dv * B2;
    hist_contract_pencil<N, T, false>(sF + dv * BLK + ab * PS);
  }
}

// Phase A: the node's sum w (sx Px + sy Py + sz Pz) of the contracted slice.
template <int N, typename T>
__device__ __forceinline__ void hist_sum(T* r, const T* sF, const HistNode& n, T ax, T ay, T az) {
  constexpr int BLK = Ord<N>::BLK;
#pragma unroll
  for (int v = 0; v < V; ++v) {
    r[v] = ax * sF[(0 * V + v) * BLK + n.ox] + ay * sF[(1 * V + v) * BLK + n.oy] + az * sF[(2 * V + v) * BLK + n.oz];
  }
}

// Time tables in the arithmetic of the sweep, read where they are used.
template <int N, typename T>
struct HistTab {
  static constexpr bool DP = std::is_same<T, double>::value;
  int tz;
  __device__ __forceinline__ T iK1(int a, int b) const { return DP ? (T)c_tab[N + tz].iK1[a][b] : (T)c_tabf[N + tz].iK1[a][b]; }
  __device__ __forceinline__ T w(int t) const { return DP ? (T)c_tab[N + tz].w[t] : (T)c_tabf[N + tz].w[t]; }
  __device__ __forceinline__ T a(int t) const { return hist_tables<T>(N + tz).a[t]; }
  __device__ __forceinline__ T b(int t) const { return hist_tables<T>(N + tz).b[t]; }
};

// The slices of one sweep: the iterate q to its successor
// qn[t'] = a[t'] u - sum_t iK1[t'][t] R[t],
// R[t] = w_t dt (Px/(w_x dx) + Py/(w_y dy) + Pz/(w_z dz)).
// F of slice t+1 stores where A of slice t has read, by the same thread, so a
// slice takes two barriers.
// Levels below PARK of q are read from the LDS (park).
template <int N, typename T, typename TQ, int PARK>
__device__ __forceinline__ void hist_slices(const TQ (&q)[Ord<N>::B][V], T (&qn)[Ord<N>::B][V],
                                   const double* __restrict__ luh_node, T* sF, const TQ* park, const HistNode& n,
                                   T sx, T sy, T sz, T gamma) {
  constexpr int B = Ord<N>::B, B3 = Ord<N>::B3;
  {
    const HistTab<N, T> tab{opaque_zero()};
    T u[V];
#pragma unroll
    for (int v = 0; v < V; ++v) u[v] = (T)luh_node[v * B3 + tab.tz];
#pragma unroll
    for (int t = 0; t < B; ++t)
#pragma unroll
      for (int v = 0; v < V; ++v) qn[t][v] = tab.a(t) * u[v];
  }
#pragma unroll
  for (int t = 0; t < B; ++t) {
    const HistTab<N, T> tab{opaque_zero()};
    const T wt = tab.w(t);
    T Q[V];
#pragma unroll
    for (int v = 0; v < V; ++v) Q[v] = t < PARK ? (T)park[(t * V + v) * B3] : (T)q[t][v];
    hist_store_flux<N, T>(Q, sF, n, gamma);
    __syncthreads();
    hist_contract<N, T>(sF, n.s, (n.rot + t) % (Ord<N>::NT / 64));
    __syncthreads();
    T r[V];
    hist_sum<N, T>(r, sF, n, sx * wt, sy * wt, sz * wt);
#pragma unroll
    for (int t2 = 0; t2 < B; ++t2)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        qn[t2][v] -= tab.iK1(t2, t) * r[v];
        pin(qn[t2][v]);
      }
  }
}

// x plus the x of the lane that the DPP control selects (0 where it has none).
template <int CTRL, int ROWS>
__device__ __forceinline__ double add_dpp(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xf, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xf, false);
  return x + __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

// Sum over the wave, in lane 63: within rows of 16 lanes (row_shr 1, 2, 4,
// 8), then rows 0 into 1 and 2 into 3 (row_bcast 15), then 0-1 into 2-3
// (row_bcast 31).
__device__ __forceinline__ double wave_sum_dpp(double x) {
  x = add_dpp<0x111, 0xf>(x);
  x = add_dpp<0x112, 0xf>(x);
  x = add_dpp<0x114, 0xf>(x);
  x = add_dpp<0x118, 0xf>(x);
  x = add_dpp<0x142, 0xa>(x);
  return add_dpp<0x143, 0xc>(x);
}

// Whether the workgroup's sum is below tol2, in every thread.  red: the
// words of this sum, which no sum one earlier or later uses.
template <int NT>
__device__ __forceinline__ bool hist_below(double res, double tol2, double* red) {
  constexpr int NW = NT / 64;
  res = wave_sum_dpp(res);
  if ((threadIdx.x & 63) == 63) red[threadIdx.x >> 6] = res;
  __syncthreads();
  double sum = 0.0;
#pragma unroll
  for (int i = 0; i < NW; ++i) sum += red[i];
  return __builtin_amdgcn_readfirstlane(sum < tol2 ? 1 : 0) != 0;
}

// Picard sweeps from q[t] = u (FROM_U, the first of them through the time
// tables a, b) or from the iterate in r: r the final iterate, q the last
// sweep's input iterate.  Returns the sweeps executed.
template <int N, typename T, bool FROM_U, int PARK>
__device__ __forceinline__ int hist_sweeps(T (&q)[Ord<N>::B][V], T (&r)[Ord<N>::B][V], const double* __restrict__ luh_node,
                                  T* sF, T* park, double* red, const HistNode& n, T sx, T sy, T sz, T gamma, int max_sweeps,
                                  double tol2) {
  using O = Ord<N>;
  constexpr int B = O::B, B3 = O::B3;
  int it = 0;
  bool done = false;
  if (FROM_U) {
    ++it;
    T u[V], L[V];
#pragma unroll
    for (int v = 0; v < V; ++v) u[v] = (T)luh_node[v * B3];
    hist_store_flux<N, T>(u, sF, n, gamma);
    __syncthreads();
    hist_contract<N, T>(sF, n.s, n.rot);
    __syncthreads();
    hist_sum<N, T>(L, sF, n, -sx, -sy, -sz);
    T rt = T(0);
    const HistTab<N, T> tab{opaque_zero()};
#pragma unroll
    for (int t = 0; t < B; ++t)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        r[t][v] = tab.a(t) * u[v] + tab.b(t) * L[v];
        const T dd = u[v] - r[t][v];
        rt += dd * dd;
        if (t >= PARK) q[t][v] = u[v];
      }
    done = hist_below<O::NT>(n.act ? (double)rt : 0.0, tol2, red + 16) || max_sweeps == 1;
    if (PARK > 0 && done && n.act)
#pragma unroll
      for (int t = 0; t < PARK; ++t)
#pragma unroll
        for (int v = 0; v < V; ++v) park[(t * V + v) * B3] = u[v];
  }
  while (!done) {
    ++it;
#pragma unroll
    for (int t = 0; t < B; ++t)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        pin(r[t][v]);
        if (t >= PARK)
          q[t][v] = r[t][v];
        else if (n.act)
          park[(t * V + v) * B3] = r[t][v];
      }
    hist_slices<N, T, T, PARK>(q, r, luh_node, sF, park, n, sx, sy, sz, gamma);
    T rt = T(0);
#pragma unroll
    for (int t = 0; t < B; ++t)
#pragma unroll
      for (int v = 0; v < V; ++v) {
        const T dd = (t < PARK ? (T)park[(t * V + v) * B3] : q[t][v]) - r[t][v];
        rt += dd * dd;
      }
    done = hist_below<O::NT>(n.act ? (double)rt : 0.0, tol2, red + 16 * (it & 1)) || it == max_sweeps;
  }
  return it;
}

// One workgroup per cell, thread s owns node s.  Per slice t of a sweep:
//   F  node owners evaluate the flux of q[t] and store it in the direction
//      layouts;
//   P  the 3 V B^2 pencils of the slice are contracted with Kxi in place;
//   A  node owners form R = w_t dt (Px/(w_x dx) + Py/(w_y dy) + Pz/(w_z dz))
//      and take iK1[t'][t] R off every level t' of the next iterate qn, which
//      starts from a[t'] u.
// The input iterate q stays beside qn, partly in the LDS (park), for the
// residual at the end of the sweep and the flux averages after the last one.
// The first sweep starts from data constant in time and needs one slice
// (tables a, b).
// MIXED: FP32 sweeps to the FP32 rounding floor of the cell, then fp64_sweeps
// FP64 sweeps.  ONE: fp64_sweeps is 1, so that sweep needs no residual and
// its input iterate stays in FP32 and dies slice by slice.  USKIP: a cell
// uniform to FP32 resolution takes the FP64 sweeps alone (the adaptive mesh's
// variant).
template <int N, bool MIXED, bool ONE, bool USKIP>
__global__ __launch_bounds__(Ord<N>::NT) __attribute__((amdgpu_waves_per_eu(
    MIXED && ONE && !USKIP ? HistOrd<N>::WPEMX : HistOrd<N>::WPE64,
    MIXED && ONE && !USKIP ? HistOrd<N>::WPEMX : HistOrd<N>::WPE64))) void
k_predictor_history(const double* __restrict__ luh, double* __restrict__ lduh, double* __restrict__ qf,
                    double* __restrict__ ff, int* __restrict__ iters, const double* __restrict__ dtp, double dx0,
                    double dx1, double dx2, double gamma, int fp64_sweeps,
                    unsigned long long* __restrict__ sweep_count, PredictorDebug, Ens ens) {
  static_assert(MIXED || (!USKIP && !ONE), "variants of the FP32 sweeps");
  using O = Ord<N>;
  constexpr int B = O::B, B2 = O::B2, B3 = O::B3, PS = O::PS, BLK = O::BLK;
  constexpr int MaxIterations = 2 * (N + 1);
  constexpr int NITEMS = 3 * V * B2;
  constexpr double tol2 = 1e-7 * 1e-7;
  extern __shared__ double sm[];
  double* red = sm + 3 * V * BLK;
  const DGTables& T = c_tab[N];
  const size_t cell = blockIdx.x;
  HistNode n;
  n.act = threadIdx.x < B3;
  n.s = threadIdx.x;
  n.rot = (int)(cell % (O::NT / 64));
  // threads past the last node repeat node 0 and store nothing
  const int s0 = n.act ? n.s : 0;
  const int z = s0 / B2, y = (s0 / B) % B, x = s0 % B;
  n.ox = (z * B + y) * PS + x;
  n.oy = (z * B + x) * PS + y;
  n.oz = (y * B + x) * PS + z;
  double dt;
  if (ens.cell_inst) {
    const InstParams& P = ens.inst[ens.cell_inst[cell]];
    dt = P.dt_cur;
    dx0 = P.dx[0];
    dx1 = P.dx[1];
    dx2 = P.dx[2];
    gamma = P.gamma;
  } else {
    dt = *dtp;
  }
  const double* luh_node = luh + cell * V * B3 + s0;
  constexpr int PARK = HistOrd<N>::PARK64;
  double* park = sm + HistOrd<N>::SLICE + s0;
  float* parkf = reinterpret_cast<float*>(sm + HistOrd<N>::SLICE) + s0;
  const double sx = dt / (dx0 * T.w[x]), sy = dt / (dx1 * T.w[y]), sz = dt / (dx2 * T.w[z]);
  double qa[V], fh[3][V];  // time averages of the final iterate and of the last sweep's fluxes
  int it = 0;
  auto averages = [&](auto parked, const auto* in_lds, const auto& q, const double (&r)[B][V]) __attribute__((always_inline)) {
    constexpr int PK = decltype(parked)::value;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      qa[v] = 0.0;
#pragma unroll
      for (int t = 0; t < B; ++t) qa[v] += r[t][v] * T.w[t];
    }
#pragma unroll
    for (int t = 0; t < B; ++t) {
      double Q[V], F[3][V];
#pragma unroll
      for (int v = 0; v < V; ++v) Q[v] = t < PK ? (double)in_lds[(t * V + v) * B3] : (double)q[t][v];
      hist_flux<double>(Q, F, gamma);
#pragma unroll
      for (int d = 0; d < 3; ++d)
#pragma unroll
        for (int v = 0; v < V; ++v) fh[d][v] = t == 0 ? F[d][v] * T.w[t] : fh[d][v] + F[d][v] * T.w[t];
    }
  };
  bool uniform = false;
  if constexpr (MIXED) {
    // rounding floor of sum((dq)^2) over the cell in FP32: count * (4 eps |u|max)^2
    double um = 0.0, dev = 0.0;
#pragma unroll
    for (int v = 0; v < V; ++v) {
      const double uv = luh_node[v * B3];
      um = fmax(um, fabs(uv));
      if constexpr (USKIP) dev = fmax(dev, fabs(uv - luh[cell * V * B3 + v * B3]));
    }
    um = -block_min(-um, red);
    const double eps = 5.96e-8;
    if constexpr (USKIP) uniform = -block_min(-dev, red) <= 4.0 * eps * um;
    __syncthreads();
    if (!uniform) {
      const double floor_lp = (double)(V * O::B4) * (4.0 * eps * um) * (4.0 * eps * um);
      float qs[B][V], rs[B][V];
      it = hist_sweeps<N, float, true, 0>(qs, rs, luh_node, reinterpret_cast<float*>(sm), parkf, red, n, (float)sx, (float)sy,
                                       (float)sz, (float)gamma, MaxIterations, fmax(tol2, floor_lp));
      double r[B][V];
      if constexpr (ONE) {
        ++it;
        constexpr int PF = HistOrd<N>::PARKMX;
        if (PF > 0 && n.act)
#pragma unroll
          for (int t = 0; t < PF; ++t)
#pragma unroll
            for (int v = 0; v < V; ++v) parkf[(t * V + v) * B3] = rs[t][v];
        hist_slices<N, double, float, PF>(rs, r, luh_node, sm, parkf, n, sx, sy, sz, gamma);
        averages(std::integral_constant<int, PF>{}, parkf, rs, r);
      } else {
        double q[B][V];
#pragma unroll
        for (int t = 0; t < B; ++t)
#pragma unroll
          for (int v = 0; v < V; ++v) r[t][v] = (double)rs[t][v];
        it += hist_sweeps<N, double, false, PARK>(q, r, luh_node, sm, park, red, n, sx, sy, sz, gamma, fp64_sweeps, tol2);
        averages(std::integral_constant<int, PARK>{}, park, q, r);
      }
    }
  }
  if (!MIXED || uniform) {
    double q[B][V], r[B][V];
    it = hist_sweeps<N, double, true, PARK>(q, r, luh_node, sm, park, red, n, sx, sy, sz, gamma, MaxIterations, tol2);
    averages(std::integral_constant<int, PARK>{}, park, q, r);
  }

  // face values of the time-averaged state (aderExtrapolatorNonlinear :400-519)
  __syncthreads();
  if (n.act) {
#pragma unroll
    for (int v = 0; v < V; ++v) sm[v * B3 + n.s] = qa[v];
  }
  __syncthreads();
  double* qf_cell = qf + cell * 6 * V * B2;
  double* ff_cell = ff + cell * 6 * V * B2;
#pragma unroll 1
  for (int i = n.s; i < NITEMS; i += O::NT) {
    const int dv = i / B2, ab = i - dv * B2, d = dv / V, v = dv - d * V, a = ab / B, b = ab - a * B;
    const int base = d == 0 ? a * B2 + b * B : (d == 1 ? a * B2 + b : a * B + b);
    const int step = d == 0 ? 1 : (d == 1 ? B : B2);
    double qL = 0.0, qR = 0.0;
#pragma unroll
    for (int l = 0; l < B; ++l) {
      const double qv = sm[v * B3 + base + l * step];
      qL += qv * T.FL[l];
      qR += qv * T.FR[l];
    }
    qf_cell[((2 * d) * V + v) * B2 + ab] = qL;
    qf_cell[((2 * d + 1) * V + v) * B2 + ab] = qR;
  }
  __syncthreads();
  if (n.act) {
#pragma unroll
    for (int v = 0; v < V; ++v) {
      sm[(0 * V + v) * BLK + n.ox] = fh[0][v];
      sm[(1 * V + v) * BLK + n.oy] = fh[1][v];
      sm[(2 * V + v) * BLK + n.oz] = fh[2][v];
    }
  }
  __syncthreads();
  // face fluxes and the volume integral's contraction from one read of each pencil
#pragma unroll 1
  for (int i = n.s; i < NITEMS; i += O::NT) {
    const int dv = i / B2, ab = i - dv * B2, d = dv / V, v = dv - d * V;
    double* pf = sm + dv * BLK + ab * PS;
    double fL = 0.0, fR = 0.0;
#pragma unroll
    for (int l = 0; l < B; ++l) {
      const double fv = pf[l];
      fL += fv * T.FL[l];
      fR += fv * T.FR[l];
    }
    ff_cell[((2 * d) * V + v) * B2 + ab] = fL;
    ff_cell[((2 * d + 1) * V + v) * B2 + ab] = fR;
    hist_contract_pencil<N, double, true>(pf);
  }
  __syncthreads();
  if (n.act) {
    // volumeIntegralNonlinear.cpph:26-125, and the update's volume part if asked for
    const double usx = (T.w[z] * T.w[y]) / dx0, usy = (T.w[z] * T.w[x]) / dx1, usz = (T.w[y] * T.w[x]) / dx2;
    const double updateSize = dt / (T.w[z] * T.w[y] * T.w[x]);
#pragma unroll
    for (int v = 0; v < V; ++v) {
      double out = usx * sm[(0 * V + v) * BLK + n.ox] + usy * sm[(1 * V + v) * BLK + n.oy] +
                   usz * sm[(2 * V + v) * BLK + n.oz];
      if (ens.fold_update) out = luh_node[v * B3] + out * updateSize;
      lduh[cell * V * B3 + v * B3 + n.s] = out;
    }
  }
  if (n.s == 0) {
    if (iters) iters[cell] = it;
    count_sweeps(sweep_count, cell, it);
  }
}

}  // namespace exa

#pragma clang fp contract(fast)
