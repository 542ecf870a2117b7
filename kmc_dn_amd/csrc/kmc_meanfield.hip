// Mean-field estimators of the Go library.
//
// probSimulate (goSimulation/probabilitySimulation.go:53-157, behind
// wrapperSimulateProbability, simulationWrapper.go:235-250) integrates
// fractional occupations deterministically.  Each step:
//   * site energies from the occupations (:82-90), FP64;
//   * every pair's rate t_ij = p_ij * nu * min(1, exp(-dE/kT)) * tc_ij with the
//     occupation factor p_ij of probTransitionPossible (:40-50) (calcProbTransitions
//     :8-38), and their total;
//   * a step that moves each occupation by its net flow over the total, capped so
//     that none leaves [0, 1] (:96-110), the clock advancing 0.98 x that step;
//   * occupation, electrode occupation and net traffic moved by rate x cap / total.
// A workgroup runs one network: its threads form the terms of all pairs, then one
// lane per site adds its row (rates out) and its column (rates in) from LDS, in
// ascending order, and wave 0 finishes the step.  Sums run in a different order
// than the reference's row-major loops, so results agree to rounding, not bit for
// bit.
//
// calcAverageCurrent (goSimulation/simulation.go:671-736, the second half of
// wrapperSimulateCombined) evaluates the same rates once at a time-averaged
// occupation, with the reference's FP32 site energies and energy differences
// (the wrapper casts its inputs to float32), and returns each electrode's net
// inflow over the total rate divided by the reference's time step 0.98 / total.
#include "kmc_device.h"

namespace kmc {

namespace {

// probTransitionPossible (probabilitySimulation.go:40-50)
__device__ __forceinline__ double occupation_factor(int i, int j, int N, double oi, double oj) {
  if (i >= N && j >= N) return 0.0;
  if (i >= N) return 1.0 - oj;
  if (j >= N) return oi;
  return (1.0 - oj) * oi;
}

__device__ __forceinline__ double wave_sum_f64(double x) {
  const double incl = wave_scan_f64(x);
  return readlane_f64(incl, 63);
}

__device__ __forceinline__ double wave_min_f64(double x) {
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const double y = __shfl_xor(x, o, 64);
    x = y < x ? y : x;
  }
  return x;
}

// The terms of the pair (i, j): t_ij = p_ij * m(e_j - e_i - cd) * tc_ij and t_ji, with
// m(dE) = nu * min(1, exp(-dE/kT)).  With cd >= 0 at most one of the two energy
// differences is positive, so one exp serves both (cd < 0: a second one).
__device__ __forceinline__ void pair_terms(int i, int j, int N, double oi, double oj, double ei,
                                           double ej, double cd, double tij, double tji, double nu,
                                           double kT, double& out, double& in) {
  const double dout = ej - ei - cd;   // i -> j
  const double din = ei - ej - cd;    // j -> i
  const bool first = dout > din;
  const double hi = first ? dout : din, lo = first ? din : dout;
  // (kT = 1, energies in units of kT, is the common case: no division)
  const double x = kT == 1.0 ? hi : hi / kT;
  const double mh = hi > 0 ? nu * exp(-x) : nu;
  double ml = nu;
  if (lo > 0) ml = nu * exp(-lo / kT);
  out = occupation_factor(i, j, N, oi, oj) * (first ? mh : ml) * tij;
  in = occupation_factor(j, i, N, oj, oi) * (first ? ml : mh) * tji;
}

// What a network's step works on, in LDS: the acceptors' occupations, all sites'
// energies, their rows' and columns' sums, and occupation x time (acceptors) or
// electrode occupation (electrodes) so far.
template <int C>
struct Sites {
  double occ[64 * C], se[64 * C], row[64 * C], col[64 * C], sum[64 * C], time, f;
  __device__ __forceinline__ void init(const MeanfieldParams& p, int k, int N, int tid, int n) {
    for (int s = tid; s < 64 * C; s += n) {
      occ[s] = s < N ? p.occ[(size_t)k * NMAX + s] : 0.0;
      se[s] = sum[s] = 0.0;
    }
    if (tid == 0) time = 0.0;
  }
  // The end of a step, by one wave whose lanes own the sites lane + 64c: the total
  // rate, the step that keeps every occupation in [0, 1] (:96-110) and the clock;
  // f: the step's length, by which every pair's term counts.
  __device__ __forceinline__ void rate(int N, int S, int lane, double& step_time) {
    double part = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c)
      if (lane + 64 * c < S) part += row[lane + 64 * c];
    const double tot = wave_sum_f64(part);
    double cap = 1.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      if (s >= N) continue;
      const double dr = (col[s] - row[s]) / tot, o = occ[s];
      const double nv = o + dr;
      if (nv < 0) {
        const double r = o / -dr;
        cap = r < cap ? r : cap;
      }
      if (nv > 1) {
        const double r = (1.0 - o) / dr;
        cap = r < cap ? r : cap;
      }
    }
    const double max_change = wave_min_f64(cap);
    step_time = 0.98 * max_change / tot;
    if (lane == 0) {
      time += step_time;
      f = max_change / tot;
    }
    wave_lds_sync();
  }
  // Moves the occupations (the same wave).
  __device__ __forceinline__ void move(int N, int S, int lane, double step_time) {
    const double ff = f;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      if (s < N) {
        sum[s] += occ[s] * step_time;
        double o = occ[s] + (col[s] - row[s]) * ff;
        o = o < 0 ? 0.0 : (o > 1 ? 1.0 : o);   // (:146-155)
        occ[s] = o;
      } else if (s < S) {
        sum[s] += (col[s] - row[s]) * ff;
      }
    }
  }
  __device__ __forceinline__ void write(const MeanfieldParams& p, int k, int N, int S, int lane) const {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      if (s < N) {
        p.occ[(size_t)k * NMAX + s] = occ[s];
        if (p.se) p.se[(size_t)k * NMAX + s] = se[s];
        if (p.avg) p.avg[(size_t)k * NMAX + s] = sum[s];
      } else if (s < S) {
        p.eo[(size_t)k * PMAX + (s - N)] = sum[s];
      }
    }
    if (lane == 0 && p.time) p.time[k] = time;
  }
};

// Sum of n values, `stride` doubles apart, added in order; eight loads in flight.
__device__ __forceinline__ double sum_in_order(const double* x, int stride, int n) {
  double a = 0.0;
  for (; n >= 8; n -= 8) {
    double t[8];
#pragma unroll
    for (int g = 0; g < 8; ++g) {
      t[g] = *x;
      x += stride;
    }
#pragma unroll
    for (int g = 0; g < 8; ++g) a += t[g];
  }
  for (; n > 0; --n, x += stride) a += *x;
  return a;
}

}  // namespace

// probSimulate, S <= MF_LDS_SITES and tables symmetric to the bit.  Bound by the pairs'
// FP64 work (an exp, three divisions).  Each unordered pair i <= j belongs to
// one of W * 64 threads, which keeps its constants and its net traffic in registers
// (up to Q pairs) and writes t_ij and t_ji into the S x S table t in LDS, of odd
// row length: the lanes that add the rows (stride ld) and those that add the
// columns (stride 1) both read it without conflicts.  64 networks of 28
// to 108 sites, 300 steps with records: 3.14 ms, 10.5 us a step of the largest (about
// 4 us of it the pairs at the FP64 rate of one CU, the rest the sums' and the step's
// dependent additions and the barriers).  Eight waves of twice the pairs: 3.72 ms;
// the sums' loads 16 ahead, which costs spilled registers: 3.7 ms.  Before, one wave
// ran a network and formed every pair's terms from both ends, and once more for the
// traffic, with two exps and two divisions each: 75 ms.
// p.ld: row length of t, the launch's largest S rounded up to an odd number.
template <int C, int Q, int W>
__global__ void __launch_bounds__(64 * W) __attribute__((amdgpu_waves_per_eu(4)))
kmc_meanfield_kernel(MeanfieldParams p) {
  extern __shared__ __align__(16) double t[];   // [S][ld]
  __shared__ Sites<C> x;
  const int k = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const LayoutDev L = p.layouts[p.layout_of[k]];
  const EsetDev es = p.esets[p.eset_of[k]];
  const int N = L.N, S = L.S, ld = p.ld, pairs = S * (S + 1) / 2;
  const double nu = L.nu, kT = L.kT, I0R = L.I0R;
  x.init(p, k, N, tid, 64 * W);
  // pair q of this thread: number tid + q * 64 W of the rows' (i, i..S-1)
  constexpr bool kKeep = Q <= 6;   // constants in registers; more of them do not fit
  constexpr int K = kKeep ? Q : 1;
  int ij[Q];
  double d[K], cd[K], tc[K], tr[Q];
  auto distance = [&](int i, int j) { return i < N && j < N ? L.dist64[__umul24(i, S) + j] : 1.0; };
  auto coulomb = [&](int i, int j, double dd) { return i < N && j < N ? I0R / dd : 0.0; };
  {
    int i = 0, j = tid;   // number = those of the rows before i, plus j - i
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      ij[q] = -1;
      tr[q] = 0.0;
      if (kKeep) cd[q % K] = tc[q % K] = d[q % K] = 0.0;
      while (i < S && j >= S) {   // past row i: on with row i + 1, which starts at i + 1
        j -= S - (i + 1);
        ++i;
      }
      if (tid + q * 64 * W < pairs) {
        ij[q] = i << 8 | j;
        if (kKeep) {
          tc[q % K] = L.tc64[__umul24(i, S) + j];
          d[q % K] = distance(i, j);
          cd[q % K] = coulomb(i, j, d[q % K]);
        }
      }
      j += 64 * W;
    }
  }
  __syncthreads();
  auto at = [ld](int i, int j) { return __umul24(i, ld) + j; };
  // The pairs' addresses are formed anew in each phase: kept, they would push the
  // constants out of the registers.
  auto renew = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < Q; ++q) asm volatile("" : "+v"(ij[q]));
  };
  for (int64_t step = 0; step < p.steps; ++step) {
    renew();
    // the terms of the site energies (:82-90); a site adds nothing to itself
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ij[q] >> 8, j = ij[q] & 255;
      if (ij[q] >= 0 && j < N) {   // (i <= j)
        const double dd = kKeep ? d[q % K] : distance(i, j);
        t[at(j, i)] = i == j ? 0.0 : (1.0 - x.occ[j]) / dd;
        if (i != j) t[at(i, j)] = (1.0 - x.occ[i]) / dd;
      }
      __builtin_amdgcn_sched_barrier(0);   // (registers: pair after pair)
    }
    __syncthreads();
    if (wave < C) {
      const int s = lane + 64 * wave;
      if (s < N) x.se[s] = es.E[s] - I0R * sum_in_order(t + s, ld, N);
      else if (s < S) x.se[s] = es.V[s - N];
    }
    __syncthreads();
    renew();
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ij[q] >> 8, j = ij[q] & 255;
      if (ij[q] >= 0) {
        double out, in;
        const double tcq = kKeep ? tc[q % K] : L.tc64[__umul24(i, S) + j];
        pair_terms(i, j, N, x.occ[i], x.occ[j], x.se[i], x.se[j],
                   kKeep ? cd[q % K] : coulomb(i, j, distance(i, j)),
                   tcq, tcq, nu, kT, out, in);
        t[at(i, j)] = out;
        t[at(j, i)] = in;   // (i == j: the same)
      }
      __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    if (wave < 2 * C) {
      const bool rows = wave < C;
      const int s = lane + 64 * (rows ? wave : wave - C);
      double a = 0.0;
      if (s < S) a = sum_in_order(t + (rows ? s * ld : s), rows ? 1 : ld, S);
      (rows ? x.row : x.col)[s] = a;
    }
    __syncthreads();
    if (wave == 0) {
      double step_time;
      x.rate(N, S, lane, step_time);
      x.move(N, S, lane, step_time);
    }
    __syncthreads();
    if (p.traffic) {
      const double f = x.f;
      renew();
#pragma unroll
      for (int q = 0; q < Q; ++q) {   // (t_ij and t_ji are this thread's until it writes them)
        const int i = ij[q] >> 8, j = ij[q] & 255;
        if (ij[q] >= 0 && i < N) tr[q] += (t[at(i, j)] - t[at(j, i)]) * f;
      }
    }
  }
  renew();
  if (p.traffic) {
    double* o = p.traffic + (size_t)k * p.tstride;
#pragma unroll
    for (int q = 0; q < Q; ++q) {
      const int i = ij[q] >> 8, j = ij[q] & 255;
      if (ij[q] < 0) continue;
      o[i * S + j] = tr[q];
      if (i != j) o[j * S + i] = 0.0 - tr[q];
    }
  }
  if (wave == 0) x.write(p, k, N, S, lane);
}

// probSimulate for the networks that kmc_meanfield_kernel does not take: the table
// of a larger one does not fit in LDS, and with asymmetric tables the terms that a
// row and a column see differ.  The terms out of and into every site go through
// LDS in tiles of MF_TILE partners; the same bits.  One such network sends a call's
// every network here (a launch has one kernel): 64 networks of 28 to 108 sites, 100 steps
// with records, 4.5 ms a call for an asymmetric table instead of 1.8 (25.6 with one
// wave per network); with one of 158 sites 7.7, which is that network's own time (16 of
// them 7.0; 56 and 59 with one wave each).
constexpr int MF_TILE_WAVES = 16;
template <int C>
__global__ void __launch_bounds__(64 * MF_TILE_WAVES) kmc_meanfield_tiled_kernel(MeanfieldParams p) {
  extern __shared__ __align__(16) double t[];   // [2][MF_TILE][ld]
  __shared__ Sites<C> x;
  constexpr int ld = 64 * C + 1;
  double* const t2 = t + MF_TILE * ld;
  const int k = blockIdx.x;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int jj = tid % MF_TILE, s0 = tid / MF_TILE;   // this thread's column and first row of a tile
  constexpr int SSTEP = 64 * MF_TILE_WAVES / MF_TILE;
  const LayoutDev L = p.layouts[p.layout_of[k]];
  const EsetDev es = p.esets[p.eset_of[k]];
  const int N = L.N, S = L.S;
  const double *dist = L.dist64, *tc = L.tc64;
  const double nu = L.nu, kT = L.kT, I0R = L.I0R;
  x.init(p, k, N, tid, 64 * MF_TILE_WAVES);
  __syncthreads();
  auto terms = [&](int s, int j, double& out, double& in) {
    const double cd = s < N && j < N ? I0R / dist[s * S + j] : 0.0;
    pair_terms(s, j, N, x.occ[s], x.occ[j], x.se[s], x.se[j], cd, tc[s * S + j], tc[j * S + s], nu,
               kT, out, in);
  };
  for (int64_t step = 0; step < p.steps; ++step) {
    double acc = 0.0;
    for (int j0 = 0; j0 < N; j0 += MF_TILE) {
      const int n = min(MF_TILE, N - j0), j = j0 + jj;
      if (jj < n)
        for (int s = s0; s < N; s += SSTEP)
          t[jj * ld + s] = s == j ? 0.0 : (1.0 - x.occ[j]) / dist[s * S + j];
      __syncthreads();
      if (wave < C && lane + 64 * wave < N)
        for (int g = 0; g < n; ++g) acc += t[g * ld + lane + 64 * wave];
      __syncthreads();
    }
    if (wave < C) {
      const int s = lane + 64 * wave;
      if (s < N) x.se[s] = es.E[s] - I0R * acc;
      else if (s < S) x.se[s] = es.V[s - N];
    }
    __syncthreads();
    acc = 0.0;
    for (int j0 = 0; j0 < S; j0 += MF_TILE) {
      const int n = min(MF_TILE, S - j0);
      if (jj < n)
        for (int s = s0; s < S; s += SSTEP) terms(s, j0 + jj, t[jj * ld + s], t2[jj * ld + s]);
      __syncthreads();
      if (wave < 2 * C) {
        const bool rows = wave < C;
        const int s = lane + 64 * (rows ? wave : wave - C);
        if (s < S)
          for (int g = 0; g < n; ++g) acc += (rows ? t : t2)[g * ld + s];
      }
      __syncthreads();
    }
    if (wave < C) x.row[lane + 64 * wave] = acc;
    else if (wave < 2 * C) x.col[lane + 64 * (wave - C)] = acc;
    __syncthreads();
    double step_time = 0.0;
    if (wave == 0) x.rate(N, S, lane, step_time);
    if (p.traffic) {
      __syncthreads();
      const double f = x.f;
      double* tr = p.traffic + (size_t)k * p.tstride;
      for (int j = jj; j < S; j += MF_TILE)
        for (int s = s0; s < S; s += SSTEP) {
          if (s >= N && j >= N) continue;
          double out, in;
          terms(s, j, out, in);
          tr[s * S + j] += (out - in) * f;
        }
      __syncthreads();   // (all read the occupations before they move)
    }
    if (wave == 0) x.move(N, S, lane, step_time);
    __syncthreads();
  }
  if (wave == 0) x.write(p, k, N, S, lane);
}

// calcAverageCurrent (simulation.go:671-736) at the occupations p.occ; writes the
// currents into p.eo.  Site energies and energy differences are FP32 as in the
// reference (its inputs are float32 copies); rates and sums are FP64.
template <int C>
__global__ void __launch_bounds__(64) kmc_avg_current_kernel(MeanfieldParams p) {
  __shared__ double occ_l[64 * C];
  __shared__ float se_l[64 * C];
  const int k = blockIdx.x;
  if (k >= p.n) return;
  const int lane = threadIdx.x;
  const LayoutDev L = p.layouts[p.layout_of[k]];
  const EsetDev es = p.esets[p.eset_of[k]];
  const int N = L.N, S = L.S;
  const double* d = L.dist64;
  const double* tc = L.tc64;
  const float nu = (float)L.nu, kT = (float)L.kT, I0 = (float)L.I0, R = (float)L.R;
  double occ[C];
  float se[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    occ[c] = s < N ? p.occ[(size_t)k * NMAX + s] : 0.0;
    occ_l[s] = occ[c];
  }
  wave_lds_sync();
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    se[c] = 0.f;
    if (s < N) {
      double ai = 0.0;
      for (int j = 0; j < N; ++j)
        if (j != s) ai += (1.0 - occ_l[j]) / (double)(float)d[(size_t)s * S + j];
      se[c] = (float)es.E[s] - I0 * R * (float)ai;
    } else if (s < S) {
      se[c] = (float)es.V[s - N];
    }
    se_l[s] = se[c];
  }
  wave_lds_sync();
  double row[C], col[C];
#pragma unroll
  for (int c = 0; c < C; ++c) row[c] = col[c] = 0.0;
  for (int j = 0; j < S; ++j) {
    const double oj = j < N ? occ_l[j] : 0.0;
    const float sej = se_l[j];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      if (s >= S) continue;
      const bool acc = s < N && j < N;
      const float cd = acc ? I0 * R / (float)d[(size_t)s * S + j] : 0.f;
      const float dout = acc ? sej - se[c] - cd : sej - se[c];
      const float din = acc ? se[c] - sej - cd : se[c] - sej;
      const double mout = dout > 0 ? (double)nu * exp((double)(-dout / kT)) : (double)nu;
      const double min_ = din > 0 ? (double)nu * exp((double)(-din / kT)) : (double)nu;
      row[c] += occupation_factor(s, j, N, occ[c], oj) * mout * (double)(float)tc[(size_t)s * S + j];
      col[c] += occupation_factor(j, s, N, oj, occ[c]) * min_ * (double)(float)tc[(size_t)j * S + s];
    }
  }
  double part = 0.0;
#pragma unroll
  for (int c = 0; c < C; ++c)
    if (lane + 64 * c < S) part += row[c];
  const double tot = wave_sum_f64(part);
  const double time_step = 0.98 / tot;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    if (s >= N && s < S) p.eo[(size_t)k * PMAX + (s - N)] = ((col[c] - row[c]) / tot) / time_step;
  }
}

template __global__ void kmc_meanfield_kernel<1, 5, 8>(MeanfieldParams);
template __global__ void kmc_meanfield_kernel<2, 6, 16>(MeanfieldParams);
template __global__ void kmc_meanfield_kernel<3, 10, 16>(MeanfieldParams);
template __global__ void kmc_meanfield_tiled_kernel<1>(MeanfieldParams);
template __global__ void kmc_meanfield_tiled_kernel<2>(MeanfieldParams);
template __global__ void kmc_meanfield_tiled_kernel<3>(MeanfieldParams);
template __global__ void kmc_avg_current_kernel<1>(MeanfieldParams);
template __global__ void kmc_avg_current_kernel<2>(MeanfieldParams);
template __global__ void kmc_avg_current_kernel<3>(MeanfieldParams);

}  // namespace kmc
