// Team kernels of the FP32 batched path: T waves (one workgroup) per trajectory,
// by members of the walked set or by site chunks.
//
// For long trajectories on a GPU that the batch does not fill, the hop latency
// of one trajectory bounds the launch.  A team splits the walked set of every
// hop over T waves on different SIMDs (Team in kmc_traj.h); the remaining
// per-hop work is replicated.  Workgroups pull one trajectory at a time from
// the atomic queue.  FORM: 1 {lt, lt+c} + c table, 2 {lt, c} table, 3 positions;
// table forms keep the layout's table in LDS while consecutive trajectories
// share it.
#include "kmc_traj.h"

namespace kmc {

// PH: the phase-timing instantiation (run_trajectory).
template <int C, int T, bool REC, int FORM, bool PH>
__global__ void __launch_bounds__(64 * T) kmc_team_kernel(BatchParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  Team<T, C> team;
  team.wave = wave;
  team.red = reinterpret_cast<float*>(smem);
  unsigned char* area = p.states + ((size_t)blockIdx.x * T + wave) * p.state_area;
  unsigned char* rest = smem + (size_t)2 * T * C * 64 * sizeof(float);
  __shared__ int s_group;
  __shared__ int s_layout;
  if (threadIdx.x == 0) s_layout = -1;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_group = atomicAdd(p.queue, 1);
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(s_group);
    if (g >= p.ngroups) break;
    const GroupDev gd = p.groups[g];
    const LayoutDev L = p.layouts[gd.layout];
    if constexpr (FORM == 3) {
      float4* pos = reinterpret_cast<float4*>(rest);
      for (int k = threadIdx.x; k < L.S; k += 64 * T) pos[k] = L.pos4[k];
      __syncthreads();
      PosPolicy<C> pol;
      pol.init(pos, L, lane);
      for (int i = 0; i < gd.count; ++i)
        run_trajectory<C, REC, PosPolicy<C>, T, true, PH>(p, gd.first + i, L, pol, lane, team, area);
    } else {
      // the waves' electrode factors (T*2*PMAX floats), the electrode weights,
      // the pair table and, for FORM 1, the c table
      constexpr bool BT = FORM == 1;
      float* evc = reinterpret_cast<float*>(rest) + wave * 2 * PMAX;
      float* elw = reinterpret_cast<float*>(rest) + T * 2 * PMAX;
      float2* tab = reinterpret_cast<float2*>(elw + elw_lds_floats(L.P, C));
      float* ctab = reinterpret_cast<float*>(tab + L.S * L.S + 64 * C);
      if (gd.layout != __builtin_amdgcn_readfirstlane(s_layout)) {
        load_elw<C>(elw, L, threadIdx.x, 64 * T);
        const int n = L.S * L.S + 64 * C;
        const float2* src = BT ? L.tabB : L.tab32;
        for (int k = threadIdx.x; k < n; k += 64 * T) tab[k] = src[k];
        if (BT) {
          const int nc = L.N * L.S + 64 * C;
          for (int k = threadIdx.x; k < nc; k += 64 * T) ctab[k] = L.ccol[k];
        }
        __syncthreads();
        if (threadIdx.x == 0) s_layout = gd.layout;
      }
      __syncthreads();
      const TabPolicy<C, BT> pol = TabPolicy<C, BT>::make(tab, ctab, elw, evc, L.S, lane);
      for (int i = 0; i < gd.count; ++i)
        run_trajectory<C, REC, TabPolicy<C, BT>, T, true, PH>(p, gd.first + i, L, pol, lane, team, area);
    }
  }
}

// One trajectory of several site chunks per workgroup of C waves, the row sums of
// each new state split by chunks: the bits of the solo kernels, which give a
// trajectory one wave.  For launches whose trajectories leave SIMDs idle, where
// a trajectory's latency is what counts: the row sums are most of a new state
// (about 4,500 of 6,500 cycles a hop for one that finds a new state on every
// hop, S = 130 in the positions form).  A network of S <= 64 runs in one-chunk
// code on wave 0.
template <int C, bool REC, int FORM>
__global__ void __launch_bounds__(64 * C) kmc_split_kernel(BatchParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int lane = threadIdx.x & 63;
  unsigned char* area = p.states + ((size_t)blockIdx.x * C + wave) * p.state_area;
  __shared__ int s_group;
  __shared__ int s_layout;
  __shared__ int s_flag;
  Team<C, C, true> team;
  team.wave = wave;
  team.red = reinterpret_cast<float*>(smem);
  team.flag = &s_flag;
  unsigned char* rest = smem + (size_t)2 * C * 64 * sizeof(float);
  if (threadIdx.x == 0) s_layout = -1;
  for (;;) {
    __syncthreads();
    if (threadIdx.x == 0) s_group = atomicAdd(p.queue, 1);
    __syncthreads();
    const int g = __builtin_amdgcn_readfirstlane(s_group);
    if (g >= p.ngroups) break;
    const GroupDev gd = p.groups[g];
    const LayoutDev L = p.layouts[gd.layout];
    const bool one = L.S <= 64;
    if constexpr (FORM == 3) {
      float4* pos = reinterpret_cast<float4*>(rest);
      for (int k = threadIdx.x; k < L.S; k += 64 * C) pos[k] = L.pos4[k];
      __syncthreads();
      if (one) {
        if (wave == 0) {
          PosPolicy<1> pol;
          pol.init(pos, L, lane);
          for (int i = 0; i < gd.count; ++i)
            run_trajectory<1, REC, PosPolicy<1>, 1, true, false, false>(
                p, gd.first + i, L, pol, lane, Team<1, 1>{}, area);
        }
      } else {
        PosPolicy<C> pol;
        pol.init(pos, L, lane);
        PosPolicy<1> polw;
        polw.init(pos, L, lane + 64 * wave);
        polw.elm[0] = chunk_mask(L.N, L.S, wave);
        for (int i = 0; i < gd.count; ++i)
          run_trajectory<C, REC, PosPolicy<C>, C, true, false, false, Team<C, C, true>>(
              p, gd.first + i, L, pol, lane, team, area, &polw);
      }
    } else {
      // the waves' electrode factors, the electrode weights, the pair table and,
      // for FORM 1, the c table
      constexpr bool BT = FORM == 1;
      const int Ce = one ? 1 : C;
      float* evc = reinterpret_cast<float*>(rest) + wave * 2 * PMAX;
      float* elw = reinterpret_cast<float*>(rest) + C * 2 * PMAX;
      float2* tab = reinterpret_cast<float2*>(elw + elw_lds_floats(L.P, Ce));
      float* ctab = reinterpret_cast<float*>(tab + L.S * L.S + 64 * Ce);
      if (gd.layout != __builtin_amdgcn_readfirstlane(s_layout)) {
        if (one) load_elw<1>(elw, L, threadIdx.x, 64 * C);
        else load_elw<C>(elw, L, threadIdx.x, 64 * C);
        const int n = L.S * L.S + 64 * Ce;
        const float2* src = BT ? L.tabB : L.tab32;
        for (int k = threadIdx.x; k < n; k += 64 * C) tab[k] = src[k];
        if (BT) {
          const int nc = L.N * L.S + 64 * Ce;
          for (int k = threadIdx.x; k < nc; k += 64 * C) ctab[k] = L.ccol[k];
        }
        __syncthreads();
        if (threadIdx.x == 0) s_layout = gd.layout;
      }
      __syncthreads();
      if (one) {
        if (wave == 0) {
          const TabPolicy<1, BT> pol = TabPolicy<1, BT>::make(tab, ctab, elw, evc, L.S, lane);
          for (int i = 0; i < gd.count; ++i)
            run_trajectory<1, REC, TabPolicy<1, BT>, 1, true, false, false>(
                p, gd.first + i, L, pol, lane, Team<1, 1>{}, area);
        }
      } else {
        const TabPolicy<C, BT> pol = TabPolicy<C, BT>::make(tab, ctab, elw, evc, L.S, lane);
        const TabPolicy<1, BT> polw =
            TabPolicy<1, BT>::make(tab, ctab, elw, evc, L.S, lane + 64 * wave);
        for (int i = 0; i < gd.count; ++i)
          run_trajectory<C, REC, TabPolicy<C, BT>, C, true, false, false, Team<C, C, true>>(
              p, gd.first + i, L, pol, lane, team, area, &polw);
      }
    }
  }
}

#define KMC_SPLIT(C)                                                  \
  template __global__ void kmc_split_kernel<C, false, 1>(BatchParams); \
  template __global__ void kmc_split_kernel<C, true, 1>(BatchParams);  \
  template __global__ void kmc_split_kernel<C, false, 2>(BatchParams); \
  template __global__ void kmc_split_kernel<C, true, 2>(BatchParams);  \
  template __global__ void kmc_split_kernel<C, false, 3>(BatchParams); \
  template __global__ void kmc_split_kernel<C, true, 3>(BatchParams);
KMC_SPLIT(2) KMC_SPLIT(3)
#undef KMC_SPLIT

#define KMC_TEAM(C, T)                                                           \
  template __global__ void kmc_team_kernel<C, T, false, 1, false>(BatchParams); \
  template __global__ void kmc_team_kernel<C, T, true, 1, false>(BatchParams);  \
  template __global__ void kmc_team_kernel<C, T, false, 2, false>(BatchParams); \
  template __global__ void kmc_team_kernel<C, T, true, 2, false>(BatchParams);  \
  template __global__ void kmc_team_kernel<C, T, false, 3, false>(BatchParams); \
  template __global__ void kmc_team_kernel<C, T, true, 3, false>(BatchParams);
KMC_TEAM(1, 2) KMC_TEAM(1, 4) KMC_TEAM(2, 2) KMC_TEAM(2, 4) KMC_TEAM(3, 2) KMC_TEAM(3, 4)
#undef KMC_TEAM
// phase timing: teams of 4 on two- and three-chunk networks
#define KMC_TEAM(C, F) template __global__ void kmc_team_kernel<C, 4, false, F, true>(BatchParams);
KMC_TEAM(2, 1) KMC_TEAM(2, 2) KMC_TEAM(2, 3) KMC_TEAM(3, 1) KMC_TEAM(3, 2) KMC_TEAM(3, 3)
#undef KMC_TEAM

// LDS bytes of a workgroup of the kernels that split by site chunks.
size_t split_lds_bytes(int form, int C, int S, int N, int P) {
  size_t b = (size_t)2 * C * 64 * sizeof(float);
  if (form == 3) return b + (size_t)64 * C * sizeof(float4);
  b += (size_t)C * 2 * PMAX * sizeof(float);
  b += (size_t)elw_lds_floats(P, C) * sizeof(float);
  b += ((size_t)S * S + 64 * C) * sizeof(float2);
  if (form == 1) b += ((size_t)N * S + 64 * C) * sizeof(float);
  return b;
}

// LDS bytes of a team workgroup: partial row sums plus the form's tables or
// positions (an upper bound for layouts with at most S, N and P).
size_t team_lds_bytes(int form, int C, int T, int S, int N, int P) {
  size_t b = (size_t)2 * T * C * 64 * sizeof(float);
  if (form == 3) return b + (size_t)64 * C * sizeof(float4);
  b += (size_t)T * 2 * PMAX * sizeof(float);
  b += (size_t)elw_lds_floats(P, C) * sizeof(float);
  b += ((size_t)S * S + 64 * C) * sizeof(float2);
  if (form == 1) b += ((size_t)N * S + 64 * C) * sizeof(float);
  return b;
}

}  // namespace kmc
