// FP32-rate / FP64-accumulate hop loop of one trajectory (device code shared by
// the solo kernels, kmc_batch.hip, and the team kernels, kmc_team.hip).
//
// Same model as _simulate_discrete_record (kmc_dopant_networks.py:33-135) and
// Go's simulate (goSimulation/simulation.go:194-325), organised for CDNA4:
//
//  * Each lane owns sites s = lane + 64*c (c < C).  Site energies live in
//    registers as e~ = se * log2(e)/kT; electrodes hold V * log2(e)/kT.
//  * With lt = log2(nu * tc) and c = scaled Coulomb term I_0*R/d a rate is
//        2^(lt + min(0, e~_src - e~_dst + c)) = 2^min(lt, b + e~_src - e~_dst),
//    b = lt + c: one v_exp_f32 per pair and no FP32 underflow of the 10^-50
//    prefactors.  Where the pair terms come from is a policy:
//      TabB  {lt, b} pair table + c table in LDS, shared by the W waves of a
//            workgroup that run W trajectories of one layout (fewest VALU ops);
//      TabC  {lt, c} pair table in LDS (smaller; largest networks);
//      Pos   positions only (16 B per site in LDS per wave): d, lt and c are
//            computed per pair, ~2.5x the VALU work but no table, so waves of
//            different layouts fill a CU independently.
//  * Per hop, the smaller of {sources} (occupied acceptors + electrodes) and
//    {targets} (empty acceptors + electrodes) is walked in blocks of four
//    members (the last block exactly the members left) while the lanes cover
//    every site of the other role: row sums R_lane accumulate in registers with
//    no cross-lane traffic.
//  * Table policies leave the electrodes out of the walked set: with
//    w = nu * tc[s][e] the rates between acceptor s and all electrodes sum to
//        sum_e w * min(1, 2^e~_s * 2^-V~_e)   (s occupied, hops into them) or
//        sum_e w * min(1, 2^-e~_s * 2^V~_e)   (s empty, hops out of them),
//    one product (its clamp is the min) and one FMA per electrode and no exp2
//    per pair (elec_sums).  The per-trajectory factors 2^+-V~_e sit in LDS.  In
//    one-wave kernels a hop on which no lane of the other role has its energy
//    inside the electrodes' voltage window takes per-lane sums fixed for the
//    trajectory instead.
//  * Event pick: FP64 wave prefix sum of R (DPP), Philox event uniform * total,
//    ballot for the first lane whose prefix exceeds it, then one lane-parallel
//    pass over that lane's pairs (FP32 DPP scan) for the partner site.
//  * Hop: each wave keeps the transitions its trajectory takes, one per lane, and
//    the states between them (run_trajectory): a hop by a kept transition is one
//    lane-parallel test, and only new transitions and new states take the steps
//    above.  The clock is accumulated in FP64.  A new
//    state's energies get O(N) Coulomb column updates (makeJump,
//    simulation.go:107-130): in one-chunk solo code the last FP64 recompute's
//    energies plus one column per acceptor whose occupation changed since, in
//    ascending site order (a function of the occupation alone); elsewhere the
//    previous state's plus the rank-1 update of the hop.
//  * At every multiple of `recompute_interval` hops the energies are rebuilt in
//    FP64 from E_constant and the I_0*R/d table (the Go reference never
//    re-synchronises).
//  * Uniforms come from one Philox block per lane every 64 hops (lane k holds
//    hop h0+k), so the RNG costs two readlanes per hop.
//  * A trajectory runs the absolute hop range [h_begin, h_end) of its budget
//    and, with `resume`, starts from the state its previous launch wrote.
//    Ranges that start at multiples of the recompute interval continue the
//    trajectory exactly as one long launch would (same energies, same stream).
//  * A team of T waves (one workgroup) can run one trajectory: wave w walks
//    the members u of the walked set with u = w (mod T), the partial row sums
//    meet in LDS (one barrier per new state) and are added in wave order, so
//    every wave continues with the same bits; the rest of the hop is replicated.
#pragma once
#include "kmc_device.h"

namespace kmc {

// LDS floats of a layout's electrode weights: P rounded up to 4 rows (padding
// rows zero) of 64C lane sites, so every load of a block of four electrodes has
// an immediate offset.
__host__ __device__ inline int elw_lds_floats(int P, int C) { return ((P + 3) & ~3) * 64 * C; }

// Copies the electrode weights (global rows of 192 sites) into LDS rows of 64C.
template <int C>
__device__ __forceinline__ void load_elw(float* dst, const LayoutDev& L, int tid, int nthreads) {
  const int n = elw_lds_floats(L.P, C);
  for (int k = tid; k < n; k += nthreads) dst[k] = L.elw[(k / (64 * C)) * 192 + k % (64 * C)];
}

template <int C>
__device__ __forceinline__ void recompute_energies(float (&se)[C], const uint64_t (&occ)[C],
                                                   const LayoutDev& L, const EsetDev& es,
                                                   int lane) {
  const int N = L.N, S = L.S;
  const double sc = (double)L.scale2;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    float v = 0.f;
    if (s < N) {
      // the sum over the empty acceptors in ascending order; the terms of eight
      // acceptors are loaded together (one memory round trip per eight; an
      // index past the last loads the last's term and adds nothing)
      const double e = es.E[s];
      const double* col = L.coul64 + s;
      double acc = 0.0;
      if constexpr (C == 1) {
        for (int j0 = 0; j0 < N; j0 += 8) {
          double t[8];
#pragma unroll
          for (int g = 0; g < 8; ++g) t[g] = col[min(j0 + g, N - 1) * N];
#pragma unroll
          for (int g = 0; g < 8; ++g) {
            const int j = j0 + g;
            acc += (j < N && !((occ[0] >> (j & 63)) & 1ull) && j != s) ? t[g] : 0.0;
          }
        }
      } else {
        for (int j = 0; j < N; ++j)
          if (!((occ[j >> 6] >> (j & 63)) & 1ull) && j != s) acc += col[j * N];
      }
      v = (float)((e - acc) * sc);
    } else if (s < S) {
      v = (float)(es.V[s - N] * sc);
    }
    se[c] = v;
  }
}

// A wave-uniform 64-bit value in SGPRs (no instruction when it is there already).
__device__ __forceinline__ uint64_t uniform_u64(uint64_t x) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)x);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(x >> 32));
  return ((uint64_t)hi << 32) | lo;
}
// Lowest set bit of a wave-uniform mask, -1 when it is empty (s_ff1 returns -1
// for 0, which __builtin_ctzll leaves undefined).
__device__ __forceinline__ int lowest_bit(uint64_t m) {
  int r;
  m = uniform_u64(m);
  asm("s_ff1_i32_b64 %0, %1" : "=s"(r) : "s"(m));
  return r;
}

// Set bits of a wave-uniform mask as a 32-bit scalar (s_bcnt1 sets SCC).
__device__ __forceinline__ int popcount64(uint64_t m) {
  int r;
  m = uniform_u64(m);
  asm("s_bcnt1_i32_b64 %0, %1" : "=s"(r) : "s"(m) : "scc");
  return r;
}

// m with bit (b mod 64) cleared.
__device__ __forceinline__ uint64_t clear_bit(uint64_t m, int b) {
  m = uniform_u64(m);
  asm("s_bitset0_b64 %0, %1" : "+s"(m) : "s"(b));
  return m;
}

// Lanes l of site chunk c (site l + 64c) with lo <= site < hi, as a lane mask.
__device__ __forceinline__ uint64_t chunk_mask(int lo, int hi, int c) {
  const int a = lo - 64 * c < 0 ? 0 : lo - 64 * c;
  const int b = hi - 64 * c > 64 ? 64 : hi - 64 * c;
  if (b <= a) return 0ull;
  const uint64_t below_b = b >= 64 ? ~0ull : ((1ull << b) - 1);
  return below_b & ~((1ull << a) - 1);
}

// min(a, b) for non-NaN operands as one v_min_f32.  fminf (and fmed3 with an
// infinite operand, which the compiler folds into it) first canonicalises any
// operand loaded from LDS with an extra v_max_f32 under IEEE mode; the pair
// terms are never NaN, so the plain instruction is exact here.
__device__ __forceinline__ float min_f32(float a, float b) {
  float r;
  asm("v_min_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

// ---------------------------------------------------------------------------
// Pair-term policies.  For a uniform member u of the walked set and the lane
// sites s = lane + 64c, pair(pre(u), c, diff) is log2 of the rate of the pair
// (src, dst) with e~_src - e~_dst = diff; coul(u, c) is c(s, u) for
// the energy update (u an acceptor).  prefetch(u) issues the loads that
// pair() needs, so four members can be in flight together.
// ---------------------------------------------------------------------------
template <int C, bool BT>
struct TabPolicy {
  static constexpr bool kElec = true;   // electrodes in closed form (elec_sums)
  // coul(N, c) is 0: column N of the c table lies in its zero padding, and column
  // N of the pair table is an electrode column (or, with no electrodes, the
  // padding), c = 0
  static constexpr bool kZeroColumnN = true;
  // [S*S + 64C]: entry (s, u) at u*S + s; the 64C padding entries (lt = -inf)
  // take the reads of the lanes past S in column S - 1
  const float2* tab;
  const float* ctab;   // BT: [N*S + 64C] c at u*S + s
  const float* elw;    // [4*ceil(P/4)][64C] electrode weights of the lane sites
  float* evc;          // this wave's [2][PMAX]: 2^V~_e, then 2^-V~_e
  int S, lane;
  // column strides in bytes (S * 8, S * 4), held in vector registers so that a
  // member's column address is one v_mad_u32_u24 of its scalar index
  int stride2, stride1;
  __device__ __forceinline__ static TabPolicy make(const float2* tab, const float* ctab,
                                                   const float* elw, float* evc, int S, int lane) {
    TabPolicy p{tab, ctab, elw, evc, S, lane, S * 8, S * 4};
    asm("" : "+v"(p.stride2), "+v"(p.stride1));
    return p;
  }
  // the lane's entry of column u: tab + lane + u*S
  __device__ __forceinline__ const float2* col(int u) const {
    return reinterpret_cast<const float2*>(reinterpret_cast<const char*>(tab + lane) +
                                           __umul24((unsigned)u, (unsigned)stride2));
  }
  struct Pre {
    float2 e[C];
  };
  // u in [0, S)
  __device__ __forceinline__ Pre prefetch(int u) const {
    Pre p;
    const float2* cl = col(u);
#pragma unroll
    for (int c = 0; c < C; ++c) p.e[c] = cl[64 * c];
    return p;
  }
  // energy difference e~_src - e~_dst = sg * d (sg = +-1, exact)
  __device__ __forceinline__ float pair(const Pre& p, int c, float d, float sg) const {
    if constexpr (BT) return min_f32(p.e[c].x, fmaf(sg, d, p.e[c].y));
    else return p.e[c].x + min_f32(0.f, fmaf(sg, d, p.e[c].y));
  }
  __device__ __forceinline__ float coul(int u, int c) const {
    if constexpr (BT)
      return reinterpret_cast<const float*>(reinterpret_cast<const char*>(ctab + lane) +
                                            __umul24((unsigned)u, (unsigned)stride1))[64 * c];
    else return col(u)[64 * c].y;
  }
};

template <int C>
struct PosPolicy {
  static constexpr bool kElec = false;   // electrodes are walked as members
  static constexpr bool kZeroColumnN = false;
  const float* elw = nullptr;
  float* evc = nullptr;
  const float4* pos;   // [S] per wave: x, y, z, 1 for acceptors / 0 for electrodes
  float px[C], py[C], pz[C], kcl[C];   // the lane sites' coordinates and c scale
  uint64_t elm[C];     // lanes of chunk c that hold electrodes
  float l0, mkl;       // lt = l0 + mkl * d
  int lane, N, S;
  struct Pre {
    float4 q;
    bool el;           // wave-uniform: the member is an electrode
  };
  __device__ __forceinline__ void init(const float4* p, const LayoutDev& L, int ln) {
    pos = p;
    lane = ln;
    N = L.N;
    S = L.S;
    l0 = L.pos_l0;
    mkl = L.pos_mkl;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      const float4 q = s < L.S ? pos[s] : make_float4(1e6f, 1e6f, 1e6f, 0.f);
      px[c] = q.x;
      py[c] = q.y;
      pz[c] = q.z;
      kcl[c] = q.w * L.pos_kc;
      elm[c] = chunk_mask(L.N, L.S, c);
    }
  }
  // u in [0, S)
  __device__ __forceinline__ Pre prefetch(int u) const {
    Pre p;
    p.q = pos[u];
    p.el = u >= N;
    return p;
  }
  __device__ __forceinline__ float dist_rinv(const float4& q, int c, float& rinv) const {
    const float dx = px[c] - q.x, dy = py[c] - q.y, dz = pz[c] - q.z;
    // explicit FMAs: the same bits in every instantiation, whatever the
    // compiler would contract around it
    const float d2 = fmaxf(fmaf(dz, dz, fmaf(dy, dy, dx * dx)), 1e-30f);
    rinv = __builtin_amdgcn_rsqf(d2);
    return d2 * rinv;
  }
  // energy difference e~_src - e~_dst = sg * dd (sg = +-1, exact)
  __device__ __forceinline__ float pair(const Pre& p, int c, float dd, float sg) const {
    float rinv;
    const float d = dist_rinv(p.q, c, rinv);
    const float lt = fmaf(mkl, d, l0);
    const float cc = rinv * kcl[c] * p.q.w;
    const float x = lt + min_f32(0.f, fmaf(sg, dd, cc));
    // electrode-electrode pairs (an electrode with itself included) have no
    // rate: a wave-uniform lane mask selects them
    return __builtin_amdgcn_inverse_ballot_w64(p.el ? elm[c] : 0ull) ? -INFINITY : x;
  }
  __device__ __forceinline__ float coul(int u, int c) const {
    const float4 q = pos[u];
    float rinv;
    (void)dist_rinv(q, c, rinv);
    return (u == lane + 64 * c) ? 0.f : rinv * kcl[c] * q.w;
  }
};

// T waves sharing one trajectory, in one of two ways:
//  * by members (SPLIT false): wave w walks the members u = w (mod T) for every
//    lane site; the partial sums meet in LDS and are added in wave order.  red:
//    LDS [2][T][C][64] partial row sums;
//  * by site chunks (SPLIT, T = C): wave w walks every member for the lane sites
//    of chunk w, in the order one wave takes, so the sums have one wave's bits.
//    red: LDS [2][C][64] row sums; flag: LDS, wave 0's word on a time limit.
// Both double-buffered by reduction, so one barrier per reduction suffices.
template <int T, int C, bool SPLIT = false>
struct Team {
  static constexpr bool kSplit = SPLIT;
  int wave = 0;        // rank in the team (wave-uniform)
  float* red = nullptr;
  int* flag = nullptr;
  // members u of the walked set this wave takes: u = wave (mod T)
  __device__ __forceinline__ uint64_t own() const {
    if constexpr (T == 1 || SPLIT) return ~0ull;
    else if constexpr (T == 2) return 0x5555555555555555ull << wave;
    else return 0x1111111111111111ull << wave;
  }
  __device__ __forceinline__ bool writer() const { return T == 1 || wave == 0; }
  // Sum of the T partial row sums, added in wave order (same bits in every wave);
  // SPLIT: the waves' chunks, mine in R[wave].
  __device__ __forceinline__ void reduce(float (&R)[C], int parity, int lane) const {
    if constexpr (SPLIT) {
      float* all = red + parity * C * 64 + lane;
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (c == wave) all[c * 64] = R[c];
      __syncthreads();
#pragma unroll
      for (int c = 0; c < C; ++c) R[c] = all[c * 64];
    } else if constexpr (T > 1) {
      float* mine = red + ((parity * T + wave) * C) * 64;
#pragma unroll
      for (int c = 0; c < C; ++c) mine[c * 64 + lane] = R[c];
      __syncthreads();
      const float* all = red + (parity * T) * C * 64;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        float acc = all[c * 64 + lane];
#pragma unroll
        for (int w = 1; w < T; ++w) acc += all[(w * C + c) * 64 + lane];
        R[c] = acc;
      }
    }
  }
};

// K members of the walked set (the lowest K bits of m, all present; K <= the
// number of bits left): their columns are loaded together, then their terms added.
template <int K, int C, class Pol>
__device__ __forceinline__ void row_block(const Pol& pol, int S, int cu, uint64_t& m,
                                          const float (&v)[C], const float (&se)[C], float sg,
                                          float (&R)[C]) {
  int b[K];
  typename Pol::Pre pre[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    b[k] = lowest_bit(m);
    m = clear_bit(m, b[k]);
  }
#pragma unroll
  for (int k = 0; k < K; ++k) pre[k] = pol.prefetch(64 * cu + b[k]);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float su = readlane_f32(se[cu], b[k]);
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && 64 * c >= S) break;   // chunk past this layout's sites
      R[c] += fast_exp2(pol.pair(pre[k], c, v[c] - su, sg));
    }
  }
}

// Row sums over the uniform set U (bits of umask & own), lanes covering the
// other role.  sg = +1: U = targets, lanes = sources (e~_src - e~_dst = v - su);
// sg = -1: U = sources, lanes = targets.  One code path for both: the sign is a
// scalar operand of the pair term's FMA.  Members go in blocks of four; the last
// block takes exactly the members left (a scalar branch on their count), so no
// lane computes a padding term.  The members are counted once, not before every
// block: the scalar chain between the blocks is a good part of a new state's cost
// (one trajectory of 1e5 hops, N = 30 at 300 kT, 129 -> 117 ms; 512 x 1e4 hops, N = 40,
// 14.7 -> 13.5 ms).  Blocks across the chunks save LDS round trips but
// cost scalar selects per member: 64 x 21,000 hops of N = 100 18.2 -> 19.6 ms.
template <int C, class Pol>
__device__ __forceinline__ void row_sums(const Pol& pol, int S, const uint64_t (&umask)[C],
                                         uint64_t own, const float (&v)[C],
                                         const float (&se)[C], float sg, float (&R)[C]) {
#pragma unroll
  for (int cu = 0; cu < C; ++cu) {
    uint64_t m = umask[cu] & own;
    int n = popcount64(m);
    for (; n >= 4; n -= 4) row_block<4>(pol, S, cu, m, v, se, sg, R);
    if (n == 3) row_block<3>(pol, S, cu, m, v, se, sg, R);
    else if (n == 2) row_block<2>(pol, S, cu, m, v, se, sg, R);
    else if (n == 1) row_block<1>(pol, S, cu, m, v, se, sg, R);
  }
}

// The same for one chunk of lane sites: pol is the policy of that chunk alone, v
// its energies, se all the chunks' (the members').
template <int K, int C, class Pol1>
__device__ __forceinline__ void row_block_one(const Pol1& pol, int cu, uint64_t& m, float v,
                                              const float (&se)[C], float sg, float& R) {
  int b[K];
  typename Pol1::Pre pre[K];
#pragma unroll
  for (int k = 0; k < K; ++k) {
    b[k] = lowest_bit(m);
    m = clear_bit(m, b[k]);
  }
#pragma unroll
  for (int k = 0; k < K; ++k) pre[k] = pol.prefetch(64 * cu + b[k]);
#pragma unroll
  for (int k = 0; k < K; ++k) {
    const float su = readlane_f32(se[cu], b[k]);
    R += fast_exp2(pol.pair(pre[k], 0, v - su, sg));
  }
}
template <int C, class Pol1>
__device__ __forceinline__ void row_sums_one(const Pol1& pol, const uint64_t (&umask)[C], float v,
                                             const float (&se)[C], float sg, float& R) {
#pragma unroll
  for (int cu = 0; cu < C; ++cu) {
    uint64_t m = umask[cu];
    int n = popcount64(m);
    for (; n >= 4; n -= 4) row_block_one<4>(pol, cu, m, v, se, sg, R);
    if (n == 3) row_block_one<3>(pol, cu, m, v, se, sg, R);
    else if (n == 2) row_block_one<2>(pol, cu, m, v, se, sg, R);
    else if (n == 1) row_block_one<1>(pol, cu, m, v, se, sg, R);
  }
}

// Closed-form electrode terms of the row sums (table policies).  v: the lane
// sites' scaled energies; the sums of lanes outside the role are discarded by
// the caller, and electrode lanes have w = 0.  The exponent is clamped to 126
// (then x -+ V~ >= 26 and the min is 1 either way); |V~| <= 100 keeps 2^-+V~
// finite and nonzero, so the product is never NaN, and min(1, product) of a
// non-negative product is the multiply's own clamp to [0, 1].
// Electrodes go in blocks of four (all loads of a block issued together); rows
// past P have w = 0 and factor 1.  A team splits the blocks: wave w takes the
// blocks j = w (mod T).  The blocks are unrolled to the PMAX / 4 a layout can
// have, so every load takes an immediate offset from one base per hop; a
// wave-uniform branch skips the blocks past P.
// CS: site chunks of a row of the weights (a chunk on its own: C = 1, the lanes
// shifted by the policy).
template <int C, int T, class Pol, int CS = C>
__device__ __forceinline__ void elec_sums(const Pol& pol, int P, int S, bool udst, int wave,
                                          const float (&v)[C], float (&R)[C]) {
  float ex[C];
#pragma unroll
  for (int c = 0; c < C; ++c) ex[c] = fast_exp2(min_f32(udst ? v[c] : -v[c], 126.f));
  const float* k = pol.evc + (udst ? PMAX : 0) + 4 * wave;
  const float* w = pol.elw + pol.lane + 4 * wave * 64 * CS;
  const int nb = (P + 3) >> 2;
  constexpr int kBlocks = (PMAX / 4 + T - 1) / T;
#pragma unroll
  for (int i = 0; i < kBlocks; ++i) {
    if (wave + T * i >= nb) break;
    const float4 k4 = *reinterpret_cast<const float4*>(k + 4 * T * i);
    const float kq[4] = {k4.x, k4.y, k4.z, k4.w};
    float wq[4][C];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int c = 0; c < C; ++c) wq[q][c] = w[(4 * T * i + q) * 64 * CS + 64 * c];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (c > 0 && 64 * c >= S) break;
        R[c] = fmaf(wq[q][c], __builtin_amdgcn_fmed3f(ex[c] * kq[q], 0.f, 1.f), R[c]);
      }
  }
}

// (float)x of lane l: converted on every lane, then one readlane (the compiler
// would otherwise read both halves of x and convert the scalar pair)
__device__ __forceinline__ float readlane_as_f32(double x, int l) {
  float f = (float)x;
  asm("" : "+v"(f));
  return readlane_f32(f, l);
}

template <int C>
__device__ __forceinline__ float pick_lane_value(const float (&x)[C], int site) {
  const int cs = site >> 6, ls = site & 63;
  float r = readlane_f32(x[0], ls);
#pragma unroll
  for (int c = 1; c < C; ++c)
    if (cs == c) r = readlane_f32(x[c], ls);
  return r;
}

template <int C>
__device__ __forceinline__ double pick_lane_f64(const double (&x)[C], int site) {
  const int cs = site >> 6, ls = site & 63;
  double r = readlane_f64(x[0], ls);
#pragma unroll
  for (int c = 1; c < C; ++c)
    if (cs == c) r = readlane_f64(x[c], ls);
  return r;
}

// x in VGPRs: an inline-asm result with a VGPR operand counts as varying
// across lanes, so x and what is computed from it stay in VGPRs.  For
// wave-uniform values that only vector instructions (or rare paths) use,
// keeping them out of the SGPRs that the hop loop runs short of; also a product
// that must not be contracted into a later subtraction.
__device__ __forceinline__ uint64_t in_vgpr(uint64_t x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ double in_vgpr(double x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ int in_vgpr_i(int x) {
  asm("" : "+v"(x));
  return x;
}
__device__ __forceinline__ float in_vgpr(float x) {
  asm("" : "+v"(x));
  return x;
}
// `old` with lane l (its low six bits) set to the wave-uniform x: the compiler
// has the intrinsic but no builtin for it, and sees its wait states (a
// v_writelane in inline asm would hide them).
extern "C" __device__ int writelane_i32(int x, int l, int old) __asm("llvm.amdgcn.writelane.i32");
__device__ __forceinline__ uint64_t readlane_u64(uint64_t x, int l) {
  const uint32_t lo = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)x, l);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(x >> 32), l);
  return ((uint64_t)hi << 32) | lo;
}

// The hop loop.  A trajectory revisits a few states and leaves each of them by a
// few events (of the hops of a network at N = 30 and 1 kT 0.5-1.5 % take an event
// not taken since the last recompute; at +-300 kT 10-50 %), so a wave keeps up
// to 63 transitions, one per lane, all in registers: the state it leaves, the
// bounds of the event uniform u that select it, the clock's rate factor and the
// state it leads to.  A hop then is one lane-parallel test of its uniform and a
// ballot, with no memory access (a new transition costs the row selection and a
// pass over the row's partners, a new state its row sums besides, 1,000 to
// 3,000 cycles).  The general selection is
//
//   target = u * total            selects row sel iff lo <= target < hi
//   rr = (float)(target - exs)    selects its partner iff plo <= rr < phi
//
// with hi the row's FP64 inclusive prefix, exs the prefix before it, phi the
// partner's FP32 inclusive prefix; it takes the first lane whose prefix exceeds
// the target, so lo and plo are the largest prefixes before.  The prefixes are
// tree sums of non-negative terms, monotone up to their rounding (at most 8
// roundings each), so the prefix just before, times 1 + 2^-48 (FP32: 1 + 2^-19),
// bounds all of them.  All of these bounds are bounds of u; rounded inwards, they
// are kept as two FP32 numbers (relative margin 2^-20, which covers every
// rounding on the way): a uniform inside them selects this transition in the
// general selection too, and one in the gaps beside them (about 1e-6 of the
// hops) takes the general selection, with the same result.  Lane 63 is no
// transition: its bounds hold every uniform and its end is unknown, so a hop
// that no kept transition takes finds it.
//
// States: up to 64 (p.state_slots) per wave, their occupation words in the lanes
// of key[], their row sums and energies (512 B per chunk, from which the prefixes
// are formed again with the same bits) in the wave's area of p.states.  That is
// global memory, read when a new transition leaves a state other than the last
// two, whose records are in registers; the oldest state makes room when all are
// taken.  A one-chunk solo state's energies are a function of its occupation
// between two recomputes (kPathFree), so there an occupation names a state and a
// new transition's end is looked up among the kept ones.  Elsewhere a state's
// energies come from the state before it (its rank-1 update), and a hop back
// into the state before the last hop takes that state as it was: a state is
// known again by the transition it was formed by, from the same kept state (of
// the new states at S = 118 and 1 kT half to two thirds), and the same occupation
// reached on another way is another state, with other rounding.  Every state and
// transition is dropped at each FP64 recompute, so ranges that start at
// multiples of the recompute interval continue exactly.  The Go library keeps a
// cache keyed by occupation too (simulation.go:254-296).
//
// Leaps: when the hops go back and forth between two states, whether hop k of
// the current uniform block does depends only on its own uniform, so the lanes
// test the 64 hops of the block in parallel, and the run of hops that pass is
// applied at once.
//
// General steps: a trajectory that finds too many new states runs whole recompute
// intervals by the steps above alone, with the current state and the one before
// it in registers (kPlainShift below); so do the teams by members over several
// chunks.  Same bits: both take a hop back to the state before it as that state
// was, and both drop everything at the recompute.
//
// Measured, before (two states in registers, an LDS store of four evicted ones,
// leaps) and now: 4096 x 1e5 hops of N = 30 at 1 kT 44.9 and 15.3 ms; one
// trajectory of 1e5 hops with records 63.4 and 9.1 ms, at 300 kT 47.7 and 26.4
// ms; 4096 x 2e4 hops of an IV sweep 10.0 and 3.7 ms; 64 x 21,000 of N = 100
// with records 25.9 and 18.1 ms.
//
// PH: the phase-timing instantiation: shader-clock reads at the phase
// boundaries of every hop (FP32_PHASES), summed into p.phases by the first wave
// of each trajectory.  The reads wait for the wave's outstanding LDS and scalar
// loads, so its hops are somewhat slower than the others'.
// ONE: the code runs in a kernel built for one site chunk (false for the
// one-chunk code of kernels over several chunks).
// area: this wave's area of p.states; null: general steps alone.
// polw: the pair terms of this wave's chunk alone (teams by site chunks).
// Always inlined: out of line (as the compiler would have it for three chunks) the
// policy's LDS pointers pass through memory, every table read is a generic load and
// the kernel takes 256 VGPRs, 40 AGPRs and 750 bytes of scratch: 512 x 3000 hops of S =
// 132 in table form 2, workgroups of four, 11.4 ms at 300 kT, inlined 8.3.
template <int C, bool REC, class Pol, int T = 1, bool PRIO = true, bool PH = false,
          bool ONE = (C == 1), class TeamT = Team<T, C>, class PolW = Pol>
__device__ __forceinline__ void run_trajectory(const BatchParams& p, int t, const LayoutDev& L, const Pol& pol,
                               int lane, const TeamT& team, unsigned char* area,
                               const PolW* polw = nullptr) {
  constexpr bool SPLIT = TeamT::kSplit;
  constexpr bool kMembers = T > 1 && !SPLIT;   // a team by members

  const int64_t t_start = wall_clock64();
  const TrajDev td = p.trajs[t];
  const EsetDev es = p.esets[td.eset];
  const int N = L.N, S = L.S;
  TrajOut* o = p.out + t;
  // hop counters are 32-bit (prehops + hops <= INT32_MAX is checked when a batch
  // is created), so their comparisons stay on the scalar unit
  const int64_t total64 = td.prehops + td.hops;
  const int64_t hb64 = p.resume ? (td.h_begin < total64 ? td.h_begin : total64) : 0;
  const int64_t he64 = p.resume ? (td.h_end < total64 ? td.h_end : total64) : total64;
  const int h_begin = (int)hb64, h_end = (int)he64, prehops = (int)td.prehops;
  const bool cont = p.resume && h_begin > 0;

  // the occupation of state oid, or of the trajectory while no kept state is
  // current (cur < 0); acceptors (N <= 64C) live in the first C words
  uint64_t occ[C];
  int oid = -1;
  float se[C];
  int eo[C];
  double ot[C];
#pragma unroll
  for (int w = 0; w < C; ++w) occ[w] = uniform_u64(cont ? o->occ[w] : td.occ[w]);
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    eo[c] = (cont && s >= N && s < S) ? (int)o->eo[s - N] : 0;
    ot[c] = (cont && REC && p.occ_time && s < N) ? p.occ_time[(size_t)t * NMAX + s] : 0.0;
  }
  double time = cont ? o->time : 0.0;
  float lg_lane = 0.f;    // log2(1 - u_clock) * -ln 2 = -ln(1 - u_clock) of hop (h & ~63) + lane
  double ue_lane = 0.0;   // event uniform of that hop
  float uf_lane = 0.f;    // the same in FP32, for the kept transitions' bounds
  // The clock: each hop's rate factor waits in its hop's lane of the uniform
  // block (lane h & 63, 0 for hops not taken) until a fixed-order FP64 wave sum
  // adds the block's FP32 waiting times -ln(1-u)/total to `time`, at every
  // special hop (uniforms, end of the prehops, recompute) and at the end of the
  // range, so its bits do not depend on how the block's hops were taken.
  float rtv = 0.f;
  int32_t status = __builtin_amdgcn_readfirstlane(cont ? o->status : (int32_t)ST_OK);
  recompute_energies<C>(se, occ, L, es, lane);
  // Energies of a new state.  One-chunk solo code: the last recompute's plus the
  // columns of the acceptors changed since.  Teams and kernels over several site
  // chunks: the previous state's plus the rank-1 update of the hop that left it
  // (two columns; the miss-heavy trajectories these run change many sites
  // between recomputes); psrc, pdst: that hop's ends, pend: its update is still
  // to be applied.
  constexpr bool kPathFree = C == 1 && T == 1;
  // Teams by members over several chunks take general steps only: a team exists
  // for the long trajectories that find a new state on every second or third hop
  // and set a batch's length (alone, a team of four, us a hop with transitions /
  // by general steps: S = 129, 47 % new states 1.74 / 1.50; S = 112, 32 % 1.05 /
  // 0.84; S = 118, 15 % 0.55 / 0.60; S = 80, 0.4 % 0.17 / 0.37), and without the
  // tables their waves leave room on the SIMDs for a batch's other launches.
  // So do the positions kernels over several chunks, which serve the launches that
  // fill the chip: the 2048 networks of the bench batch 1,042 ms with the tables, 975 by
  // general steps (both at two waves per SIMD; kmc_batch_pos_kernel holds more now).
  constexpr bool kGeneral = C > 1 && (kMembers || (T == 1 && !Pol::kElec));
  int psrc = 0, pdst = 0;
  bool pend = false;
  float base_se[C];
  uint64_t base_occ[C];
#pragma unroll
  for (int c = 0; c < C; ++c) {
    base_se[c] = se[c];
    base_occ[c] = occ[c];
  }
  uint64_t accm[C], elm[C];   // lanes of chunk c holding acceptors / electrodes
#pragma unroll
  for (int c = 0; c < C; ++c) {
    accm[c] = chunk_mask(0, N, c);
    elm[c] = chunk_mask(N, S, c);
  }
  // electrodes in closed form when the policy has the weights and every scaled
  // voltage satisfies |V~| <= 100; otherwise they are walked as members
  bool elec = false;
  // Hops on which every lane of the other role has all its electrode terms
  // saturated (x >= max V~ side) or all below 1 take per-lane sums fixed for the
  // trajectory: sum_e w, or 2^x sum_e w 2^-+V~ (x = +-v as in elec_sums).
  float esum_w[C], esum_dst[C], esum_src[C];   // sum w, sum w 2^-V~, sum w 2^V~
  float vt_max = 0.f, vt_min = 0.f;
  if constexpr (Pol::kElec) {
    const float vt = lane < L.P ? (float)(es.V[lane] * (double)L.scale2) : 0.f;
    elec = L.P > 0 && L.elw_ok && ballot(!(fabsf(vt) <= 100.f)) == 0;
    if (lane < PMAX) {   // 2^0 = 1 past P: finite factors for the zero padding rows
      pol.evc[lane] = fast_exp2(vt);
      pol.evc[PMAX + lane] = fast_exp2(-vt);
    }
    wave_lds_sync();
#pragma unroll
    for (int c = 0; c < C; ++c) esum_w[c] = esum_dst[c] = esum_src[c] = 0.f;
    if (elec && !kMembers) {
      vt_max = -INFINITY;
      vt_min = INFINITY;
      for (int e = 0; e < L.P; ++e) {
        const float ve = readlane_f32(vt, e);
        vt_max = fmaxf(vt_max, ve);
        vt_min = fminf(vt_min, ve);
        const float ks = pol.evc[e], kd = pol.evc[PMAX + e];
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const float w = pol.elw[e * 64 * C + 64 * c + lane];
          esum_w[c] += w;
          esum_dst[c] = fmaf(w, kd, esum_dst[c]);
          esum_src[c] = fmaf(w, ks, esum_src[c]);
        }
      }
    }
  }
  uint64_t walk[C];   // sites that may be walked: acceptors, plus electrodes unless elec
#pragma unroll
  for (int c = 0; c < C; ++c) walk[c] = elec ? accm[c] : ~0ull;

  const int K = p.recompute_interval;
  // next FP64 recompute (a multiple of K; INT32_MAX: none left in this range)
  auto next_multiple = [K](int64_t x) {
    const int64_t n = (x / K + 1) * K;
    return (int)(n < INT32_MAX ? n : INT32_MAX);
  };
  int next_rc = next_multiple(h_begin);
  int h_stop = status == ST_OK ? h_end : h_begin;   // a stopped trajectory stays
  int h = h_begin;
  // uniforms of hops (hh & ~63) + lane: at the start and at every multiple of 64
  auto refill = [&](int hh) {
    double uc;
    stream_uniforms(td.seed, td.hop0 + (uint64_t)((hh & ~(int64_t)63) + lane), uc, ue_lane);
    lg_lane = fast_log2((float)(1.0 - uc)) * -0.69314718055994531f;
    uf_lane = (float)ue_lane;
  };
  if (h < h_stop && (h & 63) != 0) refill(h);
  // the next hop with work besides the hop itself: a multiple of 64 (uniforms),
  // the end of the prehops (tallies restart) or a multiple of K (recompute)
  // (32-bit unsigned arithmetic: hh <= INT32_MAX, so r <= 2^31 and no 64-bit
  // compare, which the scalar unit lacks, is needed)
  auto next_special = [&](int hh, bool inclusive) {
    const unsigned r = inclusive ? ((unsigned)hh + 63u) & ~63u : ((unsigned)hh | 63u) + 1u;
    int n = (int)(r < (unsigned)INT32_MAX ? r : (unsigned)INT32_MAX);
    if (next_rc < n) n = next_rc;
    if ((inclusive ? prehops >= hh : prehops > hh) && prehops < n) n = prehops;
    return n;
  };
  int special = next_special(h, true);
  // hops below h_lim need nothing besides the hop itself
  int h_lim = special < h_stop ? special : h_stop;
  uint64_t ph[FP32_PHASES] = {};
  uint64_t tp = PH ? __builtin_amdgcn_s_memtime() : 0;
  bool ph_back = false;
  auto mark = [&](int k) {
    if constexpr (PH) {
      const uint64_t now = __builtin_amdgcn_s_memtime();
      ph[k] += now - tp;
      tp = now;
    }
  };
  int nred = 0;   // team reductions so far
  // New states of the current recompute interval, and whether the last interval
  // had more than 16 (held in VGPRs: touched on new states and at recomputes
  // only).  Such a trajectory is among the slowest of a batch, whose launch
  // lasts as long as they do: its waves issue at priority 2 instead of 1
  // outside the hop's chain, ahead of the faster waves that share their SIMDs.
  // One-chunk kernels with graded priority only: in an uneven batch the solo
  // kernel's miss-heavy waves would go ahead of the team waves that carry its
  // longest trajectories (3.5 % longer).  No result depends on it.
  // Kept transitions pay where trajectories come back to their states; one that
  // finds a new state on most hops would write records and bounds that nothing
  // reads.  So an interval ends by general steps once it has found more than K /
  // 2^kPlainShift new states (tested every 64 hops), and a spell of them follows: 2
  // intervals, 8 if the interval after it finds as many again, then
  // kPlainIntervals, each over as soon as an interval
  // of it evaluates fewer (the rest of the one it began in counts as many).  Where the
  // energies follow from the path, the last two states pass on as the general steps'
  // entries (until this did, such an interval ran to its end with transitions: 512 x
  // 4000 hops of S = 109 with records, nearly every hop new, 11.2 ms, now 9.0).  (Spells of 15 always: a trajectory whose first hops find many
  // states spent most of 20,000 hops without leaps.)  20,000 hops of N = 30 (a = I_0 = 1,
  // nearly every hop new): alone 42.8 ms with transitions, 26.4 with this rule
  // (with two states and hops back only, 36.9); N = 56, 4096 of them 114.6, 78.3
  // (90.5).  At 1/2 instead of 1/4 the N = 56 network at 30 kT takes 62.3 ms
  // instead of 42.4; at 1/8 100,000 hops of the N = 30 network at 300 kT 32.3
  // instead of 26.4 ms.  Several chunks: at 1/8 a served population takes 27.4 ms
  // instead of 29.0 at 1/4; at 1/16 S = 109 gains 1 to 3 % and 600 trajectories of S =
  // 148 at 300 kT lose 10.  One-chunk teams, S = 58 at 1 / 300 kT: 1/4 0.92 / 2.84 ms,
  // 1/8 0.92 / 2.61, 1/16 1.15 / 2.46.
  constexpr int kPlainShift = kPathFree ? 2 : 3, kPlainIntervals = 32;
  constexpr int kAlways = 255;   // a spell that does not end (no area)
  constexpr bool kSlowPrio = PRIO && ONE && T == 1;
  int nnew = 0, slowv = 0;
  // intervals left that keep no transitions, and (<< 8) the length of the next such spell
  int plainv = 0;
  if constexpr (!kGeneral) {
    nnew = in_vgpr_i(0);
    slowv = in_vgpr_i(0);
    plainv = in_vgpr_i((area ? 0 : kAlways) | 2 << 8);
  }
  auto base_prio = [&]() __attribute__((always_inline)) {
    if constexpr (kSlowPrio) {
      if (__builtin_amdgcn_readfirstlane(slowv)) __builtin_amdgcn_s_setprio(2);
      else __builtin_amdgcn_s_setprio(1);
    } else {
      __builtin_amdgcn_s_setprio(PRIO ? 1 : 0);
    }
  };

  // ---- states: lane k's occupation words, its record in the area ----------
  uint64_t key[C];
#pragma unroll
  for (int c = 0; c < C; ++c) key[c] = 0;
  const int nslots = kPathFree && ONE ? p.state_slots : STATE_SLOTS;
  int nstates = 0;      // lanes of key[] in use
  int svictim = 0;      // the oldest of them once all are
  // record k in the area: per chunk 64 FP32 row sums, then per chunk 64 FP32 energies
  auto rec = [&](int k) {
    return reinterpret_cast<float*>(area + k * (C * STATE_RECORD_BYTES)) + lane;
  };
  int cur = -1, prev = -1;   // current state (-1: `occ`, not looked up yet) and the one before
  int lastsig = 0;           // what the hop between them toggled (sig below)
  // two records in registers, with their prefixes: states rid's (and its total and
  // rate factor) and pid's
  int rid = -1, pid = -1;
  double rinc[C], pinc[C];
  float rrow[C], rse[C], prow[C], pse[C];
  double rtot = 0.0;
  float rrt = 0.f;
#pragma unroll
  for (int c = 0; c < C; ++c) {
    rinc[c] = pinc[c] = 0.0;
    rrow[c] = rse[c] = prow[c] = pse[c] = 0.f;
  }
  // FP64 prefix over the lane rows of rrow, the total and the rate factor;
  // false: no rate is positive and finite
  auto prefixes = [&]() __attribute__((always_inline)) -> bool {
    double total = 0.0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && 64 * c >= S) {
        rinc[c] = total;
        continue;
      }
      rinc[c] = c == 0 ? wave_scan_f64((double)rrow[c]) : wave_scan_f64((double)rrow[c]) + total;
      total = readlane_f64(rinc[c], 63);
    }
    rtot = in_vgpr(total);
    rrt = __builtin_amdgcn_rcpf((float)total);
    return total > 0.0 && total < INFINITY;
  };
  // the record of state rid becomes state pid's
  auto shelve = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (!kPathFree) pinc[c] = rinc[c];
      prow[c] = rrow[c];
      pse[c] = rse[c];
    }
    pid = rid;
  };

  // ---- transitions, one per lane -----------------------------------------
  constexpr uint64_t kNone = 1ull << 63;   // lane 63: no transition
  int tsrc = -1;                // state it leaves; -1: none
  int tdst = 255;               // state it leads to (255: unknown)
  int tinfo = 0;                // from | to << 8 | one of them is an electrode << 16
  int tsig = 0;                 // the acceptors it toggles (kPathFree: unused)
  uint64_t tout = kNone;        // the transitions out of the state it leads to (lanes)
  float tlo = lane == 63 ? -1.f : INFINITY, thi = INFINITY;   // bounds of u
  float trt = 0.f;              // the clock's rate factor
  int tcnt = 0;                 // hops that took it since the tallies were last brought up
  int tnext = 0;                // the lane a new one takes
  // the transition that took hop (h & ~63) + lane (-1: none, or brought up)
  int jv = -1;
  uint64_t curout = kNone, prevout = kNone;   // the transitions out of cur and prev
  int lastj = -1, lastj2 = -1;  // the one taken last and the one before it (-1: gone)
  // a leap's transitions X -> Y and Y -> X (lanes; -1: none), state X and their
  // bounds and rate factors
  int px = -1, py = -1, sx = -1;
  bool tryleap = false;         // the trajectory goes back and forth between X and Y
  struct Half {
    float lo, hi, rt;
  };
  Half xb{}, yb{};

  // the hops of jv into the clock's rate factors and the transitions' counts
  auto settle = [&]() __attribute__((always_inline)) {
    if constexpr (kGeneral) return;
    uint64_t m = ballot(jv >= 0);
    if (!m) return;
    const int at = jv << 2;
    const float rt = __int_as_float(__builtin_amdgcn_ds_bpermute(at, __float_as_int(trt)));
    if (jv >= 0) rtv = rt;
    // counts matter for electrodes, and for the traffic
    if (!(REC && p.traffic)) {
      const int info = __builtin_amdgcn_ds_bpermute(at, tinfo);
      m &= ballot(info >> 16 != 0);
    }
    while (m) {
      const int j = readlane_i32(jv, lowest_bit(m));
      const uint64_t same = m & ballot(jv == j);
      if (lane == j) tcnt += popcount64(same);
      m &= ~same;
    }
    jv = -1;
  };
  auto flush_clock = [&]() __attribute__((always_inline)) {
    settle();
    time += readlane_f64(wave_scan_f64((double)(lg_lane * rtv)), 63);
    rtv = 0.f;
  };
  // brings the tallies of lane l's transition up
  auto flush_lane = [&](int l) __attribute__((always_inline)) {
    const int n = readlane_i32(tcnt, l);
    const int info = readlane_i32(tinfo, l);
    const int from = info & 255, to = (info >> 8) & 255;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const int s = lane + 64 * c;
      eo[c] += (s == to ? n : 0) - (s == from ? n : 0);
    }
    // net traffic, Go convention (simulation.go:310-311), of tallied hops; whole
    // numbers, so the order of the additions is free
    if (REC && p.traffic && h > prehops && lane == 0 && team.writer()) {
      double* tr = p.traffic + (size_t)t * p.traffic_stride;
      unsafeAtomicAdd(tr + from * S + to, (double)n);
      unsafeAtomicAdd(tr + to * S + from, -(double)n);
    }
  };
  auto flush_tallies = [&]() __attribute__((always_inline)) {
    if constexpr (kGeneral) return;
    settle();
    uint64_t m = ballot(tcnt > 0);
    while (m) {
      const int l = lowest_bit(m);
      m &= m - 1;
      flush_lane(l);
    }
    tcnt = 0;
  };
  auto current_occ = [&]() __attribute__((always_inline)) {
    if constexpr (kGeneral) return;
    if (cur >= 0 && oid != cur) {
#pragma unroll
      for (int c = 0; c < C; ++c) occ[c] = readlane_u64(key[c], cur);
      oid = cur;
    }
  };

  // The row sums of the state with energies se and occupation occ; true: its rows are
  // sources.  (Summed in an array of its own: in the caller's, the compiler holds
  // three chunks as a tuple and copies it at every block's end, 5 % more vector
  // instructions and 2.5 % on the teams that set an uneven batch's length.)
  auto evaluate = [&](float (&rows)[C]) __attribute__((always_inline)) -> bool {
    float R[C];
    // roles of the lanes' sites, as wave-uniform lane masks (scalar ops only):
    // sources = occupied acceptors + electrodes, targets = empty acceptors + electrodes
    uint64_t srcm[C], dstm[C];
    int nocc = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      const uint64_t oc = occ[c] & accm[c];
      srcm[c] = oc | elm[c];
      dstm[c] = (accm[c] ^ oc) | elm[c];
      nocc += popcount64(oc);
    }
    const bool udst = N - nocc <= nocc;   // walk the smaller set (empty vs occupied)
    // every lane sums over the walked members; the sums of lanes outside the
    // other role (and past S) are discarded after the reduction
    uint64_t um[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      R[c] = 0.f;
      um[c] = (udst ? dstm[c] : srcm[c]) & walk[c];
    }
    const float (&v)[C] = se;
    if constexpr (Pol::kElec) {
      if (elec && kMembers) {
        // teams run large networks, where some lane is nearly always in the
        // window: no test
        elec_sums<C, T>(pol, L.P, S, udst, team.wave, v, R);
      } else if (elec) {
        // the lanes whose electrode terms are neither all saturated nor all
        // below 1 (acceptors of the other role); none: the per-lane sums
        const float thr = udst ? vt_max : -vt_min, tlw = udst ? vt_min : -vt_max;
        float x[C];
        uint64_t hi[C], mid = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          x[c] = min_f32(udst ? v[c] : -v[c], 126.f);
          hi[c] = ballot(x[c] >= thr);
          const uint64_t lo = ballot(x[c] < tlw);
          mid |= (udst ? srcm[c] : dstm[c]) & accm[c] & ~(hi[c] | lo);
        }
        if (mid == 0) {
#pragma unroll
          for (int c = 0; c < C; ++c)
            R[c] = __builtin_amdgcn_inverse_ballot_w64(hi[c])
                       ? esum_w[c] : fast_exp2(x[c]) * (udst ? esum_dst[c] : esum_src[c]);
        } else if constexpr (SPLIT) {
          float v1[1] = {v[0]}, R1[1] = {0.f};
#pragma unroll
          for (int c = 1; c < C; ++c)
            if (c == team.wave) v1[0] = v[c];
          elec_sums<1, 1, PolW, C>(*polw, L.P, S, udst, 0, v1, R1);
#pragma unroll
          for (int c = 0; c < C; ++c) R[c] = R1[0];   // (this wave's chunk counts)
        } else {
          elec_sums<C, T>(pol, L.P, S, udst, team.wave, v, R);
        }
      }
    }
    // +1: walked targets, e~_src - e~_dst = v - su; -1: walked sources
    const float sgr = __int_as_float(udst ? (int)0x3f800000 : (int)0xbf800000);
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);
    if constexpr (SPLIT) {
      float v1 = v[0], R1 = R[0];
#pragma unroll
      for (int c = 1; c < C; ++c) {
        if (c == team.wave) {
          v1 = v[c];
          R1 = R[c];
        }
      }
      row_sums_one<C>(*polw, um, v1, se, sgr, R1);
#pragma unroll
      for (int c = 0; c < C; ++c) R[c] = R1;
    } else {
      row_sums<C>(pol, S, um, team.own(), v, se, sgr, R);
    }
    // the team's partial sums alternate between two LDS buffers by reduction
    // (kept states reduce nothing and pass no barrier; the waves agree on
    // every lookup, so they count the same reductions)
    team.reduce(R, nred & 1, lane);
    ++nred;
#pragma unroll
    for (int c = 0; c < C; ++c)
      rows[c] = __builtin_amdgcn_inverse_ballot_w64(udst ? srcm[c] : dstm[c]) ? R[c] : 0.f;
    mark(1);

    // From here to the hop the work is one dependency chain (scans, readlanes,
    // the partner row's LDS loads); the waves sharing a SIMD fill its gaps with
    // their row sums of the walked members.  A raised issue priority lets the
    // chain's instructions go as soon as they are ready: 3 from the scan to the
    // hop, 1 elsewhere, 0 for the row sums.  PRIO false: the variant for
    // launches whose groups queue behind full SIMDs.
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(3);
    return udst;
  };

  // A lane of key[] for a new state: the next free one, else the oldest one that
  // is not the state the trajectory comes from; the transitions out of the state
  // that leaves go, those into it lose their end.
  auto take_state = [&]() __attribute__((always_inline)) -> int {
    if (nstates < nslots) return nstates++;
    int v = svictim;
    if (v == prev) v = v + 1 == nslots ? 0 : v + 1;
    svictim = v + 1 == nslots ? 0 : v + 1;
    // (their hops still count: a lane keeps its ends and counts until it is taken again)
    const uint64_t gone = ballot(tsrc == v);
    if (tsrc == v) tsrc = -1;
    if (tdst == v) tdst = 255;
    tout &= ~gone;
    prevout &= ~gone;
    px = py = -1;
    tryleap = false;
    return v;
  };

  // Energies of the state with occupation occ from the last recompute's: those plus the
  // Coulomb columns of the acceptors whose occupation differs from the recompute's
  // (+ where now occupied, - where now empty), added in ascending site order; the
  // columns of up to G sites are loaded together (a site past the last loads the
  // first's column and adds nothing).
  auto base_energies = [&]() __attribute__((always_inline)) {
    if constexpr (kPathFree) {
      constexpr int G = 8;
      se[0] = base_se[0];
      uint64_t dm = (occ[0] ^ base_occ[0]) & accm[0];
      while (dm) {
        int js[G];
        const int j0 = __builtin_ctzll(dm);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          js[g] = dm ? __builtin_ctzll(dm) : -1;
          dm &= dm - 1;
        }
        float cv[G];
#pragma unroll
        for (int g = 0; g < G; ++g) cv[g] = pol.coul(js[g] < 0 ? j0 : js[g], 0);
#pragma unroll
        for (int g = 0; g < G; ++g) {
          if (js[g] < 0) break;
          const bool on = (occ[0] >> js[g]) & 1ull;
          se[0] += on ? cv[g] : -cv[g];
        }
      }
    }
  };
  // ... from the energies of the state before it.
  auto rank1_energies = [&](const float (&bse)[C]) __attribute__((always_inline)) {
    const bool src_acc = psrc < N, dst_acc = pdst < N;
    float cs[C], cd[C];
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if constexpr (Pol::kZeroColumnN) {   // column N holds c = 0: no select per lane
        cs[c] = (c == 0 || 64 * c < S) ? pol.coul(min((unsigned)psrc, (unsigned)N), c) : 0.f;
        cd[c] = (c == 0 || 64 * c < S) ? pol.coul(min((unsigned)pdst, (unsigned)N), c) : 0.f;
      } else {
        cs[c] = (c == 0 || 64 * c < S) && src_acc ? pol.coul(psrc, c) : 0.f;
        cd[c] = (c == 0 || 64 * c < S) && dst_acc ? pol.coul(pdst, c) : 0.f;
      }
    }
#pragma unroll
    for (int c = 0; c < C; ++c) se[c] = (bse[c] - cs[c]) + cd[c];
  };

  // The current state (occupation occ) looked up or evaluated; false: it has no
  // positive finite rate.
  auto resolve = [&]() __attribute__((always_inline)) -> bool {
    if constexpr (kPathFree) {
      const uint64_t m = ballot(key[0] == occ[0]) & (nstates < 64 ? (1ull << nstates) - 1 : ~0ull);
      if (m) {
        cur = lowest_bit(m);
      } else {
        base_energies();
      }
    } else if (pend) {
      // the previous state's energies plus the last hop's rank-1 update
      // (both Coulomb columns loaded together; an electrode end
      // contributes 0); after a recompute, the recomputed ones
      float bse[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        bse[c] = rid == prev ? rse[c] : pse[c];
        if (rid != prev && pid != prev && (c == 0 || 64 * c < S)) bse[c] = rec(prev)[64 * (C + c)];
      }
      rank1_energies(bse);
    }
    if (cur >= 0) {
      curout = ballot(tsrc == cur) | kNone;
      if constexpr (PH) ++ph[10];
      mark(1);
    } else {
      nnew = in_vgpr_i(nnew + 1);
      const int k = take_state();
      if (rid == prev) shelve();   // (else pid is prev, or there is none)
      (void)evaluate(rrow);
#pragma unroll
      for (int c = 0; c < C; ++c) rse[c] = se[c];
      if (!prefixes()) return false;
#pragma unroll
      for (int c = 0; c < C; ++c)
        if (lane == k) key[c] = occ[c];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (c > 0 && 64 * c >= S) break;
        rec(k)[64 * c] = rrow[c];
        rec(k)[64 * (C + c)] = rse[c];
      }
      wave_lds_sync();   // (memory order within the wave)
      if (pid == k) pid = -1;
      rid = cur = k;
      curout = kNone;
      mark(2);
    }
    oid = cur;
    if (lane == lastj) {
      tdst = cur;
      tout = curout;
    }
    return true;
  };

  // A hop whose transition is not kept: the general selection.  The transition's
  // lane (and its ends and what it toggles), or -1: no partner has a positive rate.
  auto new_transition = [&](int& src, int& dst, int& sig) __attribute__((always_inline)) -> int {
    if (rid != cur) {
      // (one-chunk kernels are held to 128 VGPRs: they form the prefixes again)
      const bool held = pid == cur, whole = !kPathFree && held;
      double inc[C];
      float row[C], e[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        inc[c] = whole ? pinc[c] : 0.0;
        row[c] = prow[c];
        e[c] = pse[c];
        if (!held) {
          row[c] = c > 0 && 64 * c >= S ? 0.f : rec(cur)[64 * c];
          e[c] = c > 0 && 64 * c >= S ? 0.f : rec(cur)[64 * (C + c)];
        }
      }
      shelve();
#pragma unroll
      for (int c = 0; c < C; ++c) {
        rinc[c] = inc[c];
        rrow[c] = row[c];
        rse[c] = e[c];
      }
      rid = cur;
      if (whole) {   // the total from its prefix
        const double total = readlane_f64(rinc[C - 1], 63);
        rtot = in_vgpr(total);
        rrt = __builtin_amdgcn_rcpf((float)total);
      } else {
        (void)prefixes();
      }
    }
    current_occ();
    int nocc = 0;
#pragma unroll
    for (int c = 0; c < C; ++c) nocc += popcount64(occ[c] & accm[c]);
    const bool udst = N - nocc <= nocc;
    if constexpr (PRIO) __builtin_amdgcn_s_setprio(3);
    const double target = readlane_f64(in_vgpr(ue_lane * rtot), h & 63);
    double exc[C];   // the prefix before the lane
#pragma unroll
    for (int c = 0; c < C; ++c) exc[c] = rinc[c] - (double)rrow[c];

    // the selected lane l and the remainder rr = target - (incl - R) at l, formed
    // on every lane (FP64 difference, rounded to FP32) and read from l
    int sel = -1;
    float rr = 0.f;
    double lo = -INFINITY, hi = 0.0, exs = 0.0;
    bool keep = true;   // the bounds describe the selection
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && 64 * c >= S) break;
      const uint64_t m = ballot(rinc[c] > target);
      if (sel < 0 && m) {
        const int l = __builtin_ctzll(m);
        sel = 64 * c + l;
        rr = readlane_as_f32(target - exc[c], l);
        hi = readlane_f64(rinc[c], l);
        exs = readlane_f64(exc[c], l);
        if (l > 0) lo = readlane_f64(rinc[c], l - 1) * (1.0 + 0x1p-48);
      } else if (sel < 0) {
        lo = readlane_f64(rinc[c], 63) * (1.0 + 0x1p-48);
      }
    }
    if (sel < 0) {   // target rounded onto the total: last lane with a nonzero row
      keep = false;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (c > 0 && 64 * c >= S) break;
        const uint64_t m = ballot(rrow[c] > 0.f);
        if (m) {
          const int l = 63 - __builtin_clzll(m);
          sel = 64 * c + l;
          rr = readlane_as_f32(target - exc[c], l);
        }
      }
    }
    mark(3);

    // partner of `sel`: the prefix of its row over the lanes in site order (a
    // lane-parallel pass over the row)
    const float s_sel = pick_lane_value<C>(rse, sel);
    // sign of the lane-parallel difference: a scalar constant
    const float sg = __int_as_float(udst ? (int)0xbf800000 : (int)0x3f800000);
    const typename Pol::Pre pre = pol.prefetch(sel);
    float run = 0.f, plo = -INFINITY, phi = 0.f;
    int pick = -1, last_nz = -1;
#pragma unroll
    for (int c = 0; c < C; ++c) {
      if (c > 0 && 64 * c >= S) break;
      // partners: targets of a source row, sources of a target row
      const uint64_t oc = occ[c] & accm[c];
      const uint64_t inu = (udst ? accm[c] ^ oc : oc) | elm[c];
      // udst ? s_sel - se : se - s_sel (the sign is exact)
      float r = fast_exp2(pol.pair(pre, c, rse[c] - s_sel, sg));
      r = __builtin_amdgcn_inverse_ballot_w64(inu) ? r : 0.f;
      const float pcum = wave_scan_f32(r) + run;
      const uint64_t pnz = ballot(r > 0.f);
      run = readlane_f32(pcum, 63);
      const uint64_t hit = pnz & ballot(pcum > rr);
      if (pick < 0) {
        if (pnz) last_nz = 64 * c + 63 - __builtin_clzll(pnz);
        if (hit) {
          const int l = __builtin_ctzll(hit);
          pick = 64 * c + l;
          phi = readlane_f32(pcum, l);
          if (l > 0) plo = readlane_f32(pcum, l - 1) * (1.f + 0x1p-19f);
        } else {
          plo = run * (1.f + 0x1p-19f);
        }
      }
    }
    if (pick < 0) {
      keep = false;
      pick = last_nz;
    }
    if (pick < 0) return -1;
    mark(4);
    src = udst ? sel : pick;
    dst = udst ? pick : sel;

    // the bounds of u, rounded inwards (a, b: of the target)
    double a = lo, b = hi;
    if (plo > 0.f) a = fmax(a, (exs + (double)plo * (1.0 + 0x1p-20)) * (1.0 + 0x1p-51));
    b = fmin(b, (exs + (double)phi * (1.0 - 0x1p-20)) * (1.0 - 0x1p-51));
    float ul = -1.f, uh = (float)b * rrt * (1.f - 0x1p-20f);
    // (uniforms are multiples of 2^-53: 1e-17 bounds the positive ones)
    if (a > 0.0) ul = fmaxf(fmaxf((float)a, 0x1p-126f) * rrt * (1.f + 0x1p-20f), 1e-17f);
    // totals whose reciprocal leaves FP32's normal range: not kept
    if (!(rrt > 1e-30f && rrt < 1e30f) || !keep) ul = INFINITY;

    // into the next lane
    const int j = tnext;
    tnext = tnext == 62 ? 0 : tnext + 1;
    if (ballot(jv == j)) settle();
    if (readlane_i32(tcnt, j) > 0) flush_lane(j);
    if (j == px || j == py) px = py = -1;
    if (j == lastj) lastj = -1;
    // lane j no longer leaves the state it left, but the current one
    const uint64_t bit = 1ull << j;
    curout |= bit;
    if (prev != cur) prevout &= ~bit;
    tout = tdst == cur ? tout | bit : tout & ~bit;
    if (lane == j) {
      tsrc = cur;
      tdst = 255;
      tinfo = src | dst << 8 | (src >= N || dst >= N ? 1 << 16 : 0);
      tcnt = 0;
      tlo = ul;
      thi = uh;
      trt = rrt;
    }
    if constexpr (!kPathFree) {
      const int x = src < N ? src : 255, y = dst < N ? dst : 255;
      sig = x < y ? x | y << 8 : y | x << 8;
      if (lane == j) tsig = sig;
    }
    base_prio();
    return j;
  };

  // Takes the hop of transition j from the current state into kept state d, which
  // the transitions `out` leave, or (255) into one still to be looked up.
  auto take = [&](int j, int d, uint64_t out) __attribute__((always_inline)) {
    jv = writelane_i32(j, h, jv);
    if (REC && h >= prehops) {
      // exponential waiting time -ln(1-u)/total, an FP32 quotient
      const double dt = (double)readlane_f32(lg_lane * readlane_f32(trt, j), h & 63);
      const int info = readlane_i32(tinfo, j);
      const int from = info & 255, to = (info >> 8) & 255;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        uint64_t oc = readlane_u64(key[c], cur);
        if (p.post_hop_record) {
          if ((from >> 6) == c) oc &= ~(1ull << (from & 63));
          if ((to >> 6) == c) oc |= 1ull << (to & 63);
        }
        if (__builtin_amdgcn_inverse_ballot_w64(oc & accm[c])) ot[c] += dt;
      }
    }
    if constexpr (PH) {
      // a hop from a state that the hop before led back into
      if (ph_back) ++ph[7];
      ph_back = prev >= 0 && d == prev;
    }
    prev = cur;
    cur = d;
    prevout = curout;
    curout = out;
    lastj2 = lastj;
    lastj = j;
    ++h;
  };
  // Where transition j leads: a hop back into the state before the last hop takes
  // that state as it was.
  auto end_of = [&](int j, uint64_t& out) __attribute__((always_inline)) -> int {
    int d = readlane_i32(tdst, j);
    out = readlane_u64(tout, j);
    if constexpr (!kPathFree) {
      const int sig = readlane_i32(tsig, j);
      if (prev >= 0 && sig == lastsig) {
        d = prev;
        out = prevout;
      }
    }
    return d;
  };
  // The hop of transition j (its ends, and what it toggles) into a state it has
  // not reached before: the occupation, looked up or evaluated when the next hop
  // needs it.
  auto take_unknown = [&](int j, int from, int to, int sig) __attribute__((always_inline)) {
    int d = 255;
    uint64_t out = kNone;
    if constexpr (!kPathFree) {
      if (prev >= 0 && sig == lastsig) {
        d = prev;
        out = prevout;
      }
      lastsig = sig;
    }
    if (d == 255) {
      current_occ();
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if ((from >> 6) == c) occ[c] &= ~(1ull << (from & 63));
        if (to < N && (to >> 6) == c) occ[c] |= 1ull << (to & 63);
      }
      oid = -1;
      if constexpr (kPathFree) {
        // the state before the last hop needs no lookup
        if (prev >= 0 && occ[0] == readlane_u64(key[0], prev)) {
          d = oid = prev;
          out = prevout;
          if (lane == j) {
            tdst = d;
            tout = out;
          }
        }
      }
      psrc = from;
      pdst = to;
      pend = true;
    }
    take(j, d, out);
    if (cur == 255) cur = -1;
  };
  // The last two hops went back and forth by transitions y = lastj and x =
  // lastj2: their bounds for the leap.
  auto load_pair = [&](int x, int y) __attribute__((always_inline)) {
    if ((px == x && py == y) || (px == y && py == x)) return;
    auto half = [&](int l) {
      return Half{in_vgpr(readlane_f32(tlo, l)), in_vgpr(readlane_f32(thi, l)),
                  in_vgpr(readlane_f32(trt, l))};
    };
    px = x;
    py = y;
    sx = cur;
    xb = half(px);
    yb = half(py);
  };

  // The run of hops back and forth between X and Y from here, applied at once;
  // the hops taken (0: the next hop is another one).
  auto leap = [&]() __attribute__((always_inline)) -> int {
    const int hl = h & 63;
    const uint64_t okx = ballot(uf_lane >= xb.lo) & ballot(uf_lane < xb.hi);
    const uint64_t oky = ballot(uf_lane >= yb.lo) & ballot(uf_lane < yb.hi);
    // lanes k that start their hop in X: k - hl even when X is the current state
    const bool fromx = cur == sx;
    const uint64_t inx = ((hl & 1) != 0) != fromx ? 0x5555555555555555ull : 0xAAAAAAAAAAAAAAAAull;
    const uint64_t run = ((okx & inx) | (oky & ~inx)) >> hl;
    // trailing ones (s_ff1 of an all-ones complement is -1: the whole block)
    int n = lowest_bit(~run);
    const int nmax = 64 - hl < h_lim - h ? 64 - hl : h_lim - h;
    if ((unsigned)n > (unsigned)nmax) n = nmax;
    if (n == 0) return 0;
    const uint64_t lanes = (~0ull << hl) & (hl + n < 64 ? ~(~0ull << (hl + n)) : ~0ull);
    const float rtl = __builtin_amdgcn_inverse_ballot_w64(inx) ? xb.rt : yb.rt;
    if (__builtin_amdgcn_inverse_ballot_w64(lanes)) rtv = rtl;
    const int nx = popcount64(lanes & inx);
    tcnt += (lane == px ? nx : 0) + (lane == py ? n - nx : 0);
    if (REC && h >= prehops) {   // (a run ends where the prehops do)
      const int oth = fromx ? readlane_i32(tsrc, py) : sx;
      const int sa = p.post_hop_record ? oth : cur, sb = p.post_hop_record ? cur : oth;
      bool a[C], b[C];
#pragma unroll
      for (int c = 0; c < C; ++c) {
        a[c] = __builtin_amdgcn_inverse_ballot_w64(readlane_u64(key[c], sa) & accm[c]);
        b[c] = __builtin_amdgcn_inverse_ballot_w64(readlane_u64(key[c], sb) & accm[c]);
      }
      const float dtl = lg_lane * rtl;
      int k = 0;
      for (; k + 2 <= n; k += 2) {
        const double d0 = (double)readlane_f32(dtl, hl + k), d1 = (double)readlane_f32(dtl, hl + k + 1);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          if (a[c]) ot[c] += d0;
          if (b[c]) ot[c] += d1;
        }
      }
      if (k < n) {
        const double d0 = (double)readlane_f32(dtl, hl + k);
#pragma unroll
        for (int c = 0; c < C; ++c)
          if (a[c]) ot[c] += d0;
      }
    }
    if constexpr (PH) {
      ph[7] += n;
      ph[8] += n;
      ph[9] += n;
      ph_back = true;
    }
    h += n;
    // n odd: the other state, by the transition out of the one it was in
    const bool atx = fromx == ((n & 1) == 0);
    lastj = atx ? py : px;
    lastj2 = atx ? px : py;
    if (n & 1) {
      const int oth = fromx ? readlane_i32(tsrc, py) : sx;
      prev = cur;
      cur = oth;
      const uint64_t out = curout;
      curout = prevout;
      prevout = out;
    }
    return n;
  };

  // The kept states and transitions go (their tallies are brought up).
  auto drop_kept = [&]() __attribute__((always_inline)) {
    if constexpr (kGeneral) return;
#pragma unroll
    for (int c = 0; c < C; ++c) key[c] = 0;
    tout = curout = prevout = kNone;
    tdst = 255;
    oid = -1;
    tsrc = jv = cur = prev = rid = pid = lastj = lastj2 = px = py = -1;
    tinfo = tsig = tcnt = 0;
    tlo = lane == 63 ? -1.f : INFINITY;
    thi = INFINITY;
    trt = 0.f;
    tryleap = false;
    nstates = svictim = tnext = 0;
    if constexpr (PH) ph_back = false;
  };
  // The work of a special hop but for the recompute: the clock's block sum,
  // uniforms, the end of the prehops.
  auto block_work = [&]() __attribute__((always_inline)) {
    flush_clock();
    if ((h & 63) == 0) refill(h);
    if (h == prehops) {
      time = 0.0;
      tcnt = 0;   // (settled by the clock's flush)
#pragma unroll
      for (int c = 0; c < C; ++c) {
        eo[c] = 0;
        ot[c] = 0.0;
      }
    }
  };
  // A spell of general steps begins (more: intervals besides its length); the next
  // one is four times as long.
  auto next_spell = [&](int spell, int more) __attribute__((always_inline)) -> int {
    const int n = spell >> 8;
    return (n + more) | (n < kPlainIntervals ? 4 * n : n) << 8;
  };
  // The work of a special hop before the hop itself: the clock's block sum,
  // uniforms, the end of the prehops, the FP64 recompute (which drops the kept
  // states and transitions).
  // false: the launch's time limit has passed at this recompute point, and the
  // trajectory stops here (a multiple of the recompute interval, from which a
  // resumed range continues exactly as one long launch would).  The waves of a
  // team by members read their clocks apart and could disagree, so those carry no
  // limit (the host refuses one).
  // empty: what else the recompute empties, here (the general steps' entries, reset
  // ahead of this call, stayed live through the recompute: 30 to 44 VGPRs of the
  // kernels over several chunks).
  auto special_work = [&](auto empty) __attribute__((always_inline)) -> bool {
    if (!kMembers && p.time_limit > 0 && h == next_rc && h > h_begin) {
      bool over = wall_clock64() - t_start > p.time_limit;
      if constexpr (SPLIT) {
        // wave 0's clock decides (its next word follows the barrier of the first
        // evaluation after this recompute)
        if (team.wave == 0) *team.flag = over;
        __syncthreads();
        over = __builtin_amdgcn_readfirstlane(*team.flag) != 0;
      }
      if (over) {
        h_stop = h;
        h_lim = h;
        return false;
      }
    }
    block_work();
    if (h == next_rc) {
      current_occ();
      recompute_energies<C>(se, occ, L, es, lane);
#pragma unroll
      for (int c = 0; c < C; ++c) {
        base_se[c] = se[c];
        base_occ[c] = occ[c];
      }
      next_rc = next_multiple(h);
      pend = false;
      empty();
      if constexpr (!kGeneral) {
        flush_tallies();
        drop_kept();
        const int spell = __builtin_amdgcn_readfirstlane(plainv), left = spell & 255;
        const int nn = __builtin_amdgcn_readfirstlane(nnew);
        if (left > 0) {
          if (left != kAlways) plainv = in_vgpr_i(nn > K >> kPlainShift ? spell - 1 : spell - left);
        } else {
          if constexpr (kSlowPrio) slowv = in_vgpr_i(nn > 16 ? 1 : 0);
          plainv = in_vgpr_i(nn > K >> kPlainShift ? next_spell(spell, 0) : 2 << 8);
        }
        nnew = in_vgpr_i(0);
      }
      base_prio();
    } else if constexpr (!kGeneral && !PH) {
      if (__builtin_amdgcn_readfirstlane(nnew) > K >> kPlainShift) {
        current_occ();
        flush_tallies();
        if constexpr (kPathFree) drop_kept();
        if constexpr (kSlowPrio) slowv = in_vgpr_i(1);
        // (the rest of this interval besides)
        plainv = in_vgpr_i(next_spell(__builtin_amdgcn_readfirstlane(plainv), 1));
        // (the interval has found that many, whatever its rest evaluates)
        nnew = in_vgpr_i((K >> kPlainShift) + 1);
      }
    }
    special = next_special(h, false);
    h_lim = special < h_stop ? special : h_stop;
    mark(0);
    return true;
  };

  // The hops up to the next recompute by general steps, which keep the current
  // state and the one before it, in registers, and no transitions.  Within an interval,
  // where the energies follow from the path, they go on from the kept ones.  The entries
  // swap roles on every hop; the loop is unrolled by two hops, one for each
  // assignment of the roles, so a hop back moves no data.  (The tables of kept
  // states and transitions hold nothing here, and no registers.)
  auto general = [&]() __attribute__((always_inline)) {
    struct Entry {
      uint64_t key[C];   // occupation words
      uint64_t nzr[C];   // lanes whose row sum is nonzero (in VGPRs: used on rare hops)
      uint64_t pnz[C];   // lanes whose rate in row psel is nonzero
      double tot;        // total rate, in a VGPR
      float rtot;        // its reciprocal, the clock's rate factor, in a VGPR
      double inc[C];     // FP64 inclusive prefix of the row sums over lanes
      double exc[C];     // inc - row sum: the prefix before the lane
      float se[C];       // FP32 site energies of the state
      float pcum[C];     // FP32 prefix of row psel's rates over its partners, in site order
      int psel;          // lane of that row (-2: none yet; never a lane or the -1 of no lane)
      int udst;          // rows are sources, the walked set is the targets
      int val;
    };
    // The partner prefix of row `sel` of F's state into F: the prefix of the
    // row's rates over the lanes in site order, and the lanes whose rate is
    // nonzero (a lane-parallel pass over the row).
    auto partner_pass = [&](Entry& F, int sel) __attribute__((always_inline)) {
      uint64_t inu[C];   // partners: targets of a source row, sources of a target row
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint64_t o = occ[c] & accm[c];
        inu[c] = (F.udst ? accm[c] ^ o : o) | elm[c];
      }
      const float s_sel = pick_lane_value<C>(F.se, sel);
      // sign of the lane-parallel difference: a scalar constant
      const float sg = __int_as_float(F.udst ? (int)0xbf800000 : (int)0x3f800000);
      const typename Pol::Pre pre = pol.prefetch(sel);
      float run = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        F.pcum[c] = 0.f;
        F.pnz[c] = 0;
        if (c > 0 && 64 * c >= S) continue;
        // udst ? s_sel - se : se - s_sel (the sign is exact)
        float r = fast_exp2(pol.pair(pre, c, F.se[c] - s_sel, sg));
        r = __builtin_amdgcn_inverse_ballot_w64(inu[c]) ? r : 0.f;
        F.pcum[c] = wave_scan_f32(r) + run;
        F.pnz[c] = ballot(r > 0.f);
        run = readlane_f32(F.pcum[c], 63);
      }
      F.psel = sel;
    };

    // One hop from the current state F (its entry valid); B: the other entry.
    // Returns 1 when the state it leads to is B's, 0 when that state is new,
    // -1 when the trajectory stops.
    auto hop = [&](Entry& F, const Entry& B) __attribute__((always_inline)) -> int {
      if constexpr (PRIO) __builtin_amdgcn_s_setprio(3);
      // exponential waiting time -ln(1-u)/total, an FP32 quotient
      const double dt = REC ? (double)readlane_f32(lg_lane * F.rtot, h & 63) : 0.0;
      // event uniform x total, multiplied on every lane and read from this hop's
      const double target = readlane_f64(ue_lane * F.tot, (int)(h & 63));

      // the selected lane l and the remainder rr = target - (incl - R) at l, formed
      // on every lane (FP64 difference, rounded to FP32) and read from l
      int sel = -1;
      float rr = 0.f;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        const uint64_t m = ballot(F.inc[c] > target);
        if (sel < 0 && m) {
          const int l = __builtin_ctzll(m);
          sel = 64 * c + l;
          rr = readlane_as_f32(target - F.exc[c], l);
        }
      }
      if (sel < 0) {   // target rounded onto the total: last lane with a nonzero row
#pragma unroll
        for (int c = 0; c < C; ++c) {
          const uint64_t m = uniform_u64(F.nzr[c]);
          if (m) {
            const int l = 63 - __builtin_clzll(m);
            sel = 64 * c + l;
            rr = readlane_as_f32(target - F.exc[c], l);
          }
        }
      }
      mark(3);

      // partner of `sel`: the prefix of its row over the lanes in site order (and
      // the lanes whose rate is nonzero), from the entry when it was formed for
      // the same row, else by a lane-parallel pass over the row
      if (sel != F.psel) {
        partner_pass(F, sel);
      } else if constexpr (PH) {
        ++ph[8];
      }
      int pick = -1, last_nz = -1;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (c > 0 && 64 * c >= S) break;
        const uint64_t hit = F.pnz[c] & ballot(F.pcum[c] > rr);
        if (pick < 0) {
          if (F.pnz[c]) last_nz = 64 * c + 63 - __builtin_clzll(F.pnz[c]);
          if (hit) pick = 64 * c + __builtin_ctzll(hit);
        }
      }
      if (pick < 0) pick = last_nz;
      if (pick < 0) return -1;
      mark(4);
      base_prio();
      const int src = F.udst ? sel : pick;
      const int dst = F.udst ? pick : sel;
      const bool tally = h >= prehops;

      if (REC && tally && !p.post_hop_record) {
#pragma unroll
        for (int c = 0; c < C; ++c)
          if (__builtin_amdgcn_inverse_ballot_w64(occ[c] & accm[c])) ot[c] += dt;
      }
      // net traffic, Go convention (simulation.go:310-311)
      if (REC && p.traffic && tally && lane == 0 && team.writer()) {
        double* tr = p.traffic + (size_t)t * p.traffic_stride;
        unsafeAtomicAdd(tr + src * S + dst, 1.0);
        unsafeAtomicAdd(tr + dst * S + src, -1.0);
      }
      // perform hop: occupation (acceptors live in the words of the C chunks),
      // tallies; a new state's energies are formed when it is evaluated
      const bool src_acc = src < N, dst_acc = dst < N;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        // the source's bit is cleared whether it is an acceptor or not: bits of
        // electrode sites are never set (a one-chunk kernel has S <= 64 sites)
        if (C == 1 || (src >> 6) == c) occ[c] &= ~(1ull << (src & 63));
        if (dst_acc && (C == 1 || (dst >> 6) == c)) occ[c] |= 1ull << (dst & 63);
      }
      psrc = src;
      pdst = dst;
      // electrode tallies (a wave-uniform branch: most hops join two acceptors);
      // they move on the lanes of both ends; only electrode lanes' are kept
      if (__builtin_expect(!src_acc || !dst_acc, 0)) {
#pragma unroll
        for (int c = 0; c < C; ++c) {
          if (lane + 64 * c == src) eo[c] -= 1;
          if (lane + 64 * c == dst) eo[c] += 1;
        }
      }
      if (REC && tally && p.post_hop_record) {
#pragma unroll
        for (int c = 0; c < C; ++c)
          if (__builtin_amdgcn_inverse_ballot_w64(occ[c] & accm[c])) ot[c] += dt;
      }
      if (lane == (h & 63)) rtv = F.rtot;
      mark(5);
      bool same = B.val != 0;
#pragma unroll
      for (int c = 0; c < C; ++c) same = same && B.key[c] == occ[c];
      return same ? 1 : 0;
    };

    Entry E0, E1;
    E0.val = E1.val = 0;
    bool cur_ok = false;   // the current state's entry holds it
    // The prefix over F's rows R, its total and what follows from them into F;
    // false: no rate is positive and finite.
    auto sums = [&](Entry& F, const float (&R)[C]) __attribute__((always_inline)) -> bool {
      double total = 0.0;
#pragma unroll
      for (int c = 0; c < C; ++c) {
        if (c > 0 && 64 * c >= S) {
          F.inc[c] = F.exc[c] = total;
          F.nzr[c] = in_vgpr((uint64_t)0);
          continue;
        }
        F.inc[c] = c == 0 ? wave_scan_f64((double)R[c]) : wave_scan_f64((double)R[c]) + total;
        F.exc[c] = F.inc[c] - (double)R[c];
        F.nzr[c] = in_vgpr(ballot(R[c] > 0.f));
        total = readlane_f64(F.inc[c], 63);
      }
      F.tot = in_vgpr(total);
      F.rtot = __builtin_amdgcn_rcpf((float)total);
      F.psel = -2;
      F.val = 1;
      return total > 0.0 && total < INFINITY;
    };
    if constexpr (!kGeneral && !kPathFree) {
      // kept state k into F
      auto hand_over = [&](Entry& F, int k) __attribute__((always_inline)) {
        float R[C];
        int nocc = 0;
#pragma unroll
        for (int c = 0; c < C; ++c) {
          F.key[c] = readlane_u64(key[c], k);
          nocc += popcount64(F.key[c] & accm[c]);
          R[c] = k == rid ? rrow[c] : prow[c];
          F.se[c] = k == rid ? rse[c] : pse[c];
          if (k != rid && k != pid) {
            R[c] = c > 0 && 64 * c >= S ? 0.f : rec(k)[64 * c];
            F.se[c] = c > 0 && 64 * c >= S ? 0.f : rec(k)[64 * (C + c)];
          }
        }
        F.udst = N - nocc <= nocc;
        (void)sums(F, R);
      };
      if (prev >= 0) hand_over(E1, prev);
      if (cur >= 0) {
        hand_over(E0, cur);
        cur_ok = true;
      }
      drop_kept();
    }
    // One hop whose current state's entry is F (B: the entry of the state
    // before); false: the trajectory stops here, its range ends or the next hop
    // starts with a recompute.
    auto step = [&](Entry& F, Entry& B) __attribute__((always_inline)) -> bool {
      if constexpr (kGeneral) {
        if (__builtin_expect(h == special, 0) && !special_work([&]() __attribute__((always_inline)) {
              cur_ok = false;
              E0.val = E1.val = 0;
            }))
          return false;
      }
      if (!cur_ok) {
        if constexpr (!kGeneral) nnew = in_vgpr_i(nnew + 1);
        if constexpr (kPathFree) base_energies();
        else if (pend) rank1_energies(B.se);
        float R[C];
        F.udst = evaluate(R);
#pragma unroll
        for (int c = 0; c < C; ++c) {
          F.key[c] = occ[c];
          F.se[c] = se[c];
        }
        const bool ok = sums(F, R);
        mark(2);
        if (!ok) {
          status = ST_ZERO_RATE;
          return false;
        }
      } else if constexpr (PH) {
        ++ph[7];
      }
      const int r = hop(F, B);
      if (r < 0) {
        status = ST_ZERO_RATE;
        return false;
      }
      cur_ok = r > 0;
      pend = true;
      ++h;
      mark(5);
      if constexpr (kGeneral) return h < h_stop;
      if (h < h_lim) return true;
      if (h >= h_stop || h == next_rc) return false;
      block_work();
      special = next_special(h, false);
      h_lim = special < h_stop ? special : h_stop;
      mark(0);
      return true;
    };
    for (;;) {
      if (!step(E0, E1)) break;
      if (!step(E1, E0)) break;
    }
    if constexpr (!kGeneral) drop_kept();
  };

  base_prio();
  if constexpr (kGeneral) {
    if (h < h_stop) general();
  }
  while (!kGeneral && h < h_stop) {
    if (h == special && !special_work([] {})) break;
    if (__builtin_amdgcn_readfirstlane(plainv) & 255) {
      general();
      if (status != ST_OK) break;
      continue;
    }
    if constexpr (!kGeneral) {
      if (cur < 0 && !resolve()) {
        status = ST_ZERO_RATE;
        break;
      }
      // hops of this uniform block from kept states
      while (h < h_lim && cur >= 0) {
        if (tryleap) {
          const int n = leap();
          tryleap = n > 0 && h == h_lim;   // the block's end, not the run's, ended it
          mark(6);
          if (n > 0) continue;
        }
        // hops by kept transitions, in a loop of its own: the transitions whose
        // bounds hold the hop's uniform (whatever state they leave; the next hop's
        // are formed while this hop's chain runs), of them the one out of the
        // current state, and where it leads.  A wave pays about 5 cycles for an
        // instruction here and 28 for a value that crosses from the vector to the
        // scalar unit and back.
        auto pass = [&](int hh) __attribute__((always_inline)) -> uint64_t {
          const float u = readlane_f32(uf_lane, hh & 63);
          return ballot(u >= tlo) & ballot(u < thi);
        };
        int j = 63;
        bool stop = true, alternate = false;
        if (curout != kNone) {   // (a state none leaves: a new transition)
          uint64_t in = pass(h);
          for (;;) {
            j = lowest_bit(in & curout);
            in = pass(h + 1);
            uint64_t out;
            const int d = end_of(j, out);
            if (__builtin_expect(d == 255, 0)) break;
            if constexpr (!kPathFree) lastsig = readlane_i32(tsig, j);
            if constexpr (PH) ++ph[8];
            const int j2 = lastj2, p0 = prev;
            take(j, d, out);
            if (h >= h_lim) {
              stop = false;
              break;
            }
            // back and forth by the same two transitions
            if (__builtin_expect(j == j2, 0) && d == p0 && lastj2 >= 0) {
              stop = false;
              alternate = true;
              break;
            }
          }
        }
        mark(6);
        if (alternate) {
          load_pair(lastj2, lastj);
          tryleap = true;
        }
        if (!stop) continue;
        int from, to, sig = 0;
        if (j == 63) {
          j = new_transition(from, to, sig);
          if (j < 0) {
            status = ST_ZERO_RATE;
            h_stop = h;
            break;
          }
        } else {
          const int info = readlane_i32(tinfo, j);
          from = info & 255;
          to = (info >> 8) & 255;
          if constexpr (!kPathFree) sig = readlane_i32(tsig, j);
          if constexpr (PH) ++ph[8];
        }
        take_unknown(j, from, to, sig);
        mark(5);
      }
    }
  }
  if constexpr (PRIO) __builtin_amdgcn_s_setprio(0);   // a stopped trajectory leaves the loop raised
  flush_clock();
  flush_tallies();
  current_occ();
  if (!team.writer()) return;
  if constexpr (PH) {
    if (p.phases && lane == 0)
      for (int k = 0; k < FP32_PHASES; ++k)
        atomicAdd(reinterpret_cast<unsigned long long*>(p.phases + k), (unsigned long long)ph[k]);
  }
  if (lane == 0) {
    const int64_t dt_ticks = wall_clock64() - t_start;
    o->ticks = (int32_t)(dt_ticks < INT32_MAX ? dt_ticks : INT32_MAX);
    o->time = time;
    o->hops_done = h > prehops ? h - prehops : 0;
    o->status = status;
#pragma unroll
    for (int w = 0; w < OCCW; ++w) o->occ[w] = w < C ? occ[w] : 0ull;
  }
#pragma unroll
  for (int c = 0; c < C; ++c) {
    const int s = lane + 64 * c;
    if (s >= N && s < S) o->eo[s - N] = eo[c];
    if (REC && p.occ_time && s < N) p.occ_time[(size_t)t * NMAX + s] = ot[c];
  }
}

}  // namespace kmc
