// Plain-old-data records shared by the host library and the kernels.
//
// A *layout* is one network geometry (acceptor + electrode positions and the
// constant tables derived from them); an *energy set* is one set of site
// constants E_constant[N] and electrode voltages V[P] on a layout; a
// *trajectory* is one independent KMC run (layout, energy set, RNG key, hop
// budget, initial occupation).
#pragma once
#include <stdint.h>

#include "../../include/kmc_dn_amd.h"

namespace kmc {

constexpr int NMAX = KMC_NMAX;   // acceptors per network
constexpr int PMAX = KMC_PMAX;   // electrodes per network
constexpr int OCCW = KMC_OCCW;   // 64-bit words of an occupation bitmask
constexpr int SMAX_FP32 = 192;   // sites of the FP32 batched kernel (3 lanes per site chunk)
constexpr int SMAX_FP64 = 80;    // sites of the FP64 dense kernel (LDS-resident lists)

struct LayoutDev {
  int32_t N, P, S, prune;
  double nu, kT, I0, R;
  double I0R;        // I_0 * R
  float scale2;      // log2(e) / kT: energies in kT units, base-2 exponent
  int32_t elw_ok;    // every electrode weight is finite (elw usable)
  // FP32 batched kernel.  tab32[u * S + s] = {lt, c} for the ordered pair
  // (s, u), symmetric in (s, u):
  //   lt = log2(nu * transitions_constant[s][u])  (-inf when impossible:
  //        diagonal, electrode-electrode, pruned or underflowed),
  //   c  = scale2 * I_0 * R / d[s][u] for acceptor-acceptor pairs, else 0.
  // 64 * 3 trailing entries {-inf, 0} let lanes past S read in bounds.
  const float2* tab32;
  // Same pairs as {lt, b = lt + c} (b = -inf where lt = -inf), and the c column
  // table ccol[u * S + s] = c(s, u) for acceptor columns u < N (N*S + 192 floats).
  const float2* tabB;
  const float* ccol;
  // Electrode weights elw[e * 192 + s] = nu * tc[s][N + e] for acceptor sites s
  // (0 for electrode sites, s >= N and pruned pairs; rows rounded up to a
  // multiple of 4, the padding zero): the
  // rate between acceptor s and electrode e is elw * min(1, 2^(e~_src - e~_dst)).
  const float* elw;
  const double* coul64;   // [N*N] I_0*R/d for acceptor pairs (symmetric, 0 diagonal)
  // Positions policy: site coordinates (w = 1 acceptor, 0 electrode) and the
  // closed forms lt = pos_l0 + pos_mkl * d, c = pos_kc / d (null if absent).
  const float4* pos4;
  float pos_l0, pos_mkl, pos_kc;
  int32_t has_pos;
  // FP64 dense kernel (reference arithmetic).
  const double* tc64;     // [S*S] transitions_constant
  const double* ird64;    // [S*S] (I_0*R)/d[i][j] (acceptor pairs; 0 elsewhere)
  const double* invd64;   // [N*N] 1.0/d[i][j] (0 on the diagonal)
  const double* dist64;   // [S*S] distances as given (mean-field estimators)
};



struct EsetDev {
  const double* E;   // [N] E_constant
  const double* V;   // [P] electrode voltages (site_energies[N:])
};

// Mean-field estimators of the Go library: probSimulate
// (goSimulation/probabilitySimulation.go:53-157) and calcAverageCurrent
// (goSimulation/simulation.go:671-736, one wave per network).
struct MeanfieldParams {
  const LayoutDev* layouts;
  const EsetDev* esets;
  const int32_t* layout_of;   // [n]
  const int32_t* eset_of;     // [n]
  double* occ;                // [n][NMAX] fractional occupation (in; probSimulate: out)
  double* eo;                 // [n][PMAX] electrode occupation (probSimulate) or currents
  double* se;                 // [n][NMAX] acceptor energies of the last step, or null
  double* time;               // [n] or null
  double* avg;                // [n][NMAX] occupation x time, or null
  double* traffic;            // [n][tstride] net traffic (S x S row-major), or null
  int64_t tstride;
  int64_t steps;
  int32_t n;
  int32_t ld;                 // row length of the LDS pair table (kmc_meanfield_kernel)
};

// The LDS pair table of probSimulate: S rows of S | 1 doubles, 151 KiB at most (beside
// 8 KiB of the sites' own).
constexpr int MF_LDS_SITES = 139;
constexpr int mf_row(int S) { return S | 1; }
// the tiled kernel's two tiles of MF_TILE rows of 64 C + 1
constexpr int MF_TILE = 32;

struct TrajDev {
  int32_t layout;
  int32_t eset;
  uint64_t seed;      // Philox key
  uint64_t hop0;      // Philox counter of the first hop
  int64_t prehops;    // hops run before tallies start (not counted)
  int64_t hops;       // counted hops
  uint64_t occ[OCCW]; // initial occupation bitmask
  int64_t h_begin;    // absolute hop range of this launch (with BatchParams::resume)
  int64_t h_end;
};

struct TrajOut {
  double time;
  int64_t hops_done;
  int32_t status;
  int32_t ticks;     // steady-counter ticks of the trajectory's last run (saturated)
  uint64_t occ[OCCW];
  int64_t eo[PMAX];
};

struct GroupDev {
  int32_t layout;
  int32_t first;   // first trajectory (trajectories of a group are contiguous)
  int32_t count;   // <= waves per workgroup
  int32_t pad;
};

struct BatchParams {
  const TrajDev* trajs;
  const LayoutDev* layouts;
  const EsetDev* esets;
  const GroupDev* groups;
  int32_t ngroups;
  int32_t recompute_interval;   // hops between FP64 energy recomputes (>0)
  int32_t* queue;               // work-queue head, zero before launch
  TrajOut* out;
  double* occ_time;             // [ntraj * NMAX] or null
  double* traffic;              // [ntraj * traffic_stride] net traffic, or null
  int64_t traffic_stride;       // >= S*S of every layout in the batch
  int32_t post_hop_record;      // 1: numba convention (post-hop state)
  int32_t resume;               // 1: run [h_begin, h_end) from the state in `out`
  uint64_t* phases;             // [FP32_PHASES] sums over trajectories (the phase-timing
                                // instantiations only), or null
  int64_t time_limit;           // constant-rate clock ticks a solo trajectory runs before
                                // it stops at its next recompute point; 0: none
  int32_t state_slots;          // states a one-chunk solo trajectory keeps, 2..STATE_SLOTS
                                // (the others: STATE_SLOTS)
  int32_t pad2;
  unsigned char* states;        // the waves' state records, state_area bytes per wave; null
                                // (and state_area 0): general steps alone
  int64_t state_area;
};

// States a wave of the FP32 kernels keeps (one per lane), and the bytes of one's
// record per site chunk: the FP32 row sums and energies of the 64 lanes.
constexpr int STATE_SLOTS = 64;
constexpr int STATE_RECORD_BYTES = 64 * (4 + 4);
constexpr int STORE_MAX_SLOTS = 4;   // largest kmc_run_opts.state_store

// Hop phases of the FP32 batched kernels timed by their phase-timing
// instantiations (shader cycles of each trajectory's first wave, summed over
// trajectories): 0 uniforms and FP64 recomputes, 1 energy update, electrode
// terms, row sums and team reduction of a new state (or its lookup), 2 its FP64
// prefix scan and record, 3 event selection of a new transition, 4 its partner
// selection, 5 its insertion and the hop, 6 hops by kept transitions and leaps
// (general steps: 0 to 5).  Slot 7 counts the hops from a state that the hop before
// led back into, slot 8 those by a kept transition (general steps: by a partner
// prefix formed before), slot 9 those taken by leaps, slot 10 the states found
// among the kept ones instead of evaluated.
constexpr int FP32_PHASES = 11;

struct PlainParams {
  const TrajDev* trajs;
  const LayoutDev* layouts;
  const EsetDev* esets;
  TrajOut* out;
  const double* uniforms;   // replayed stream (2 per hop) for trajectory 0, or null
  int32_t* events;          // [prehops+hops] event index from*S+to, or null
  double* totals;           // [prehops+hops] problist[-1] per hop, or null
  double* traffic;          // [ntraj * S*S] gross traffic, or null
  double* occ_time;         // [ntraj * NMAX] post-hop occupation time, or null
  double* se_out;           // [ntraj * NMAX] final site_energies[0:N], or null
  uint64_t* phases;         // [PLAIN_PHASES] shader cycles per hop phase of trajectory 0
                            // (the phase-timing instantiation only), or null
  // The state records of the workgroups: `slots` (a power of two) of state_bytes
  // each per workgroup; npairs bounds the possible pairs of every layout, smax
  // and nmax their sites and acceptors.
  unsigned char* states;
  int64_t state_bytes;
  int32_t slots;
  int32_t npairs;
  int32_t smax, nmax;
  int32_t* queue;           // trajectories beyond the grid, zero before launch; null: none
  int32_t ntraj;
  int32_t pad;
};

// Hop phases of the FP64 dense kernel timed by its phase-timing instantiation:
// energies, pair lists, rates and prefix chain of new states, storing their
// records, event search of cached states, hops, leaps and records (with
// uniforms and clock).
constexpr int PLAIN_PHASES = 7;

// Status codes written per trajectory (also returned by the C-ABI).
enum : int32_t {
  ST_OK = KMC_OK,
  ST_ZERO_RATE = KMC_ERR_ZERO_RATE,
  ST_BAD_INPUT = KMC_ERR_ARGS,
};

}  // namespace kmc
