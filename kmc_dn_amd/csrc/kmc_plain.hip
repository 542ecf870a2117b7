// FP64 dense hop loop: the reference's arithmetic on the GPU.
//
// Restates _simulate_discrete_record (kmc_dopant_networks.py:33-135) with the
// same FP64 operations in the same order, so that with a replayed uniform
// stream the event sequence equals the CPU restatement's bit for bit:
//   * site energies: se[i] = E[i] + ((-I_0)*R) * sum_{j != i} (1 - n_j)/d[i][j],
//     summed over ascending j (:59-66).  An occupied j adds an exact +0.0 to a
//     sum that is +0.0 or positive, which leaves it unchanged, so only the
//     empty acceptors are visited (ascending); 1/d is precomputed (the same
//     IEEE quotient) with a zero diagonal;
//   * rates: tc[i][j] * (dE > 0 ? nu*exp(-dE/kT) : nu) for possible pairs (:69-87);
//   * prefix sum in row-major order (:91-97).  Impossible pairs contribute an
//     exact 0.0, so the sequential chain runs over the possible pairs only, in
//     row-major order, which leaves every partial sum unchanged;
//   * hop time -log(1-u)*(1/total) and event = first k with problist[k]/total >= u
//     (:100-110); u == 0 selects k = 0 exactly as the reference's scan does.
// This file is compiled with -ffp-contract=off: no a*b+c is fused.
//
// One wave (64 lanes) per trajectory.  Three paths take a hop, all with the
// same operations on the same values, so which of them took it changes no bit:
//
//  * An evaluated state: the rates of the possible pairs and their sequential
//    prefix sum.  The possible pairs of a hop have a closed structure
//    (_transition_possible, :137-163): rows of occupied acceptors (ascending)
//    hop into [empty acceptors ascending, then the electrodes], and then each
//    electrode row hops into the empty acceptors.  Two short LDS lists
//    (occupied acceptors; empty acceptors followed by electrodes) built with
//    ballots give every list position its (row, column) by one small division,
//    so the rates are lane-parallel over the compacted list.  Only the prefix
//    chain is serial: one lane runs it from registers, 8 values per LDS block
//    in two alternating register sets (the next block's loads in flight during
//    the current block's adds).  About 10,000 cycles at N = 30, P = 8.
//  * A cached state.  Everything a hop needs of its state is a function of the
//    occupation alone (the energies are summed afresh for every state), so the
//    first visit stores it and every later one reads it: the quotients
//    problist[k]/total of the kept entries, their events, 1/total.  The event
//    is then one lane-parallel search, about 400 cycles.  Trajectories revisit
//    a few states: of 2e4 hops at N = 30, P = 8 and 1 kT 0.1-0.3 % are first
//    visits; at +-300 kT 2-10 % fall outside the last 1024 states (2-94 %
//    outside the last two, which is why the cache holds many).  The records
//    live in global memory (a state is up to 10 B per possible pair; the ones
//    in use stay in the CU's L1 and the XCD's L2), their tags in LDS: sets of
//    up to 64 ways, one tag per lane, so a lookup is one LDS read and a
//    ballot.  Storing a record costs a fifth of an evaluation, so a trajectory that
//    found states it had not seen on more than 7/8 of the hops of a uniform block sets
//    their tags alone over the next block, selects the events from the prefix sums
//    and stores a record when a tag comes back.  2000 hops of N = 30, P = 8, nearly every
//    one new (a = I_0 = 1): 19.7 ms with every record stored, now 18.0 (16.6 with no
//    records at all); at +-300 kT 1.76 and 1.78 (9.9).
//  * A run of hops back and forth between two states (a leap).  Whether the hop
//    with event uniform u leads from A to B depends on u alone: lo < u <= hi,
//    the quotients around the event.  The lanes test the 64 hops of a uniform
//    block at once; the run of hops that pass is applied together, its clock
//    and occupation times added one by one in hop order as the reference adds
//    them (about 20 cycles a hop).
//
// Uniforms and the clock's -log(1 - u) are computed lane-parallel for 64 hops
// at a time.  With STAGE the layout's tables (1/d, tc, (I_0*R)/d) are copied to
// LDS once per trajectory.  Workgroups take trajectories from a queue when the
// batch has more of them than fit on the GPU at once; the state records belong
// to the workgroup and start empty with every trajectory.
#include "kmc_device.h"

namespace kmc {

// LDS carve-up for layouts of at most S sites, N acceptors and npairs possible
// pairs, and `slots` state records (all offsets in doubles, 16-byte aligned).
struct PlainLds {
  size_t se, buf, lists, invd, tc, ird, tags, next, total;
  __host__ __device__ PlainLds(int S, int N, int npairs, int slots, bool stage) {
    auto up2 = [](size_t x) { return (x + 1) & ~(size_t)1; };
    const size_t SS = (size_t)S * S;
    se = 0;
    buf = up2(S);
    lists = buf + up2(npairs + 16);   // int16: occupied acceptors [N], targets [S], kept [npairs]
    invd = lists + up2(((size_t)N + S + npairs + 3) / 4);
    tc = invd + (stage ? up2((size_t)N * N) : 0);
    ird = tc + (stage ? up2(SS) : 0);
    tags = ird + (stage ? up2(SS) : 0);
    next = tags + 2 * (size_t)slots;   // two words per tag, then one int per set of 64 ways
    total = next + up2(((size_t)slots + 127) / 128);
  }
};

// q = x / d and r = x - q*d for 0 <= x < 2^20, 1 <= d <= 256: an FP32 estimate
// from the reciprocal (relative error ~1e-7, so q is off by at most one), fixed.
__device__ __forceinline__ int div_small(int x, int d, float rcp, int& r) {
  int q = (int)((float)x * rcp);
  r = x - q * d;
  if (r < 0) {
    q -= 1;
    r += d;
  }
  if (r >= d) {
    q += 1;
    r -= d;
  }
  return q;
}

// A state's tag: the occupation (acceptors 0-63 in the first word, 64-79 in the
// low bits of the second), bit 63 of the second word set, its kept entries
// above bit 32.  Bit 62 instead of 63: a state that was seen and has no record.
constexpr uint64_t TAG_VALID = 1ull << 63;
constexpr uint64_t TAG_SEEN = 1ull << 62;
constexpr uint64_t TAG_STATE = TAG_VALID | 0xFFFFull;

// State records of one workgroup: {1/total, total}, then the quotients of the
// kept entries, then their events (row << 8 | column).
struct StateRecord {
  double* head;
  __device__ __forceinline__ double* quot() const { return head + 2; }
  __device__ __forceinline__ uint16_t* event(int cap) const {
    return reinterpret_cast<uint16_t*>(head + 2 + cap);
  }
};

// PHASE: the phase-timing instantiation (shader-clock reads at the phase
// boundaries of every hop; the work is unchanged).
template <bool REC, bool STAGE, bool PHASE>
__device__ __forceinline__ void plain_trajectory(const PlainParams& p, const int t, const int lane,
                                 unsigned char* smem) {
  const TrajDev td = p.trajs[t];
  const LayoutDev L = p.layouts[td.layout];
  const EsetDev es = p.esets[td.eset];
  const int N = L.N, P = L.P, S = L.S, SS = S * S;
  const double nu = L.nu, kT = L.kT;
  const double nIR = (-L.I0) * L.R;
  // kT == 1 and nu == 1 make -dE/kT and nu*exp(x) exact copies of their
  // operand: the same bits with or without the operation
  const bool kT1 = kT == 1.0, nu1 = nu == 1.0;

  double* dl = reinterpret_cast<double*>(smem);
  const PlainLds off(p.smax, p.nmax, p.npairs, p.slots, STAGE);
  double* se = dl + off.se;
  double* buf = dl + off.buf;     // rates of the possible pairs, then their prefix sums
  int16_t* srcA = reinterpret_cast<int16_t*>(dl + off.lists);   // occupied acceptors
  int16_t* tgt = srcA + N;        // empty acceptors, then electrodes N..S-1
  int16_t* kidx = tgt + S;        // list positions of the kept rates
  const double* invd = L.invd64;
  const double* tcp = L.tc64;
  const double* irdp = L.ird64;
  if (STAGE) {
    double* a = dl + off.invd;
    double* b = dl + off.tc;
    double* c = dl + off.ird;
    for (int k = lane; k < N * N; k += 64) a[k] = L.invd64[k];
    for (int k = lane; k < SS; k += 64) {
      b[k] = L.tc64[k];
      c[k] = L.ird64[k];
    }
    invd = a;
    tcp = b;
    irdp = c;
  }
  // the state records' tags: sets of `ways` (a power of two, at most 64)
  uint64_t* tags = reinterpret_cast<uint64_t*>(dl + off.tags);
  int* next_way = reinterpret_cast<int*>(dl + off.next);
  const int ways = min(p.slots, 64), sets = p.slots / ways;
  for (int k = lane; k < p.slots; k += 64) tags[2 * k + 1] = 0;
  for (int k = lane; k < sets; k += 64) next_way[k] = 0;
  auto record = [&](int slot) {
    return StateRecord{reinterpret_cast<double*>(
        p.states + ((size_t)blockIdx.x * p.slots + slot) * p.state_bytes)};
  };

  // acceptors (N <= 80) live in the first two words
  uint64_t occ0 = td.occ[0], occ1 = td.occ[1];
  // lanes of site chunk c (site lane + 64c) holding acceptors; S <= 80 < 128
  const uint64_t acc0 = N >= 64 ? ~0ull : ((1ull << N) - 1);
  const uint64_t acc1 = N <= 64 ? 0ull : ((1ull << (N - 64)) - 1);

  for (int e = lane; e < P; e += 64) se[N + e] = es.V[e];
  double E0 = 0.0, E1 = 0.0;
  if (lane < N) E0 = es.E[lane];
  if (lane + 64 < N) E1 = es.E[lane + 64];
  wave_lds_sync();
  int64_t eo = 0;                 // lane e < P holds electrode e's tally
  double ot0 = 0.0, ot1 = 0.0;    // post-hop occupation time, sites lane and lane+64
  double time = 0.0;
  int32_t status = ST_OK;
  // prehops + hops <= INT32_MAX is checked when a batch is created
  const int prehops = (int)td.prehops, total_hops = (int)(td.prehops + td.hops);
  int h = 0;
  uint64_t ph[PLAIN_PHASES] = {};
  uint64_t tp = PHASE ? __builtin_amdgcn_s_memtime() : 0;
  // cycles since the last mark into phase k
  auto mark = [&](int k) {
    if constexpr (PHASE) {
      const uint64_t now = __builtin_amdgcn_s_memtime();
      ph[k] += now - tp;
      tp = now;
    }
  };
  // -log(1 - u_clock) and u_event of hop (h & ~63) + lane: 64 hops of uniforms
  // and clock logarithms at a time, read with readlane per hop (the same
  // values and operations as per hop)
  double lg_lane = 0.0, ue_lane = 0.0;
  auto refill = [&](int hh) {
    const int64_t hk = (hh & ~63) + (int64_t)lane;
    double uc = 0.5, ue = 0.5;
    if (p.uniforms) {
      if (hk < total_hops) {
        uc = p.uniforms[2 * hk];
        ue = p.uniforms[2 * hk + 1];
      }
    } else {
      stream_uniforms(td.seed, td.hop0 + (uint64_t)hk, uc, ue);
    }
    lg_lane = -log(1.0 - uc);
    ue_lane = ue;
  };

  // The pair lists and site energies of occupation (q0, q1); sets nA, cE.
  int nA = 0, cE = 0;
  auto energies = [&](uint64_t q0, uint64_t q1) {
    // occupied / empty acceptors as wave-uniform masks of the two site chunks
    const uint64_t o0 = q0 & acc0, o1 = q1 & acc1;
    const uint64_t e0 = acc0 & ~o0, e1 = acc1 & ~o1;
    // the lists: occupied acceptors, then targets (empty acceptors, electrodes)
    nA = __builtin_popcountll(o0) + __builtin_popcountll(o1);
    cE = N - nA;
    {
      const bool oc0 = (o0 >> lane) & 1ull, oc1 = (o1 >> lane) & 1ull;
      const bool em0 = (e0 >> lane) & 1ull, em1 = (e1 >> lane) & 1ull;
      const int lo_o = __builtin_popcountll(o0), lo_e = __builtin_popcountll(e0);
      if (oc0) srcA[mbcnt(o0)] = (int16_t)lane;
      if (oc1) srcA[lo_o + mbcnt(o1)] = (int16_t)(lane + 64);
      if (em0) tgt[mbcnt(e0)] = (int16_t)lane;
      if (em1) tgt[lo_e + mbcnt(e1)] = (int16_t)(lane + 64);
      if (lane < P) tgt[cE + lane] = (int16_t)(N + lane);
    }
    wave_lds_sync();
    mark(1);
    // site energies, :59-66: the empty acceptors j (tgt[0..cE), ascending),
    // four at a time with their loads issued together, added in order
    {
      double a0 = 0.0, a1 = 0.0;
      const int l0 = min(lane, N - 1), l1 = min(lane + 64, N - 1);
      for (int q0 = 0; q0 < cE; q0 += 4) {
        const int cnt = min(4, cE - q0);
        int j[4];
        double x0[4], x1[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) j[q] = tgt[q0 + min(q, cnt - 1)];
#pragma unroll
        for (int q = 0; q < 4; ++q) x0[q] = invd[j[q] * N + l0];
        if (N > 64) {
#pragma unroll
          for (int q = 0; q < 4; ++q) x1[q] = invd[j[q] * N + l1];
        }
#pragma unroll
        for (int q = 0; q < 4; ++q)
          if (q < cnt) {
            a0 += x0[q];
            if (N > 64) a1 += x1[q];
          }
      }
      if (lane < N) se[lane] = E0 + nIR * a0;
      if (lane + 64 < N) se[lane + 64] = E1 + nIR * a1;
    }
    wave_lds_sync();
    mark(0);
  };

  // Evaluates occupation (occ0, occ1): leaves the kept entries' prefix sums in
  // buf[0..ns) and their list positions in kidx, returns the total.
  int ns = 0;                // entries kept (wave-uniform)
  float rA = 0.f, rE = 0.f;
  int cA = 0, nAA = 0;
  auto pair_of = [&](int idx, int& i, int& j) {
    int r;
    if (idx < nAA) {
      const int q = div_small(idx, cA, rA, r);
      i = srcA[q];
    } else {
      const int q = div_small(idx - nAA, cE, rE, r);
      i = N + q;
    }
    j = tgt[r];
  };
  auto evaluate = [&]() -> double {
    energies(occ0, occ1);
    cA = cE + P;
    nAA = nA * cA;
    const int n = nAA + P * cE;
    // rates of the possible pairs in row-major order, :69-87; two list entries
    // per lane and round, computed side by side (entries past n are evaluated
    // at n - 1 and dropped).
    //
    // Absorbed entries are dropped too.  All rates are >= 0, so the running
    // sum s_{k-1} before entry k is at least the largest earlier rate M, and a
    // rate below half an ulp of M (so below half an ulp of s_{k-1}) leaves the
    // rounded sum unchanged: fl(s + r) == s.  M is bounded from below by the
    // running maximum of the rates' high words (their low 32 bits cleared),
    // a wave max-scan on 32-bit integers; every partial sum the prefix chain
    // forms over the kept entries is the reference's partial sum at that
    // entry, and the dropped entries' partial sums equal the kept entry's
    // before them.  The kept rates go to buf[0..ns) and their list positions
    // to kidx.
    rA = cA > 0 ? __builtin_amdgcn_rcpf((float)cA) : 0.f;
    rE = cE > 0 ? __builtin_amdgcn_rcpf((float)cE) : 0.f;
    auto rate_of = [&](int i, int j) {
      const int k = i * S + j;
      double dE;
      if (i < N && j < N) dE = se[j] - se[i] - irdp[k];
      else dE = se[j] - se[i];
      const double x = kT1 ? -dE : -dE / kT;
      const double ex = exp(x);
      const double m = dE > 0 ? (nu1 ? ex : nu * ex) : nu;
      return tcp[k] * m;
    };
    uint32_t hcarry = 0;   // running maximum of the high words (wave-uniform)
    ns = 0;
    auto keep = [&](double r, int idx) {
      const bool valid = idx < n;
      const uint32_t hi = valid ? (uint32_t)((uint64_t)__double_as_longlong(r) >> 32) : 0u;
      const uint32_t m = max(wave_max_u32(hi), hcarry);
      hcarry = (uint32_t)__builtin_amdgcn_readlane((int)m, 63);
      const uint32_t e = (m >> 20) & 0x7FFu;   // biased exponent of the bound
      const uint32_t thr = e > 53u ? (e - 53u) << 20 : 0u;   // high word of its half ulp
      const bool kp = valid && hi >= thr;
      const uint64_t km = ballot(kp);
      if (kp) {
        const int pos = ns + mbcnt(km);
        buf[pos] = r;
        kidx[pos] = (int16_t)idx;
      }
      ns += __builtin_popcountll(km);
    };
    for (int b0 = 0; b0 < n; b0 += 128) {
      const int ia = b0 + lane, ib = b0 + 64 + lane;
      int i0, j0, i1, j1;
      pair_of(ia < n ? ia : n - 1, i0, j0);
      pair_of(ib < n ? ib : n - 1, i1, j1);
      const double r0 = rate_of(i0, j0);
      const double r1 = rate_of(i1, j1);
      keep(r0, ia);
      keep(r1, ib);
    }
    wave_lds_sync();
    mark(2);
    // cumulative sum, :91-97, over the kept entries: one lane; blocks of 8 in
    // two register sets that alternate, so the next block's loads are in
    // flight during this block's adds
    double acc = 0.0;
    if (lane == 0) {
      const int nb = ns >> 3;
      double A[8], B[8];
      // the running sum through one block of 8, written back as it goes: the
      // block's registers are only read, so they are free once it is done
      auto chain = [&](const double (&v)[8], int base) {
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          acc = v[q] + acc;
          buf[base + q] = acc;
        }
      };
      if (nb > 0) {
#pragma unroll
        for (int q = 0; q < 8; ++q) A[q] = buf[q];
      }
      int blk = 0;
#pragma unroll 1
      for (; blk + 1 < nb; blk += 2) {
        // straight-line body: the reload reads an existing block even past the
        // last pair (its values are then unused)
        const int nxt = min(blk + 2, nb - 1) * 8;
#pragma unroll
        for (int q = 0; q < 8; ++q) B[q] = buf[(blk + 1) * 8 + q];
        __builtin_amdgcn_sched_barrier(0);   // keep the loads ahead of the adds
        chain(A, blk * 8);
#pragma unroll
        for (int q = 0; q < 8; ++q) A[q] = buf[nxt + q];
        __builtin_amdgcn_sched_barrier(0);
        chain(B, (blk + 1) * 8);
      }
      if (blk < nb) chain(A, blk * 8);
      for (int idx = nb << 3; idx < ns; ++idx) {
        acc = buf[idx] + acc;
        buf[idx] = acc;
      }
    }
    return readlane_f64(acc, 0);
  };

  // The way of the current state in its set (-1: not cached); sets `set`, `ns`.
  int set = 0;
  auto lookup = [&]() -> int {
    // multiplicative mix of the occupation words (few sets: any spread will do)
    uint32_t x = (uint32_t)occ0 * 0x9E3779B1u ^ (uint32_t)(occ0 >> 32) * 0x85EBCA77u ^
                 (uint32_t)occ1 * 0xC2B2AE3Du;
    x *= 0x27D4EB2Fu;
    set = (int)(x >> 20) & (sets - 1);
    const ulonglong2 tg =
        *reinterpret_cast<const ulonglong2*>(tags + 2 * (set * ways + (lane & (ways - 1))));
    const uint64_t m = ballot(tg.x == occ0 && (tg.y & TAG_STATE) == (occ1 | TAG_VALID));
    if (!m) return -1;
    const int way = __builtin_ctzll(m) & (ways - 1);
    ns = (int)((uint32_t)__builtin_amdgcn_readlane((int)(uint32_t)(tg.y >> 32), way) & 0xFFFFu);
    return way;
  };

  // The way of the current state's tag without a record in set `set` (-1: not seen).
  // (Asked of new states only: a test of the looked-up tag for both kinds cost hops from
  // recorded states 5 %.)
  auto seen_way = [&]() -> int {
    const ulonglong2 tg =
        *reinterpret_cast<const ulonglong2*>(tags + 2 * (set * ways + (lane & (ways - 1))));
    const uint64_t m = ballot(tg.x == occ0 && tg.y == (occ1 | TAG_SEEN));
    return m ? __builtin_ctzll(m) & (ways - 1) : -1;
  };

  // The hop before the current one: where it started, its event and bounds.  A
  // hop that undoes it makes (state before, current state) a pair, whose two
  // events the leap tests.
  struct Hop {
    double lo, hi, scale, total;   // the event is taken iff lo < u <= hi
    uint64_t s0, s1;               // occupation it starts from
    int from, to;
  };
  Hop A{}, B{};        // A: from the current state to B's start; B: the way back
  bool pair = false;   // A and B hold
  bool prev = false;   // B holds the hop just taken
  uint64_t last0 = occ0, last1 = occ1;   // occupation the last hop started from
  // Takes the hop whose event code is from << 8 | to (-1: no match), bounds lo < u <= hi.
  auto take = [&](int code, double ue, double lo, double hi, double scale, double total,
                  bool tally) __attribute__((always_inline)) {
    const int hl = h & 63;
    // u == 0 and no match: the reference's event 0, (0, 0)
    const bool first = ue == 0.0 || code < 0;
    const int from = first ? 0 : code >> 8, to = first ? 0 : code & 255;
    mark(5);
    // the event and the clock, :100
    const double lg = readlane_f64(lg_lane, hl);
    const double hop_time = lg * scale;
    if (t == 0 && lane == 0) {
      if (p.events) p.events[h] = from * S + to;
      if (p.totals) p.totals[h] = total;
    }
    // perform hop, :116-123
    last0 = occ0;
    last1 = occ1;
    if (from < N) {
      if (from < 64) occ0 &= ~(1ull << from);
      else occ1 &= ~(1ull << (from - 64));
    } else if (lane == from - N) {
      eo -= 1;
    }
    if (to < N) {
      if (to < 64) occ0 |= 1ull << to;
      else occ1 |= 1ull << (to - 64);
    } else if (lane == to - N) {
      eo += 1;
    }
    // record, :126-130
    if (REC && tally) {
      if (p.traffic && lane == 0) unsafeAtomicAdd(p.traffic + (size_t)t * SS + from * S + to, 1.0);
      if ((occ0 >> lane) & 1ull) ot0 += hop_time;
      if ((occ1 >> lane) & 1ull) ot1 += hop_time;
    }
    time += hop_time;
    ++h;
    // a hop back to where the one before it started: A that hop, B this one
    pair = prev && !first && occ0 == B.s0 && occ1 == B.s1;
    if (pair) A = B;
    B = Hop{lo, hi, scale, total, last0, last1, from, to};
    prev = !first;
    mark(6);
  };
  // A tag for the current state in set `set`: `mark` its second word's upper bits.
  auto tag = [&](int way, uint64_t mark) __attribute__((always_inline)) {
    if (lane == 0) {
      tags[2 * (set * ways + way)] = occ0;
      tags[2 * (set * ways + way) + 1] = occ1 | mark;
    }
  };
  // A hop of the current state, which has no tag: the tag alone is set and the event
  // selected from the prefix sums.  The lanes' 64 stretches of entries by their last ones,
  // then the stretch (at most 32 entries: 2048 pairs at S <= 80).  false: no rate.
  auto unrecorded = [&](bool tally) __attribute__((always_inline)) -> bool {
    const double total = evaluate();
    mark(3);
    if (total == 0.0) return false;
    const int way = __builtin_amdgcn_readfirstlane(next_way[set]);
    if (lane == 0) next_way[set] = (way + 1) & (ways - 1);
    tag(way, TAG_SEEN);
    const double ue = readlane_f64(ue_lane, h & 63), scale = 1.0 / total;
    double lo = 0.0, hi = 0.0;
    int code = -1;
    const int stretch = (ns + 63) >> 6;
    const double end = buf[min(ns, (lane + 1) * stretch) - 1] / total;
    const uint64_t mc = ballot(lane * stretch < ns && end >= ue);
    if (mc) {
      const int c = __builtin_ctzll(mc);
      if (c > 0) lo = readlane_f64(end, c - 1);
      const int k = min(c * stretch + min(lane, stretch - 1), ns - 1);
      const double qv = buf[k] / total;
      int i, j;
      pair_of(kidx[k], i, j);
      const int l = __builtin_ctzll(ballot(qv >= ue));   // (its last entry is one)
      hi = readlane_f64(qv, l);
      if (l > 0) lo = readlane_f64(qv, l - 1);
      code = __builtin_amdgcn_readlane(i << 8 | j, l);
    }
    wave_lds_sync();
    mark(4);
    take(code, ue, lo, hi, scale, total, tally);
    return true;
  };
  int fresh = 0;            // states of this uniform block that had no tag
  bool tags_only = false;   // this block's new states get no records
  // every scalar load of the set-up has returned before the loop: LDS
  // operations alone then complete in order, so the waits for the prefix
  // chain's blocks count only the operations issued after each block
  __builtin_amdgcn_s_waitcnt(0x0070);   // vmcnt(0) lgkmcnt(0)
  while (h < total_hops) {
    const bool tally = h >= prehops;
    if (h == prehops) {   // reset() between prehops and hops (:562-585)
      time = 0.0;
      eo = 0;
      ot0 = ot1 = 0.0;
    }
    const int hl = h & 63;
    if (hl == 0) {
      refill(h);
      tags_only = fresh > 56;
      fresh = 0;
    }
    if (pair) {
      // lane k (>= hl) starts its hop in A's state when k - hl is even
      const bool inA = ((lane ^ hl) & 1) == 0;
      const uint64_t ok = ballot(ue_lane > (inA ? A.lo : B.lo) && ue_lane <= (inA ? A.hi : B.hi));
      const uint64_t no = ~(ok >> hl);
      int n = no ? __builtin_ctzll(no) : 64;
      n = min(n, min(64 - hl, (tally ? total_hops : prehops) - h));
      if (n > 0) {
        const double dts = lg_lane * (inA ? A.scale : B.scale);
        if (t == 0 && lane >= hl && lane < hl + n) {
          const int hk = (h & ~63) + lane;
          if (p.events) p.events[hk] = inA ? A.from * S + A.to : B.from * S + B.to;
          if (p.totals) p.totals[hk] = inA ? A.total : B.total;
        }
        // the clock and, post-hop (:126-130), the occupation times in hop order
        if (REC && tally) {
          const bool a0 = (A.s0 >> lane) & 1ull, b0 = (B.s0 >> lane) & 1ull;
          const bool a1 = (A.s1 >> lane) & 1ull, b1 = (B.s1 >> lane) & 1ull;
          for (int k = 0; k < n; ++k) {
            const double d = readlane_f64(dts, hl + k);
            time += d;
            if ((k & 1) ? a0 : b0) ot0 += d;
            if (N > 64) {
              if ((k & 1) ? a1 : b1) ot1 += d;
            }
          }
          if (p.traffic && lane == 0) {
            double* tr = p.traffic + (size_t)t * SS;
            unsafeAtomicAdd(tr + A.from * S + A.to, (double)((n + 1) >> 1));
            if (n > 1) unsafeAtomicAdd(tr + B.from * S + B.to, (double)(n >> 1));
          }
        } else {
          int k = 0;
          for (; k + 4 <= n; k += 4) {
            double d[4];
#pragma unroll
            for (int q = 0; q < 4; ++q) d[q] = readlane_f64(dts, hl + k + q);
#pragma unroll
            for (int q = 0; q < 4; ++q) time += d[q];
          }
          for (; k < n; ++k) time += readlane_f64(dts, hl + k);
        }
        const int e = N + lane;
        const int dA = (lane < P && A.to == e ? 1 : 0) - (lane < P && A.from == e ? 1 : 0);
        const int dB = (lane < P && B.to == e ? 1 : 0) - (lane < P && B.from == e ? 1 : 0);
        eo += ((n + 1) >> 1) * dA + (n >> 1) * dB;
        h += n;
        last0 = (n & 1) ? A.s0 : B.s0;
        last1 = (n & 1) ? A.s1 : B.s1;
        if (n & 1) {
          const Hop x = A;
          A = B;
          B = x;
          occ0 = A.s0;
          occ1 = A.s1;
        }
        mark(6);
        continue;
      }
    }
    // the state's record: read, or evaluated and stored first
    int way = lookup();
    if (way < 0) {
      way = seen_way();
      const bool seen = way >= 0;
      if (!seen) ++fresh;
      if (!seen && tags_only) {
        if (unrecorded(tally)) continue;
        if (p.totals && t == 0 && lane == 0) p.totals[h] = 0.0;
        status = ST_ZERO_RATE;
        last0 = occ0;
        last1 = occ1;
        break;
      }
      const double total = evaluate();
      mark(3);
      if (total == 0.0) {   // reference: ZeroDivisionError at 1/problist[-1]
        if (p.totals && t == 0 && lane == 0) p.totals[h] = total;
        status = ST_ZERO_RATE;
        last0 = occ0;
        last1 = occ1;
        break;
      }
      if (!seen) {
        way = __builtin_amdgcn_readfirstlane(next_way[set]);
        if (lane == 0) next_way[set] = (way + 1) & (ways - 1);
      }
      tag(way, TAG_VALID | ((uint64_t)ns << 32));
      const StateRecord r = record(set * ways + way);
      double* q = r.quot();
      uint16_t* ev = r.event(p.npairs);
      for (int k = lane; k < ns; k += 64) {
        int i, j;
        pair_of(kidx[k], i, j);
        q[k] = buf[k] / total;
        ev[k] = (uint16_t)(i << 8 | j);
      }
      if (lane == 0) {
        r.head[0] = 1.0 / total;
        r.head[1] = total;
      }
      wave_lds_sync();   // this wave's later loads see the record (memory order within a wave)
      mark(4);
    }
    // first k with problist[k]/total >= u, :103-110 (monotone in k): a kept
    // entry, since a dropped one repeats the partial sum of the kept entry
    // before it.  Up to 256 entries are read at once; longer records first
    // find the chunk of 64 by its last entry.
    const StateRecord r = record(set * ways + way);
    const double* q = r.quot();
    const uint16_t* ev = r.event(p.npairs);
    const double scale = r.head[0], total = r.head[1];
    const double ue = readlane_f64(ue_lane, hl);
    double lo = 0.0, hi = 0.0;
    int code = -1;
    if (ns <= 256) {
      double qv[4];
      int cv[4];
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (64 * m >= ns) break;
        const int k = min(64 * m + lane, ns - 1);
        qv[m] = q[k];
        cv[m] = ev[k];
      }
#pragma unroll
      for (int m = 0; m < 4; ++m) {
        if (64 * m >= ns) break;
        const uint64_t hit = ballot(qv[m] >= ue);
        if (hit) {
          const int l = __builtin_ctzll(hit);
          hi = readlane_f64(qv[m], l);
          if (l > 0) lo = readlane_f64(qv[m], l - 1);
          code = __builtin_amdgcn_readlane(cv[m], l);
          break;
        }
        lo = readlane_f64(qv[m], 63);
      }
    } else {
      const int nch = (ns + 63) >> 6;
      const double end = q[min(64 * lane + 63, ns - 1)];
      const uint64_t mc = ballot(lane < nch && end >= ue);
      if (mc) {
        const int c = __builtin_ctzll(mc);
        if (c > 0) lo = readlane_f64(end, c - 1);
        const int k = min(64 * c + lane, ns - 1);
        const double qv = q[k];
        const int cv = ev[k];
        const int l = __builtin_ctzll(ballot(qv >= ue));
        hi = readlane_f64(qv, l);
        if (l > 0) lo = readlane_f64(qv, l - 1);
        code = __builtin_amdgcn_readlane(cv, l);
      }
    }
    take(code, ue, lo, hi, scale, total, tally);
  }
  if (PHASE && p.phases && t == 0 && lane == 0)
    for (int k = 0; k < PLAIN_PHASES; ++k) p.phases[k] = ph[k];
  TrajOut* o = p.out + t;
  if (lane == 0) {
    o->time = time;
    o->hops_done = h > prehops ? h - prehops : 0;
    o->status = status;
    o->occ[0] = occ0;
    o->occ[1] = occ1;
    o->occ[2] = td.occ[2];
    o->occ[3] = td.occ[3];
  }
  if (lane < L.P) o->eo[lane] = eo;
  if (REC && p.occ_time) {
    if (lane < N) p.occ_time[(size_t)t * NMAX + lane] = ot0;
    if (lane + 64 < N) p.occ_time[(size_t)t * NMAX + lane + 64] = ot1;
  }
  if (p.se_out && total_hops > 0) {   // the energies the last hop saw
    energies(last0, last1);
    for (int i = lane; i < N; i += 64) p.se_out[(size_t)t * NMAX + i] = se[i];
  }
}

template <bool REC, bool STAGE, bool PHASE>
__global__ void __launch_bounds__(64) kmc_plain_fp64_kernel(PlainParams p) {
  extern __shared__ __align__(16) unsigned char smem[];
  const int lane = threadIdx.x;
  int t = blockIdx.x;
  for (;;) {
    plain_trajectory<REC, STAGE, PHASE>(p, t, lane, smem);
    if (!p.queue) break;
    // (the queue counts from 0; the first gridDim.x trajectories are taken)
    if (lane == 0) t = (int)gridDim.x + atomicAdd(p.queue, 1);
    t = __builtin_amdgcn_readfirstlane(t);
    if (t >= p.ntraj) break;
    wave_lds_sync();
  }
}

template __global__ void kmc_plain_fp64_kernel<false, false, false>(PlainParams);
template __global__ void kmc_plain_fp64_kernel<true, false, false>(PlainParams);
template __global__ void kmc_plain_fp64_kernel<false, true, false>(PlainParams);
template __global__ void kmc_plain_fp64_kernel<true, true, false>(PlainParams);
template __global__ void kmc_plain_fp64_kernel<false, true, true>(PlainParams);
template __global__ void kmc_plain_fp64_kernel<false, false, true>(PlainParams);

// Possible pairs of any occupation of a layout with at most S sites and N
// acceptors: nA (cE + P) + P cE for nA occupied and cE = N - nA empty ones.
int plain_pairs(int S, int N) {
  int most = 0;
  for (int n = 0; n <= N; ++n) {
    const int P = S - n < PMAX ? S - n : PMAX;
    most = most > n * n / 4 + P * n ? most : n * n / 4 + P * n;
  }
  return (most + 3) & ~3;
}

// LDS bytes the kernel needs for S sites, N acceptors and `slots` state records.
size_t plain_lds_bytes(int S, int N, int slots, bool stage) {
  return PlainLds(S, N, plain_pairs(S, N), slots, stage).total * sizeof(double);
}

// Bytes of one state record: 1/total and total, then 10 B per possible pair.
size_t plain_state_bytes(int S, int N) {
  return (16 + 10 * (size_t)plain_pairs(S, N) + 127) & ~(size_t)127;
}

}  // namespace kmc
