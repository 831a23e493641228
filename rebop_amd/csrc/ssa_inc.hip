// ssa_inc.hip -- incremental SSA kernel for large networks: eight lanes per
// trajectory, only the propensities an event changes are evaluated again, and
// the results are those of the reference's sequential sums, bit for bit.
//
// The reference evaluates every propensity after every event and adds them in
// order (make_cumrates, src/gillespie.rs:357-364).  An event of a large
// network changes about ten of them.  This kernel keeps, per trajectory, sums
// of the propensities over blocks of reactions and updates the blocks whose
// propensities change; the total comes from the block sums and the choice
// descends super-blocks, blocks and reactions.  Those sums round differently
// from the reference's, so every decision made with them is certified, and
// one that a rounding could turn is made again the reference's way:
//
// - Propensities enter the sums quantised: q_r = rint(a_r / g), g a power of
//   two chosen so that the total Q = sum q_r lies in [2^48, 2^52).  An event's
//   differences are added one by one, so on the way a sum holds old and new
//   values at once: at most Q_old + Q_new, below 2^53 while both totals are
//   in the range.  Integers up to there are exact in binary64 whatever the
//   order of the additions, so nothing drifts.  (Where Q_new is not in the
//   range, an addition can lose a unit only above 2^53, at most
//   Q_old + Q_new - 2^53 < Q_new - 2^52 units in all, so the total found is
//   not in the range either.)  When Q leaves it the sums are rebuilt with
//   another g.
// - The reference's partial sum cum_r and g Q_r differ by at most
//   R/2 g + R 2^-53 g Q (quantisation; R rounded additions of non-negative
//   terms), which is at most 17 R 2^-53 of the total and below R units of g.
//   kappa and eps below are these bounds with room to spare.
// - The time is kept as an interval [tl, th] that holds the reference's t:
//   both ends take fl(end + E/total (1 -+ kappa)), and rounding is monotone.
//   A comparison with a sample time that the interval straddles is not
//   decided: the trajectory starts again in exact mode.  At a sample the
//   reference sets t to the sample time itself, so the interval closes there.
// - A choice whose threshold lies within epsilon of the chosen reaction's
//   boundaries is made again with the reference's sums of that state (its
//   counts are certain).
// - Exact mode: every event adds all the propensities in order and counts
//   cum_r < chosen, as the reference does.  It also serves the states the
//   bounds do not cover: a negative or NaN propensity, a negative count, a
//   total outside [1e-200, 1e200].
//
// With 512 reactions, 5e4 events and 200 samples a trajectory restarts with a
// probability of about 2e-7 and a choice is repeated about once in 1e9 events.
//
// Layout: a wave runs eight trajectories, eight lanes each.  The lanes of a
// group hold the same scalar state; they share the draws (lane j computes the
// block of the j-th of the next eight, which the group reads back from LDS one
// per event), the changed reactions (lane j takes every eighth), the scans of
// eight sums (three DPP steps) and the samples.  Counts (int32) and sums are
// in LDS, 10.3 KB a wave for 128 species and 512 reactions; the network's
// tables (reaction records, jump records with the list of reactions each jump
// changes) are read through the caches.
//
// What bounds it: VALU issue (69 % of the CU cycles with 15 waves per CU on the
// 128 x 512 network, 39 wave instructions per event against 189 of the LDS
// kernel) and the latency of an event's dependent table and LDS reads (the
// waves wait on a counter half of their time), for few trajectories that chain
// alone.  Measured against the LDS kernel: 128 species x 512
// reactions, 131072 trajectories of 13350 events 639 -> 168 ms, 64
// trajectories 217 -> 12 ms; 256 networks x 256 trajectories in one launch
// 39.1 -> 7.3 ms; 48 x 96 with 53 rate expressions, 32768 trajectories
// 510 -> 26.9 ms.
#include <hip/hip_runtime.h>

#include "rebop_expr.h"
#include "rebop_rng.h"
#include "ssa_lane.h"
#include "ssa_layout.h"

#pragma clang fp contract(off)

namespace rebop {

constexpr uint32_t kIncGroup = 8; // lanes per trajectory
constexpr uint32_t kIncTraj = 64 / kIncGroup; // trajectories per wave

// The total is kept in [kIncLo, kIncHi) units; a rebuild puts it in
// [2^kIncTarget, 2^(kIncTarget + 1)).
constexpr double kIncLo = 0x1p48, kIncHi = 0x1p52;
constexpr int32_t kIncTarget = 50;

// LDS of one wave, in bytes from its start: the draws [8][8] (E, U), a row of
// propensities per group for the sequential sums, the sums, then (STORE) the
// quantised propensities, (EXPR) the expression stacks, and the counts.
struct IncLds {
  uint32_t sum_stride, q_stride, cnt_stride; // per trajectory: doubles, doubles, int32
  uint32_t q_off, stk_off, cnt_off, bytes;
};
constexpr uint32_t kIncRow = 16u * 64u, kIncSums = kIncRow + 8u * 64u;

IncLds inc_lds(uint32_t smax, uint32_t nblk_max, uint32_t rmax, uint32_t depth, bool store) {
  IncLds l{};
  l.sum_stride = 8u + ((nblk_max + 7u) / 8u) * 8u + 1u; // odd: the groups' rows start in different banks
  l.q_stride = store ? ((rmax + 7u) / 8u) * 8u + 1u : 0u;
  l.cnt_stride = (smax + 1u) | 1u;
  l.q_off = kIncSums + 8u * kIncTraj * l.sum_stride;
  l.stk_off = l.q_off + 8u * kIncTraj * l.q_stride;
  l.cnt_off = l.stk_off + 8u * 64u * depth;
  l.bytes = (l.cnt_off + 4u * kIncTraj * l.cnt_stride + 15u) & ~15u;
  return l;
}

#if defined(__HIP_DEVICE_COMPILE__)
typedef const __attribute__((address_space(1))) uint4 *inc_g4_t;
typedef const __attribute__((address_space(1))) uint2 *inc_g2_t;
typedef const __attribute__((address_space(1))) uint32_t *inc_g1_t;
typedef __attribute__((address_space(3))) double *inc_lds_f64_t;
#else
typedef const uint4 *inc_g4_t;
typedef const uint2 *inc_g2_t;
typedef const uint32_t *inc_g1_t;
#endif

// Orders a group's LDS writes before its other lanes' reads: one wave's LDS
// operations complete in order, so only the compiler has to keep them apart.
__device__ __forceinline__ void inc_sync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

template <int CTRL>
__device__ __forceinline__ double inc_dpp(double v) {
  const uint64_t b = rebop_f64_bits(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, CTRL, 0xF, 0xF, false);
  const uint32_t hi = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), CTRL, 0xF, 0xF, false);
  return rebop_f64_from_bits(((uint64_t)hi << 32) | lo);
}
constexpr int kDppXor1 = 0xB1;    // quad_perm [1, 0, 3, 2]
constexpr int kDppXor2 = 0x4E;    // quad_perm [2, 3, 0, 1]
constexpr int kDppMirror8 = 0x141; // row_half_mirror: the other quad of an aligned eight

// STORE: the quantised propensities are kept in LDS (an update subtracts the
// stored value), else recomputed from the old counts (an LMA propensity is a
// few operations, and its LDS would cost waves).  EXPR: rate expressions.
template <bool EXPR, bool STORE>
struct IncNet {
  static_assert(STORE || !EXPR, "an expression's old value is stored, not evaluated again");
  uint32_t S, R, bsh;
  inc_g4_t rec;
  inc_g1_t irec, dep;
  inc_g4_t tok;
  uint32_t lane, j, gsh; // lane, lane in its group, the group's first lane
  double m1, m2, m4;     // 1.0 where the lane's bit is set
  int32_t *cnt;          // this trajectory's counts: [0] = 1, [s + 1] = species s
  double *sums;          // [0, 8) super-blocks, [8, ...) blocks
  double *q;             // STORE: quantised propensities
  double *row;           // eight propensities of the group
  double *stk;           // this lane's expression stack, 64 apart
  double inv_g, g;
  double eps; // units of g

  __device__ __forceinline__ double group_sum(double v) const {
    v = v + inc_dpp<kDppXor1>(v);
    v = v + inc_dpp<kDppXor2>(v);
    return v + inc_dpp<kDppMirror8>(v);
  }
  // exclusive prefix over the group's lanes; `total`: the sum (exact integers)
  __device__ __forceinline__ double scan(double v, double *total) const {
    double o = inc_dpp<kDppXor1>(v);
    double pre = o * m1;
    v = v + o;
    o = inc_dpp<kDppXor2>(v);
    pre = __builtin_fma(o, m2, pre);
    v = v + o;
    o = inc_dpp<kDppMirror8>(v);
    pre = __builtin_fma(o, m4, pre);
    *total = v + o;
    return pre;
  }
  // the group's lanes for which `p` holds, as eight bits
  __device__ __forceinline__ uint32_t group_mask(bool p) const {
    return (uint32_t)(__ballot(p) >> gsh) & 0xffu;
  }
  // v of lane `l` of the group
  __device__ __forceinline__ double group_get(double v, uint32_t l) const {
    const uint64_t b = rebop_f64_bits(v);
    const int at = (int)((gsh + l) * 4u);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)(b >> 32));
    return rebop_f64_from_bits(((uint64_t)hi << 32) | lo);
  }

  // Expr::eval (src/expr.rs:24-38) of tokens b .. e-1 (layout in
  // ssa_layout.h): the top of the stack in a register, the values below it in
  // this lane's LDS column.  The lanes of a wave run different programs.
  __device__ double expr_rate(uint32_t b, uint32_t e) const {
    double top = 0.0;
    uint32_t sp = 0;
    uint4 nx = tok[b];
    for (uint32_t i = b; i < e; ++i) {
      const uint4 t = nx;
      nx = tok[i + 1]; // the table ends with a token of padding
      const uint32_t op = t.x & 0xffu, src = t.x >> 8;
      double y = rebop_f64_from_bits(((uint64_t)t.w << 32) | t.z);
      if (src == REBOP_TOK_SPECIES) y = (double)cnt[t.y];
      double x = top;
      if (src == REBOP_TOK_STACK) {
        y = top;
        if (op != REBOP_OP_NEG && op != REBOP_OP_EXP) x = stk[--sp * 64u];
      }
      switch (op) {
      case REBOP_OP_CONST: // push
        stk[sp++ * 64u] = top;
        top = y;
        break;
      case REBOP_OP_NEG: top = -y; break;
      case REBOP_OP_EXP: top = rebop_exp64(y); break;
      case REBOP_OP_ADD: top = x + y; break;
      case REBOP_OP_SUB: top = x - y; break;
      case REBOP_OP_MUL: top = x * y; break;
      case REBOP_OP_DIV: top = x / y; break;
      case REBOP_OP_POW: top = rebop_pow64(x, y); break;
      case REBOP_OP_MAX: top = rebop_fmax64(x, y); break;
      default: top = rebop_fmin64(x, y); break;
      }
    }
    return top;
  }

  // Rate::rate (src/gillespie.rs:71-90) of a record
  __device__ __forceinline__ double rate_of(const uint4 &w) const {
    if constexpr (EXPR)
      if (w.w & REBOP_REC_SLOW_FACTORS) return expr_rate(w.x, w.y);
    double a = rebop_f64_from_bits(((uint64_t)w.y << 32) | w.x);
    a = a * (double)(cnt[w.z >> 16] - (int32_t)(w.z & 0xfffu));
    a = a * (double)(cnt[w.w >> 16] - (int32_t)(w.w & 0xfffu));
    return a;
  }
  __device__ __forceinline__ double rate(uint32_t r) const {
    const uint4 w = rec[r];
    return rate_of(w);
  }
  __device__ __forceinline__ double quant(double a) const { return __builtin_rint(a * inv_g); }

  __device__ __forceinline__ void add_sums(uint32_t r, double d) const {
    const uint32_t b = r >> bsh;
#if defined(__HIP_DEVICE_COMPILE__)
    (void)__builtin_amdgcn_ds_atomic_fadd_f64((inc_lds_f64_t)(sums + 8u + b), d);
    (void)__builtin_amdgcn_ds_atomic_fadd_f64((inc_lds_f64_t)(sums + (b >> 3)), d);
#else
    (void)b;
    (void)d;
#endif
  }

  // All propensities and sums from the counts, with a new g.  False: the
  // bounds do not cover this state.  *tq: the total in units of g.
  __device__ bool rebuild(double *tq) {
    double s = 0.0;
    bool bad = false;
#pragma unroll 1
    for (uint32_t r = j; r < R; r += kIncGroup) {
      const double a = rate(r);
      bad = bad || !(a >= 0.0);
      if constexpr (STORE) q[r] = a;
      s = s + a;
    }
    s = group_sum(s);
    *tq = 0.0;
    if (group_mask(bad) != 0u) return false;
    if (s == 0.0) { // absorbing: every propensity is zero
      g = 0.0;
      return true;
    }
    if (!(s > 1e-200 && s < 1e200)) return false;
    const int32_t e = (int32_t)(rebop_f64_bits(s) >> 52) - 1023;
    g = rebop_pow2i(e - kIncTarget);
    inv_g = rebop_pow2i(kIncTarget - e);
    const uint32_t ns = 8u + ((((R - 1u) >> bsh) >> 3) + 1u) * 8u;
    for (uint32_t i = j; i < ns; i += kIncGroup) sums[i] = 0.0;
    inc_sync();
    double t = 0.0;
#pragma unroll 1
    for (uint32_t r0 = 0; r0 < R; r0 += kIncGroup) {
      const uint32_t r = r0 + j;
      double v = 0.0;
      if (r < R) {
        if constexpr (STORE) {
          v = quant(q[r]);
          q[r] = v;
        } else {
          v = quant(rate(r));
        }
      }
      v = group_sum(v);
      t = t + v;
      if (j == 0) add_sums(r0, v);
    }
    inc_sync();
    *tq = t;
    return true;
  }

  // make_cumrates in the reference's order; with `count`, also the number of
  // partial sums below `chosen`
  __device__ double sequential(double chosen, uint32_t *count) const {
    double acc = 0.0;
    uint32_t k = 0;
#pragma unroll 1
    for (uint32_t r0 = 0; r0 < R; r0 += kIncGroup) {
      const uint32_t r = r0 + j;
      const double a = r < R ? rate(r) : 0.0;
      inc_sync(); // the previous eight are read
      row[j] = a;
      inc_sync();
      const uint32_t m = R - r0 < kIncGroup ? R - r0 : kIncGroup;
      for (uint32_t i = 0; i < m; ++i) {
        acc = acc + row[i];
        k += acc < chosen ? 1u : 0u;
      }
    }
    if (count) *count = k;
    return acc;
  }

  // The reaction whose interval of the sums holds c (units of g); false: c is
  // within eps of one of its ends.  pre: this lane's super-block prefix.
  __device__ bool choose(double c, double pre, double sup, uint32_t *out) const {
    uint32_t w = (uint32_t)__popc(group_mask(pre + sup < c));
    w = w < 7u ? w : 7u;
    double base = group_get(pre, w);
    double tot;
    double v = sums[8u + 8u * w + j];
    double p = scan(v, &tot) + base;
    uint32_t b = (uint32_t)__popc(group_mask(p + v < c));
    b = b < 7u ? b : 7u;
    base = group_get(p, b);
    const uint32_t r1 = (8u * w + b) << bsh;
    const uint32_t r2 = r1 + (1u << bsh) < R ? r1 + (1u << bsh) : R;
    bool ok = false;
#pragma unroll 1
    for (uint32_t r0 = r1; r0 < r2; r0 += kIncGroup) {
      const uint32_t r = r0 + j;
      v = 0.0;
      if (r < r2) {
        if constexpr (STORE) v = q[r];
        else v = quant(rate(r));
      }
      p = scan(v, &tot) + base;
      const uint32_t n = (uint32_t)__popc(group_mask(p + v < c));
      if (n < kIncGroup) {
        ok = group_mask(j == n && r < r2 && c - p > eps && (p + v) - c > eps) != 0u;
        *out = r0 + n;
        break;
      }
      base = base + tot;
    }
    return ok;
  }
};

template <bool EXPR, bool STORE>
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(EXPR ? 2 : 4))) ssa_inc_kernel(const rebop_dev_job *__restrict__ jobs,
                                                     const uint32_t *__restrict__ tickets,
                                                     uint32_t n_tickets, unsigned long long *counters,
                                                     unsigned long long *job_events,
                                                     unsigned long long *job_queue, IncLds lay,
                                                     uint32_t rerun) {
  extern __shared__ __attribute__((aligned(16))) char inc_lds_mem[];
  const uint32_t lane = __lane_id();
  IncNet<EXPR, STORE> net;
  net.lane = lane;
  net.j = lane & (kIncGroup - 1u);
  net.gsh = lane & ~(kIncGroup - 1u);
  const uint32_t grp = lane / kIncGroup, j = net.j;
  net.m1 = (j & 1u) ? 1.0 : 0.0;
  net.m2 = (j & 2u) ? 1.0 : 0.0;
  net.m4 = (j & 4u) ? 1.0 : 0.0;
  double2 *draws = (double2 *)inc_lds_mem + grp * kIncGroup;
  net.row = (double *)(inc_lds_mem + kIncRow) + grp * kIncGroup;
  net.sums = (double *)(inc_lds_mem + kIncSums) + grp * lay.sum_stride;
  net.q = (double *)(inc_lds_mem + lay.q_off) + grp * lay.q_stride;
  net.stk = (double *)(inc_lds_mem + lay.stk_off) + lane;
  net.cnt = (int32_t *)(inc_lds_mem + lay.cnt_off) + grp * lay.cnt_stride;
  if (j == 0) net.cnt[0] = 1; // the count an absent factor reads
  LaneTotals total;
  for (;;) {
    if (rerun && __ballot(launch_flagged(counters, REBOP_FLAG_NARROW)) != 0ull) break;
    unsigned long long got = 0ull;
    if (lane == 0) got = atomicAdd(&counters[REBOP_CTR_QUEUE], 1ull);
    const uint32_t it = __builtin_amdgcn_readfirstlane(
        (uint32_t)(got < (unsigned long long)n_tickets ? got : (unsigned long long)n_tickets));
    if (it >= n_tickets) break;
    const uint32_t jid = tickets ? __builtin_amdgcn_readfirstlane(tickets[it]) : 0u;
    const rebop_dev_job &job = jobs[jid];
    net.S = job.S;
    net.R = job.R;
    net.bsh = job.inc_bsh;
    net.rec = (inc_g4_t)(const void *)job.rec;
    net.irec = (inc_g1_t)(const void *)job.inc_rec;
    net.dep = (inc_g1_t)(const void *)job.inc_dep;
    net.tok = (inc_g4_t)(const void *)job.inc_tok;
    net.eps = 4.0 * (double)job.R + 8.0;
    net.inv_g = net.g = 0.0;
    const double kappa = (32.0 * (double)job.R + 32.0) * 0x1p-53;
    const uint64_t n = job.n_traj;
    const uint32_t nb = (uint32_t)job.nb_steps;
    const uint64_t Sn = (uint64_t)job.S * n;
    rebop_dev_run run{}; // what grid_time reads
    run.tmax = job.tmax;
    run.nb_steps = job.nb_steps;
    run.mode = REBOP_MODE_GRID;

    LaneTotals acc;
    uint64_t jl = 0, draw = 0;
    double tl = 0.0, th = 0.0, T = 0.0, tot = 0.0, tq = 0.0, pre = 0.0, sup = 0.0;
    uint32_t i = 0, ov = 0;
    bool alive = true, need = true, redo = false, exact = false, fresh = false;
    rebop_stream st = rebop_stream_of(job.seed, 0ull);
    // what a change of counts does to the totals (make_cumrates)
    auto exact_total = [&]() {
      tot = net.sequential(0.0, nullptr);
      if (tot == __builtin_inf()) {
        acc.flags |= REBOP_FLAG_RANGE; // time would stop: an absorbing state from here
        tot = 0.0;
      }
    };
    auto load_prefixes = [&]() {
      sup = net.sums[j];
      pre = net.scan(sup, &tq);
    };
#pragma unroll 1
    for (uint32_t p = 0;; p = (p + 1u) & 7u) {
      if (alive && need) {
        if (!redo) {
          // the next trajectory: one atomic per wave for all groups asking
          const uint64_t mask = __ballot(1);
          const int leader = __ffsll((unsigned long long)mask) - 1;
          unsigned long long base = 0ull;
          const bool stop = rerun && __ballot(launch_flagged(counters, REBOP_FLAG_NARROW)) != 0ull;
          if ((int)lane == leader && !stop)
            base = atomicAdd(&job_queue[jid], (unsigned long long)(__popcll(mask) / kIncGroup));
          base = __shfl(base, leader);
          jl = base + (uint64_t)(__popcll(mask & ((1ull << net.gsh) - 1ull)) / kIncGroup);
          if (stop || jl >= n) alive = false;
        }
        if (alive) {
          st = rebop_stream_of(job.seed, job.traj_begin + jl);
          const int64_t *src = job.x0_div ? job.x0 + (jl / job.x0_div) * job.S : job.x0;
          bool neg = false;
          inc_sync();
          for (uint32_t s = j; s < net.S; s += kIncGroup) {
            int64_t v = src[s];
            if (v > (int64_t)REBOP_LDS_LIMIT || v < -(int64_t)REBOP_LDS_LIMIT) {
              acc.flags |= REBOP_FLAG_NARROW;
              v = 0;
            }
            if (v > REBOP_LDS16_LIMIT || v < -REBOP_LDS16_LIMIT) acc.flags |= REBOP_FLAG_PAST16;
            net.cnt[s + 1u] = (int32_t)v;
            neg = neg || v < 0;
          }
          inc_sync();
          exact = redo || net.group_mask(neg) != 0u;
          tl = th = 0.0;
          draw = 0;
          i = 0;
          ov = 0;
          T = grid_time(run, 0);
          need = redo = false;
          fresh = true;
          if (!exact) {
            exact = !net.rebuild(&tq); // the time is certain here: no restart
            if (!exact) {
              tot = tq * net.g;
              if (0.0 < tq) load_prefixes();
            }
          }
          if (exact) exact_total();
        }
      }
      if (__ballot(alive) == 0ull) break;
      // the next eight draws of every trajectory (of a new one: those left of
      // this round), lane j's at slot j
      if (alive && (p == 0u || fresh)) {
        const rebop_u32x4 blk = rebop_stream_block(st, draw + j - p);
        inc_sync();
        draws[j] = make_double2(rebop_exp1_of(blk), rebop_unif_of(blk));
        inc_sync();
        fresh = false;
      }
      if (alive) {
        const double2 eu = draws[p];
        const bool live = 0.0 < tot;
        const double dt = eu.x / tot; // unused in an absorbing state
        const double tnl = tl + dt * (exact ? 1.0 : 1.0 - kappa);
        const double tnh = th + dt * (exact ? 1.0 : 1.0 + kappa);
        const bool rec = !live || tnl > T;
        if (live && !rec && tnh > T) {
          need = redo = true; // the interval holds the sample time
        } else if (rec) {
          draw += live ? 1u : 0u;
          ov += live ? 1u : 0u;
          if (job.out) {
            int64_t *o = job.out + (uint64_t)i * Sn + jl;
            for (uint32_t s = j; s < net.S; s += kIncGroup) o[(uint64_t)s * n] = (int64_t)net.cnt[s + 1u];
          }
          // a launch that will be rerun: drop the work once a count left int32
          if (rerun && (i & 7u) == 7u && net.group_mask(launch_flagged(counters, REBOP_FLAG_NARROW)) != 0u)
            need = true;
          tl = th = T;
          i += 1;
          if (i > nb) {
            if (job.final_x)
              for (uint32_t s = j; s < net.S; s += kIncGroup)
                job.final_x[(uint64_t)s * n + jl] = (int64_t)net.cnt[s + 1u];
            if (j == 0) {
              acc.events += draw - ov;
              acc.draws += draw;
              acc.trajectories += 1;
            }
            need = true;
          } else {
            T = grid_time(run, i);
          }
        } else {
          draw += 1;
          tl = tnl;
          th = tnh;
          uint32_t k = 0;
          if (exact || !net.choose(tq * eu.y, pre, sup, &k)) {
            const double full = exact ? tot : net.sequential(0.0, nullptr);
            (void)net.sequential(full * eu.y, &k);
            k = k < net.R ? k : net.R - 1u; // the last sum is the total: never below
          }
          // the jump (Jump::affect, src/gillespie.rs:142-152) and the
          // reactions it changes
          const uint32_t word = net.irec[k * REBOP_IREC_WORDS + (j & 3u)];
          const uint2 list = *(inc_g2_t)(net.irec + k * REBOP_IREC_WORDS + 4u);
          const uint32_t cs = (word & 0xffu) + 1u;
          const int32_t cd = j < 4u ? (int32_t)word >> 8 : 0;
          bool neg = false, bad = false;
          auto apply = [&]() {
            if (cd != 0) {
              // |count| <= 2^30 and |cd| < 2^23: no wrap before the check
              const int32_t v = (int32_t)((uint32_t)net.cnt[cs] + (uint32_t)cd);
              net.cnt[cs] = v;
              neg = v < 0;
              if (v > REBOP_LDS_LIMIT || v < -REBOP_LDS_LIMIT) acc.flags |= REBOP_FLAG_NARROW;
              if (v > REBOP_LDS16_LIMIT || v < -REBOP_LDS16_LIMIT) acc.flags |= REBOP_FLAG_PAST16;
            }
          };
          if (exact) {
            inc_sync();
            apply();
            inc_sync();
            exact_total();
          } else {
            if constexpr (STORE) {
              apply();
              inc_sync();
            }
            const uint32_t e1 = list.x + list.y;
#pragma unroll 1
            for (uint32_t e = list.x + j; e < e1; e += kIncGroup) {
              const uint32_t d = net.dep[e], r = d & 0xffffu;
              const uint4 w = net.rec[r];
              if constexpr (STORE) {
                const double a = net.rate_of(w);
                bad = bad || !(a >= 0.0);
                const double v = net.quant(a);
                const double old = net.q[r];
                net.q[r] = v;
                net.add_sums(r, v - old);
              } else {
                // the factors before the jump, and by how much it moves each
                const int32_t f1 = net.cnt[w.z >> 16] - (int32_t)(w.z & 0xfffu);
                const int32_t f2 = net.cnt[w.w >> 16] - (int32_t)(w.w & 0xfffu);
                const double kr = rebop_f64_from_bits(((uint64_t)w.y << 32) | w.x);
                const double a0 = kr * (double)f1 * (double)f2;
                const double a1 = kr * (double)(f1 + ((int32_t)(d << 8) >> 24)) *
                                  (double)(f2 + ((int32_t)d >> 24));
                net.add_sums(r, net.quant(a1) - net.quant(a0));
              }
            }
            inc_sync();
            if constexpr (!STORE) {
              apply();
              inc_sync();
            }
            if (net.group_mask(neg || bad) != 0u) {
              need = redo = true;
            } else {
              load_prefixes();
              if (!(tq >= kIncLo && tq < kIncHi)) {
                if (net.rebuild(&tq)) {
                  if (0.0 < tq) load_prefixes();
                } else {
                  need = redo = true;
                }
              }
              tot = tq * net.g;
            }
          }
          if (rerun && net.group_mask((acc.flags & REBOP_FLAG_NARROW) != 0u) != 0u) {
            // tell the others at once
            if (j == 0) atomicOr(&counters[REBOP_CTR_FLAGS], (unsigned long long)REBOP_FLAG_NARROW);
            need = true;
            redo = false;
          }
        }
      }
    }
    if (job_events) {
      unsigned long long e = acc.events;
#pragma unroll
      for (int off = 32; off >= 1; off >>= 1) e += __shfl_xor(e, off);
      if (lane == 0 && e) atomicAdd(&job_events[jid], e);
    }
    total.events += acc.events;
    total.draws += acc.draws;
    total.trajectories += acc.trajectories;
    total.flags |= acc.flags;
  }
  flush_wave_totals(total, counters);
}

static const void *inc_kernel_ptr(bool expr, bool store) {
  return expr ? (const void *)&ssa_inc_kernel<true, true>
         : store ? (const void *)&ssa_inc_kernel<false, true>
                 : (const void *)&ssa_inc_kernel<false, false>;
}

// Bytes of LDS of a wave for the largest of a set of networks.
size_t inc_lds_bytes(uint32_t smax, uint32_t nblk_max, uint32_t rmax, uint32_t depth, bool store) {
  return inc_lds(smax, nblk_max, rmax, depth, store).bytes;
}

hipError_t inc_occupancy(size_t lds, bool expr, bool store, int *blocks_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, inc_kernel_ptr(expr, store), 64, lds);
}

// tickets: job indices, one per unit of work (NULL: all of job 0).
hipError_t launch_inc(const rebop_dev_job *jobs, const uint32_t *tickets, uint32_t n_tickets,
                      unsigned long long *counters, unsigned long long *job_events,
                      unsigned long long *job_queue, int blocks, uint32_t smax, uint32_t nblk_max,
                      uint32_t rmax, uint32_t depth, bool expr, bool store, bool rerun,
                      hipStream_t stream) {
  const IncLds lay = inc_lds(smax, nblk_max, rmax, depth, store);
  if (lay.bytes > 64 * 1024) {
    const hipError_t e = hipFuncSetAttribute(inc_kernel_ptr(expr, store),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, (int)lay.bytes);
    if (e != hipSuccess) return e;
  }
  const uint32_t rr = rerun ? 1u : 0u;
  if (expr)
    hipLaunchKernelGGL((ssa_inc_kernel<true, true>), dim3(blocks), dim3(64), lay.bytes, stream, jobs,
                       tickets, n_tickets, counters, job_events, job_queue, lay, rr);
  else if (store)
    hipLaunchKernelGGL((ssa_inc_kernel<false, true>), dim3(blocks), dim3(64), lay.bytes, stream, jobs,
                       tickets, n_tickets, counters, job_events, job_queue, lay, rr);
  else
    hipLaunchKernelGGL((ssa_inc_kernel<false, false>), dim3(blocks), dim3(64), lay.bytes, stream, jobs,
                       tickets, n_tickets, counters, job_events, job_queue, lay, rr);
  return hipGetLastError();
}

} // namespace rebop
