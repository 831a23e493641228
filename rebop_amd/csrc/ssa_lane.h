// ssa_lane.h -- the per-lane SSA engine, shared by every kernel.
//
// One trajectory per lane.  Each lane runs rebop's grid loop
// (src/pyo3_gillespie.rs:200-208) around Gillespie::advance_until
// (src/gillespie.rs:315-344) as a state machine whose every iteration is one
// exponential draw (or, in an absorbing state, one sample without a draw):
//
//   tot <= 0 or NaN  -> absorbing: sample i sees the current counts, no draw
//                       (gillespie.rs:323-326)
//   t + E/tot > T_i  -> overshoot: t = T_i, sample i, the draw is discarded
//                       (gillespie.rs:327-331); counts are unchanged, so the
//                       cumulative propensities are reused for T_{i+1}
//   otherwise        -> event: chosen = tot*U, k = #{r : cum_r < chosen}
//                       (choose_cumrate_sum, gillespie.rs:402-407), apply
//                       reaction k (Jump::affect, :142-152); the propensities
//                       are recomputed in the reference's order (make_cumrates
//                       :357-364 over Rate::rate :71-90) right after the jump
//
// A watchdog the reference does not have: with run.draw_cap set, a
// trajectory whose draws in this launch reach the cap is stopped at that
// event (its state is treated as absorbing from there), so a trajectory whose
// propensity keeps growing cannot hold its wave, and the launch, forever.
// The run then reports REBOP_FLAG_CAP.  The check is compiled in only for
// policies with Net::kCap (the host launches those when a cap is set), so
// uncapped runs pay nothing for it.
//
// The network enters through a policy object `net`.  The lane's register
// state is two local arrays of lane_loop, double x[Net::MS] (counts, for
// policies that keep them in VGPRs) and double cum[Net::MR] (what choose
// needs), handed to every policy call (local arrays, not struct members, so
// that the compiler keeps them in VGPRs even when x is indexed by a
// wave-uniform runtime species index):
//   static constexpr bool kCap;  compile the draw-cap checks in
//   static constexpr uint32_t kRangeFlag;  raised when in_range fails (REBOP_FLAG_EXACT
//                                          marks f64 counts, checked every 2^31 draws)
//   static constexpr uint32_t kStopFlag;   nonzero: once this flag is raised anywhere the
//                                          launch may be rerun (bool may_stop: it will),
//                                          so lanes stop early
//   uint32_t S() const;
//   run cold_run(run);                  the launch's parameters again, for the places off the
//                                          event loop: a policy may hand out a reference whose
//                                          fields are loaded there instead of held throughout
//   void start(const rebop_dev_run &run, uint64_t j);    per-trajectory setup (rates)
//   void load_x0(X &x, const int64_t *src);                counts from an int64 row
//   void load_state(X &x, const double *st, uint64_t stride);  st[s * stride]
//   void store_state(const X &x, double *st, uint64_t stride);
//   void write_counts(const X &x, int64_t *dst, uint64_t stride);  dst[s * stride]
//   void write_raw(const X &x, int64_t *dst, uint64_t stride);     the samples: as
//        write_counts, or (counts in f64) their f64 bits, which a pass after
//        the launch converts in place (raw_counts_to_int64)
//   bool in_range(const X &x);          counts inside the exactly simulated range
//   double grid_time(const rebop_dev_run &run, uint64_t i);   sample time i
//   double props(X &x, C &cum);         make_cumrates -> total
//   uint32_t choose(X &x, C &cum, double chosen);   a reaction, or >= R for none
//   void affect(X &x, uint32_t k);                   (then no change)
// so that one loop serves counts in VGPRs (reg_* helpers below) and in LDS,
// for a data-driven network or one compiled into the kernel.
//
// A persistent launch refills a finished lane with the next trajectory id
// from a device-wide counter: one atomic per wave per refill (ballot over the
// finished lanes, rank by popcount).
#ifndef REBOP_SSA_LANE_H
#define REBOP_SSA_LANE_H

#include "rebop_rng.h"
#include "ssa_layout.h"

#if defined(__clang__)
#pragma clang fp contract(off)
#endif

namespace rebop {

__device__ __forceinline__ double grid_time(double tmax, uint64_t i, uint64_t nb) {
  // src/pyo3_gillespie.rs:202: tmax * i as f64 / nb_steps as f64
  return tmax * (double)i / (double)nb;
}

__device__ __forceinline__ double grid_time(const rebop_dev_run &run, uint64_t i) {
  if (run.mode == REBOP_MODE_TARGET) return run.tmax;
  return grid_time(run.tmax, i, run.nb_steps);
}

// The sample time from the table written before the launch (same value).
__device__ __forceinline__ double table_time(const rebop_dev_run &run, uint64_t i) {
  return run.grid[i];
}

struct LaneTotals {
  uint64_t events = 0, draws = 0;
  uint32_t trajectories = 0, flags = 0;
};

// Helpers for counts held in VGPRs as exact FP64 integers (species >= S stay 0).
template <int MS>
__device__ __forceinline__ void reg_load_x0(double (&x)[MS], const int64_t *src, uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s) x[s] = s < (int)S ? (double)src[s] : 0.0;
}
template <int MS>
__device__ __forceinline__ void reg_load_state(double (&x)[MS], const double *st, uint64_t stride,
                                               uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s) x[s] = s < (int)S ? st[(uint64_t)s * stride] : 0.0;
}
template <int MS>
__device__ __forceinline__ void reg_store_state(const double (&x)[MS], double *st, uint64_t stride,
                                                uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) st[(uint64_t)s * stride] = x[s];
}
template <int MS>
__device__ __forceinline__ void reg_write_counts(const double (&x)[MS], int64_t *dst,
                                                 uint64_t stride, uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) dst[(uint64_t)s * stride] = (int64_t)x[s];
}
// The sample's counts as their f64 bits (8 bytes each, in the int64 slots):
// the conversion, five FP64 operations per count, runs after the launch in
// a streaming pass instead of in the event loop.
template <int MS>
__device__ __forceinline__ void reg_write_raw(const double (&x)[MS], int64_t *dst, uint64_t stride,
                                              uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) dst[(uint64_t)s * stride] = (int64_t)rebop_f64_bits(x[s]);
}

// A buffer of `n` bytes at p (below 4 GiB): stores at a byte offset, dropped
// where that is n or more.
#if defined(__HIP_DEVICE_COMPILE__)
typedef __amdgpu_buffer_rsrc_t ByteBuffer;
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ ByteBuffer byte_buffer(void *p, uint32_t n) {
  return __builtin_amdgcn_make_buffer_rsrc(p, 0, (int)n, 0x00020000);
}
#else
struct ByteBuffer {};
__device__ __forceinline__ ByteBuffer byte_buffer(void *, uint32_t) { return ByteBuffer{}; }
#endif
// reg_write_raw to byte `at`, the species `stride` bytes apart
template <int MS>
__device__ __forceinline__ void reg_write_raw_buffer(const double (&x)[MS], ByteBuffer buf, uint32_t at,
                                                     uint32_t stride, uint32_t S) {
#if defined(__HIP_DEVICE_COMPILE__)
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) {
      const uint64_t b = rebop_f64_bits(x[s]);
      __builtin_amdgcn_raw_buffer_store_b64(u32x2_t{(uint32_t)b, (uint32_t)(b >> 32)}, buf, (int)at,
                                            (int)(s * stride), 0);
    }
#endif
}

// Counts in [0, 2^50), tested like reg_in_range, and their conversion: adding
// 1.5 2^52 leaves the integer (also a slightly negative one) in the low bits.
template <int MS>
__device__ __forceinline__ bool reg_small(const double (&x)[MS], uint32_t S) {
  uint32_t m = 0;
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) {
      const uint32_t h = (uint32_t)(rebop_f64_bits(x[s]) >> 32);
      m = m > h ? m : h;
    }
  return m < 0x43100000u;
}
template <int MS>
__device__ __forceinline__ void reg_write_small(const double (&x)[MS], int64_t *dst, uint32_t S) {
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) dst[s] = (int64_t)(rebop_f64_bits(x[s] + 0x1.8p52) - 0x4338000000000000ull);
}

template <int MS>
__device__ __forceinline__ bool reg_in_range(const double (&x)[MS], uint32_t S) {
  // the largest high word, as unsigned, is below 2^52's unless a count is
  // negative or near the limit: only then the counts are looked at one by one
  uint32_t m = 0;
#pragma unroll
  for (int s = 0; s < MS; ++s)
    if (s < (int)S) {
      const uint32_t h = (uint32_t)(rebop_f64_bits(x[s]) >> 32);
      m = m > h ? m : h;
    }
  bool ok = true;
  if (__builtin_expect(m >= 0x43300000u, 0)) {
#pragma unroll
    for (int s = 0; s < MS; ++s)
      if (s < (int)S) ok = ok && (__builtin_fabs(x[s]) <= REBOP_EXACT_LIMIT);
  }
  return ok;
}

// The next local trajectory index of a lane: its own `first` the first time,
// then (persistent launches) queue_offset + an index from the device queue,
// one atomic per wave (ballot over the lanes asking, rank by popcount).
template <class Run>
__device__ __forceinline__ uint64_t next_trajectory(Run &run, bool &started, uint64_t first,
                                                    uint64_t queue_offset) {
  if (!started) {
    started = true;
    return first;
  }
  if (!run.persistent) return run.n_traj;
  const uint64_t mask = __ballot(1);
  const uint32_t lane = __lane_id();
  const int leader = __ffsll((unsigned long long)mask) - 1;
  unsigned long long base = 0ull;
  if ((int)lane == leader) base = atomicAdd(run.queue, (unsigned long long)__popcll(mask));
  base = __shfl(base, leader);
  return queue_offset + base + (uint64_t)__popcll(mask & ((1ull << lane) - 1ull));
}

// Whether some lane of this launch raised `flag` (a launch that will be
// rerun: the rest of its work would be thrown away).
__device__ __forceinline__ bool launch_flagged(const unsigned long long *counters, uint32_t flag) {
  return (__hip_atomic_load(&counters[REBOP_CTR_FLAGS], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) &
          flag) != 0ull;
}
__device__ __forceinline__ bool launch_stopped(const rebop_dev_run &run, uint32_t flag) {
  return launch_flagged(run.counters, flag);
}

// The draw count at which a trajectory that started this launch with d0
// draws hits the watchdog (never, without a cap).
__device__ __forceinline__ uint64_t cap_limit(const rebop_dev_run &run, uint64_t d0) {
  const uint64_t c = run.draw_cap;
  return (c == 0ull || d0 + c < d0) ? ~0ull : d0 + c;
}

// A trajectory reached the draw cap: flag the run, count it once (`lead`),
// and return the total propensity that makes its state absorbing from here.
__device__ __forceinline__ double hit_cap(const rebop_dev_run &run, LaneTotals &acc, bool lead) {
  acc.flags |= REBOP_FLAG_CAP;
  if (lead) atomicAdd(&run.counters[REBOP_CTR_CAPPED], 1ull);
  return 0.0;
}

// How far above the usual totals' lower end `tot` is: kUsualSpan or more if it
// is not a usual total.
constexpr uint32_t kUsualSpan = 1400u << 20;
__device__ __forceinline__ uint32_t usual_distance(double tot) {
  return (uint32_t)(rebop_f64_bits(tot) >> 32) - ((1023u - 700u) << 20);
}

// Whether a total propensity lies in [2^-700, 2^700): positive, finite, and
// far from where a division of an exponential (0 or 2^-53 .. 37) by it needs
// scaling.  One range test of the high word stands for the tests for zero,
// negative, NaN and infinite totals, which then cost nothing per event.
__device__ __forceinline__ bool usual_total(double tot) {
  return usual_distance(tot) < kUsualSpan;
}

// E / tot, correctly rounded, for a usual total: Markstein's division, the
// reciprocal refined by two Newton-Raphson steps and the quotient corrected by
// its exact remainder (IBM Journal of Research and Development 34, 1990).  The
// scaling and the special cases of a general division change nothing in this
// range.
__device__ __forceinline__ double usual_quotient(double e, double tot) {
  double y = __builtin_amdgcn_rcp(tot);
  y = __builtin_fma(y, __builtin_fma(-tot, y, 1.0), y);
  y = __builtin_fma(y, __builtin_fma(-tot, y, 1.0), y);
  const double q = e * y;
  return __builtin_fma(__builtin_fma(-tot, q, e), y, q);
}

// make_cumrates after a change of the counts, and whether the total is a
// usual one.  An infinite total would stop time (E / tot == 0) for good: it
// flags the run and is returned as 0, so the trajectory runs out as an
// absorbing state and every lane finishes.
template <class Net, class X, class C>
__device__ __forceinline__ double props_checked(Net &net, X &x, C &cum, LaneTotals &acc,
                                                bool &usual) {
  double tot = net.props(x, cum);
  usual = usual_total(tot);
  if (__builtin_expect(!usual, 0)) {
    if (tot == __builtin_inf()) {
      acc.flags |= REBOP_FLAG_RANGE;
      tot = 0.0;
    }
  }
  return tot;
}

// One lane per trajectory is bound by VALU issue: an iteration of the dimer
// network's launch (10^6 trajectories, 1.7e10 events) issues about 125 vector
// instructions.  With the range test above in place of the tests for absorbing
// and infinite totals and of the division's scaling, jumps read as fields of
// a word, a seven-instruction reduction of the logarithm's argument with its
// polynomial's constants in scalar registers, and the parameters off the event
// loop loaded where they are used (75 instead of 91 VGPRs, no spilled scalar
// registers), that launch takes 84.5 ms against 97.0 ms.
//
// Runs trajectories on this lane until none is left.  `first` is the lane's
// first local trajectory index (>= run.n_traj for none); a persistent launch
// then takes indices queue_offset + atomicAdd(queue) from the device queue.
// `ln_tab`: the ln table, or the workgroup's copy of it in LDS.
template <class Net>
__device__ __forceinline__ LaneTotals lane_loop(Net &net, const rebop_dev_run &run, uint64_t first,
                                                uint64_t queue_offset,
                                                const double (*ln_tab)[4] = rebop_ln_table) {
  const uint64_t n = run.n_traj;
  const uint32_t nb = run.mode == REBOP_MODE_TARGET ? 0u : (uint32_t)run.nb_steps;
  const uint64_t Sn = (uint64_t)net.S() * n;

  double x[Net::MS];
  double cum[Net::MR];
#pragma unroll
  for (int s = 0; s < Net::MS; ++s) x[s] = 0.0;
#pragma unroll
  for (int r = 0; r < Net::MR; ++r) cum[r] = 0.0;
  double tot = 0.0, t = 0.0, T = 0.0;
  uint64_t draw = 0, draw0 = 0, mark = 0, jl = 0, dlim = ~0ull;
  int64_t *orec = nullptr; // run.out + jl + i Sn (unused without run.out)
  uint32_t i = 0, ov = 0;
  LaneTotals acc;
  bool done = true, started = false, spill = false, usual = false;
  bool stop = false; // (kStopFlag) the launch will be rerun: take nothing more
  rebop_stream st = rebop_stream_of(run.seed, 0ull);

  for (;;) {
    bool leave = false;
    if (done) {
      // next trajectory: the lane's own first index, then (persistent
      // launches) indices from the device-wide queue
      if constexpr (Net::kStopFlag != 0u)
        stop = stop || (net.may_stop && launch_stopped(run, Net::kStopFlag));
      auto &cold = net.cold_run(run);
      const uint64_t nj = stop ? n : next_trajectory(cold, started, first, queue_offset);
      if (nj >= n) {
        leave = true;
      } else {
        jl = nj;
        st = rebop_stream_of(run.seed, cold.traj_begin + jl); // the key stays in scalar registers
        net.start(run, jl);
        if (cold.st_x) {
          net.load_state(x, cold.st_x + jl, n);
          t = cold.st_t[jl];
          draw = cold.st_draw[jl];
        } else {
          net.load_x0(x, cold.x0_div ? cold.x0 + (jl / cold.x0_div) * net.S() : cold.x0);
          t = 0.0;
          draw = 0;
        }
        if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
        draw0 = draw;
        mark = draw;
        if constexpr (Net::kCap) dlim = cap_limit(run, draw);
        ov = 0;
        i = 0;
        T = net.grid_time(run, 0);
        orec = run.out + jl;
        done = false;
        tot = props_checked(net, x, cum, acc, usual);
      }
    }
    // Tail hand-off.  In a persistent launch a lane leaves the loop only when
    // the queue is empty, so a thin wave means no work is left to take: its
    // remaining lanes leave too and write their state out below, and a
    // grouped launch finishes those trajectories (lane_loop_group).  Both
    // reasons share one exit, which keeps the loop's scalar registers free.
    if (!leave && run.spill_below && (uint32_t)__popcll(__ballot(1)) <= run.spill_below) {
      spill = true;
      leave = true;
    }
    if (leave) break;

    bool rec = true; // absorbing state: sample without drawing
    double tn = 0.0, u = 0.0;
    bool live = true;
    if (__builtin_expect(!usual, 0)) live = 0.0 < tot;
    if (live) {
      const rebop_u32x4 blk = rebop_stream_block(st, draw);
      draw += 1;
      const double e = rebop_exp1_of_tab(blk, ln_tab);
      double dt = usual_quotient(e, tot);
      if (__builtin_expect(!usual, 0)) dt = e / tot;
      tn = t + dt;
      u = rebop_unif_of(blk);
      rec = tn > T; // overshoot: the draw is discarded
      ov += rec ? 1u : 0u;
    }

    if (rec) {
      if (run.out) {
        net.write_raw(x, orec, n);
        orec += Sn;
      }
      if (__builtin_expect(!net.in_range(x), 0)) acc.flags |= Net::kRangeFlag;
      if (Net::kRangeFlag == REBOP_FLAG_EXACT &&
          __builtin_expect(draw - mark >= REBOP_DRAWS_PER_CHECK, 0))
        acc.flags |= REBOP_FLAG_EXACT; // f64 counts: too many draws between two checks
      if constexpr (Net::kStopFlag != 0u) {
        // (a launch that will be rerun) this lane met the flag: tell the
        // others at once; else look every 8th sample whether another lane
        // did; either way drop the trajectory
        if (!net.may_stop) {
        } else if (acc.flags & Net::kStopFlag) {
          if (!stop) atomicOr(&run.counters[REBOP_CTR_FLAGS], (unsigned long long)Net::kStopFlag);
          stop = true;
        } else if ((i & 7u) == 7u) {
          stop = launch_stopped(run, Net::kStopFlag);
        }
        if (stop) {
          done = true;
          continue;
        }
      }
      mark = draw;
      t = T;
      i += 1;
      if (i > nb) {
        auto &cold = net.cold_run(run);
        if (cold.final_x) net.write_counts(x, cold.final_x + jl, n);
        if (cold.st_x) {
          net.store_state(x, cold.st_x + jl, n);
          cold.st_t[jl] = t;
          cold.st_draw[jl] = draw;
        }
        acc.events += (draw - draw0) - ov;
        acc.draws += draw - draw0;
        acc.trajectories += 1;
        done = true;
      } else {
        T = net.grid_time(run, i);
      }
    } else {
      t = tn;
      net.affect(x, net.choose(x, cum, tot * u));
      tot = props_checked(net, x, cum, acc, usual);
      if constexpr (Net::kCap)
        if (__builtin_expect(draw >= dlim, 0)) {
          tot = hit_cap(run, acc, true);
          usual = false;
        }
    }
  }
  if (spill) {
    auto &cold = net.cold_run(run);
    // one entry per handed-off trajectory, one atomic per wave
    const uint64_t act = __ballot(1);
    const uint32_t lane = __lane_id();
    const int leader = __ffsll((unsigned long long)act) - 1;
    unsigned long long base = 0ull;
    if ((int)lane == leader)
      base = atomicAdd(&cold.counters[REBOP_CTR_SPILL], (unsigned long long)__popcll(act));
    base = __shfl(base, leader);
    const uint64_t e = base + (uint64_t)__popcll(act & ((1ull << lane) - 1ull));
    if (e < cold.spill_cap) {
      cold.spill_j[e] = jl;
      cold.spill_draw[e] = draw;
      cold.spill_mark[e] = mark;
      cold.spill_t[e] = t;
      // bit 31: the trajectory was stopped by the draw cap (its zero total
      // is forced, not recomputed from the counts); grid positions < 2^31
      cold.spill_i[e] = i | ((Net::kCap && tot == 0.0 && draw >= dlim) ? 0x80000000u : 0u);
      net.store_state(x, cold.spill_x + e, cold.spill_cap);
    } else {
      acc.flags |= REBOP_FLAG_INTERNAL; // cannot happen: one entry per lane
    }
    acc.events += (draw - draw0) - ov;
    acc.draws += draw - draw0;
  }
  return acc;
}

// Lane q of each aligned group of K lanes (K = 2, 4 or 16) reads `v` from
// lane Q of its group: one DPP move per 32-bit half (a quad permutation, or a
// broadcast within a row of 16), no LDS traffic.
template <int K, int Q>
__device__ __forceinline__ double group_read(double v) {
  static_assert(K == 2 || K == 4 || K == 16, "groups of 2, 4 or 16 lanes");
  constexpr int ctrl = K == 16  ? 0x150 + Q
                       : K == 4 ? (Q | (Q << 2) | (Q << 4) | (Q << 6))
                                : (Q | (Q << 2) | ((2 + Q) << 4) | ((2 + Q) << 6));
  const uint64_t b = rebop_f64_bits(v);
  const uint32_t lo = (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)b, ctrl, 0xF, 0xF, false);
  const uint32_t hi =
      (uint32_t)__builtin_amdgcn_mov_dpp((int)(uint32_t)(b >> 32), ctrl, 0xF, 0xF, false);
  return rebop_f64_from_bits(((uint64_t)hi << 32) | lo);
}

// The same for a q that is a constant once the caller's loop is unrolled, or
// (groups of 16, whose careful rounds are not) known at run time.
template <int K>
__device__ __forceinline__ double group_read(double v, int q) {
  if constexpr (K == 16) {
    const int at = (int)((__lane_id() & ~15u) + (uint32_t)q) * 4;
    const uint64_t b = rebop_f64_bits(v);
    const uint32_t lo = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)b);
    const uint32_t hi = (uint32_t)__builtin_amdgcn_ds_bpermute(at, (int)(uint32_t)(b >> 32));
    return rebop_f64_from_bits(((uint64_t)hi << 32) | lo);
  } else {
    switch (q) {
    case 0: return group_read<K, 0>(v);
    case 1: return group_read<K, 1>(v);
    case 2: if constexpr (K == 4) return group_read<K, 2>(v); else return v;
    default: if constexpr (K == 4) return group_read<K, 3>(v); else return v;
    }
  }
}

// f(GroupStep<q>{}) for q = 0 .. K - 1
template <int Q>
struct GroupStep {
  static constexpr int q = Q;
};
template <int K, int Q = 0, class F>
__device__ __forceinline__ void group_steps(F &&f) {
  if constexpr (Q < K) {
    f(GroupStep<Q>{});
    group_steps<K, Q + 1>(f);
  }
}

// K lanes per trajectory, for launches with too few trajectories to give
// every SIMD more than one wave (there the time is one trajectory's serial
// event chain, and the Philox block + ln of each draw is most of an event).
// Lane `sub` of a group computes the block of draw (draw + sub) of the group's
// trajectory; the group then runs K iterations of the state machine,
// iteration q using block q (read from lane q by DPP).  That is exactly the
// draw each iteration would take: every event or overshoot consumes the next
// draw, and a trajectory in an absorbing state never draws again (its counts
// no longer change), so the blocks of a round are used in order or not at
// all.  All lanes of a group hold the same state; lane 0 of the group writes
// and counts.  Plain launches only: trajectory j is group j, or with
// run.resume the trajectory of spill entry j (the tail of a persistent
// launch, continued from its written-out state).
//
// A wave alone on its SIMD issues an instruction every five cycles or so, and
// a branch costs it 30 to 60 cycles (compare, mask, skip, restore).  In nine
// iterations of ten some of its sixteen trajectories records a sample while
// the others fire, so both paths were issued and branched over.  Now an
// iteration has one path: a trajectory that records takes no jump (reaction
// MR is none) and keeps its total.  An absorbing state has total 0, whose
// quotient is NaN, which is not at or below any sample time: it records
// without a test of its own.  Draws and overshoots are not counted along the
// way: until it is absorbed, a trajectory takes a draw in every iteration and
// overshoots once per sample.  The range of the counts is checked once a round.
//
// Straight rounds (sample times in LDS, an output below 4 GiB or none, no
// draw cap) have no branch at all.  Samples are stored with buffer instructions whose
// bounds check drops the lanes that have none.  A trajectory past its last
// sample time reads NaN for the next, so it keeps recording, out of bounds,
// until the round's end.  Totals that are not usual ones (an absorbed
// trajectory's above all) are noticed at the end of the round, which is then
// done again with the tests (the stores are the same).  10^4 SIR
// trajectories of 250 samples, a call: 636 us with both paths branched over,
// 557 us with one path and the tests, 490 us in straight rounds (59 vector
// instructions of straight code an iteration with four lanes, 51 with sixteen).
//
// Memory latency stays off the chain: `ln_tab` is the workgroup's LDS copy of
// the ln table, whose rows for the next round's draws are read while this
// round's events run (the next round's blocks are (draw + K + sub), since a
// round either consumes K draws or ends the drawing for good), and
// `grid_lds` its LDS copy of the sample times, followed by REBOP_GRID_PAD
// NaNs, read an iteration ahead.  No vector-memory wait is left
// in the loop, so the sample stores are never waited for.  GridLds: grid_lds
// holds the sample times and group_straight holds for the run (else the next
// sample time is carried, computed at each sample).
template <class Net, int K, bool GridLds>
__device__ __forceinline__ LaneTotals lane_loop_group(Net &net, const rebop_dev_run &run,
                                                      uint64_t gtid, const double (*ln_tab)[4],
                                                      const double *grid_lds) {
  constexpr bool FAST = GridLds && !Net::kCap;
  LaneTotals acc;
  const uint64_t n = run.n_traj;
  const uint64_t e = gtid / K; // group index
  uint64_t jl = e;
  if (run.resume) {
    const uint64_t cnt = __hip_atomic_load(&run.counters[REBOP_CTR_SPILL], __ATOMIC_RELAXED,
                                           __HIP_MEMORY_SCOPE_AGENT);
    if (e >= cnt || e >= run.spill_cap) return acc;
    jl = run.spill_j[e];
  } else if (jl >= n) {
    return acc;
  }
  const uint32_t sub = __lane_id() % K;
  const bool lead = sub == 0;
  const uint32_t nb = run.mode == REBOP_MODE_TARGET ? 0u : (uint32_t)run.nb_steps;
  const uint64_t Sn = (uint64_t)net.S() * n;

  double x[Net::MS];
  double cum[Net::MR];
#pragma unroll
  for (int s = 0; s < Net::MS; ++s) x[s] = 0.0;
#pragma unroll
  for (int r = 0; r < Net::MR; ++r) cum[r] = 0.0;
  net.start(run, jl);
  double t;
  uint64_t draw;
  uint32_t i = 0;
  bool dead = false; // absorbing, stopped by the cap, or finished: tot is 0
  if (run.resume) {
    net.load_state(x, run.spill_x + e, run.spill_cap);
    t = run.spill_t[e];
    draw = run.spill_draw[e];
    i = run.spill_i[e] & 0x7fffffffu;
    dead = (run.spill_i[e] >> 31) != 0u; // by the cap, before the hand-off (already counted)
    if (Net::kRangeFlag == REBOP_FLAG_EXACT && draw - run.spill_mark[e] >= REBOP_DRAWS_PER_CHECK)
      acc.flags |= REBOP_FLAG_EXACT;
  } else if (run.st_x) {
    net.load_state(x, run.st_x + jl, n);
    t = run.st_t[jl];
    draw = run.st_draw[jl];
  } else {
    net.load_x0(x, run.x0_div ? run.x0 + (jl / run.x0_div) * net.S() : run.x0);
    t = 0.0;
    draw = 0;
  }
  // a batch's time may have been set to NaN, which is past no sample time:
  // events until the state is absorbed, as from minus infinity
  if (t != t) t = -__builtin_inf();
  if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
  const uint64_t draw0 = draw;
  const uint32_t i0 = i;
  // the cap counts from the trajectory's draws at the start of this call
  // (a resumed tail entry started it in the persistent launch)
  const uint64_t dlim =
      cap_limit(run, run.resume ? (run.st_x ? run.st_draw[jl] : 0ull) : draw);
  double Tc = GridLds ? 0.0 : grid_time(run, i), tot = 0.0;
  const bool writes = run.out && lead;
  // the draws and the grid position when the trajectory was absorbed
  uint64_t end_draw = draw;
  uint32_t end_i = i;
  // some total of the wave was positive but not a usual one
  bool odd = false;
  auto absorb = [&](uint64_t d) {
    dead = true;
    tot = 0.0;
    end_draw = d;
    end_i = i;
  };
  // a new total that is not a usual one, after d draws
  auto unusual = [&](uint64_t d) {
    if (tot == __builtin_inf()) {
      acc.flags |= REBOP_FLAG_RANGE;
      tot = 0.0;
    }
    if (!(0.0 < tot)) absorb(d);
  };
  if (!dead) {
    tot = net.props(x, cum);
    if (!usual_total(tot)) unusual(draw);
  }
  odd = __ballot(!dead && !usual_total(tot)) != 0ull;
  bool finished = false;
  auto finish = [&](uint64_t d) { // after d draws, if not absorbed before
    if (!dead) absorb(d);
    finished = true;
    if (lead) {
      if (run.final_x) net.write_counts(x, run.final_x + jl, n);
      if (run.st_x) {
        net.store_state(x, run.st_x + jl, n);
        run.st_t[jl] = t;
        run.st_draw[jl] = end_draw;
      }
      acc.events += (end_draw - draw0) - (end_i - i0);
      acc.draws += end_draw - draw0;
      acc.trajectories += 1;
    }
  };
  // the straight rounds' stores: 32-bit byte offsets into run.out, and a lane
  // that writes nothing stores past its end (by a round's samples at most, so
  // below 4 GiB: group_straight), where the buffer's bounds check drops it.
  // Without run.out the buffer is empty and every offset zero.
  const uint32_t row = FAST && run.out ? (uint32_t)Sn * 8u : 0u;
  const uint32_t stride = FAST && run.out ? (uint32_t)n * 8u : 0u, past = (nb + 1u) * row;
  const ByteBuffer out = byte_buffer(run.out, past);

  // this lane's draw of the next round: ln reduced and its table row read,
  // the rest of the ln evaluated when the round starts
  rebop_ln_pre pre;
  double u_next;
  auto fetch = [&](uint64_t d) {
    const rebop_u32x4 blk = rebop_draw_block(run.seed, run.traj_begin + jl, d + sub);
    pre = rebop_ln64_begin(rebop_u01_open_closed(blk.w[0], blk.w[1]), ln_tab);
    u_next = rebop_unif_of(blk);
  };
  fetch(draw);
  while (__ballot(i <= nb) != 0ull) {
    double e_own = -rebop_ln64_finish(pre), u_own = u_next;
    const uint64_t d0 = draw;
    if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
    if (FAST && !odd) {
      double xs[Net::MS], ts = t, tots = tot, T = grid_lds[i], Tn = grid_lds[i + 1u];
#pragma unroll
      for (int s = 0; s < Net::MS; ++s) xs[s] = x[s];
      const uint32_t is = i;
      uint32_t at = lead ? i * row + (run.out ? (uint32_t)jl * 8u : 0u) : past, worst = 0;
      fetch(d0 + K);
      group_steps<K>([&](auto step) {
        constexpr int q = decltype(step)::q;
        const double e = group_read<K, q>(e_own);
        const double u = group_read<K, q>(u_own);
        const double tn = t + usual_quotient(e, tot);
        const bool rec = !(tn <= T);
        const uint32_t k = net.choose(x, cum, tot * u);
        net.affect(x, rec ? (uint32_t)Net::MR : k);
        t = rec ? T : tn;
        const double total = net.props(x, cum);
        tot = rec ? tot : total;
        const uint32_t far = usual_distance(total);
        const uint32_t seen = rec ? 0u : far;
        worst = worst > seen ? worst : seen;
        net.write_raw_buffer(x, out, rec ? at : past, stride);
        at += rec ? row : 0u;
        T = rec ? Tn : T;
        i += rec ? 1u : 0u;
        Tn = grid_lds[i + 1u];
      });
      if (__builtin_expect(__ballot(worst >= kUsualSpan) == 0ull, 1)) {
        const uint32_t extra = i > nb ? i - nb - 1u : 0u; // samples past the last one
        i -= extra;
        const bool last = i > nb && !finished;
        if (__builtin_expect(__ballot(last) != 0ull, 0))
          if (last) {
            t = grid_lds[nb];
            finish(d0 + (K - extra));
          }
        draw = d0 + K;
        continue;
      }
      // an event made a total that is not a usual one: the round again, step
      // by step (what it stored is stored again)
      t = ts;
      tot = tots;
      i = is;
#pragma unroll
      for (int s = 0; s < Net::MS; ++s) x[s] = xs[s];
      (void)net.props(x, cum);
      // (the draws again too: kept, they would cost the straight round registers)
      fetch(d0);
      e_own = -rebop_ln64_finish(pre);
      u_own = u_next;
    }
    int64_t *orec = run.out + jl + (uint64_t)i * Sn;
#pragma unroll(K <= 4 ? K : 1)
    for (int q = 0; q < K; ++q) {
      const double e = group_read<K>(e_own, q);
      const double u = group_read<K>(u_own, q);
      const double T = GridLds ? grid_lds[i] : Tc; // i <= nb + 1
      double dt = usual_quotient(e, tot);
      if (__builtin_expect(odd, 0))
        if (!dead && !usual_total(tot)) dt = e / tot;
      const double tn = t + dt;
      // (a sample time is NaN only with an infinite horizon, which has a cap)
      const bool rec = Net::kCap ? dead || tn > T : !(tn <= T);
      const uint32_t k = net.choose(x, cum, tot * u);
      net.affect(x, rec ? (uint32_t)Net::MR : k);
      t = rec ? T : tn;
      const double total = net.props(x, cum);
      tot = rec ? tot : total;
      const bool strange = !rec && !usual_total(total);
      if (__builtin_expect(__ballot(strange) != 0ull, 0)) {
        if (strange) unusual(d0 + q + 1);
        odd = odd || __ballot(strange && !dead) != 0ull;
      }
      if constexpr (Net::kCap)
        if (__builtin_expect(!rec && !dead && d0 + q + 1 >= dlim, 0)) {
          (void)hit_cap(run, acc, lead);
          absorb(d0 + q + 1);
        }
      const bool sample = rec && i <= nb;
      if (sample && writes) {
        net.write_raw(x, orec, n);
        orec += Sn;
      }
      i += sample ? 1u : 0u;
      if constexpr (!GridLds)
        if (sample) Tc = grid_time(run, i);
      const bool last = sample && i > nb;
      if (__builtin_expect(__ballot(last) != 0ull, 0)) {
        if (last) finish(d0 + q + 1);
      }
      // after the first event's sample-time read, so that waiting for that
      // read does not wait for these
      if (q == 0) fetch(d0 + K);
    }
    draw = d0 + K; // of a trajectory not yet absorbed
  }
  if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
  return acc;
}

// The nb_steps == 0 loop of Gillespie.run (src/pyo3_gillespie.rs:209-223):
// record (t, counts) before the first event and after every
// _advance_one_reaction (src/gillespie.rs:275-297) while t < tmax.  That step
// has no tmax check (the last event lies past tmax) and sets t = +inf in an
// absorbing state.  Without rec_offsets the lane only counts its records
// into n_records; with them it writes row r of trajectory j at
// rec_offsets[j] + r (the stream is deterministic, so both passes agree).
template <class Net>
__device__ __forceinline__ LaneTotals lane_events(Net &net, const rebop_dev_run &run,
                                                  uint64_t first, uint64_t queue_offset,
                                                  const double (*ln_tab)[4] = rebop_ln_table) {
  const uint64_t n = run.n_traj;
  const uint32_t S = net.S();
  double x[Net::MS];
  double cum[Net::MR];
#pragma unroll
  for (int s = 0; s < Net::MS; ++s) x[s] = 0.0;
#pragma unroll
  for (int r = 0; r < Net::MR; ++r) cum[r] = 0.0;
  LaneTotals acc;
  bool started = false;
  for (;;) {
    const uint64_t jl = next_trajectory(run, started, first, queue_offset);
    if (jl >= n) break;
    const rebop_stream st = rebop_stream_of(run.seed, run.traj_begin + jl);
    net.start(run, jl);
    net.load_x0(x, run.x0_div ? run.x0 + (jl / run.x0_div) * S : run.x0);
    if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
    const bool write = run.rec_offsets != nullptr;
    const uint64_t base = write ? run.rec_offsets[jl] : 0ull;
    // the caller's count bounds the writes: a count that does not match this
    // trajectory is reported (below), never written past
    const uint64_t cap = write ? run.n_records[jl] : 0ull;
    double t = 0.0;
    uint64_t draw = 0, rec = 0;
    const uint64_t dlim = cap_limit(run, 0ull);
    bool stop = false; // the draw cap was reached
    auto emit = [&]() {
      if (write && rec < cap) {
        run.rec_times[base + rec] = t;
        net.write_counts(x, run.rec_states + (base + rec) * S, 1);
      }
      rec += 1;
    };
    emit();
    while (t < run.tmax && !stop) {
      const double tot = net.props(x, cum);
      if (!(0.0 < tot)) {
        t = __builtin_inf();
      } else if (tot == __builtin_inf()) {
        acc.flags |= REBOP_FLAG_RANGE; // time would stop (E / tot == 0)
        t = __builtin_inf();
      } else {
        const rebop_u32x4 blk = rebop_stream_block(st, draw);
        draw += 1;
        t = t + rebop_exp1_of_tab(blk, ln_tab) / tot;
        net.affect(x, net.choose(x, cum, tot * rebop_unif_of(blk)));
        if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
        if constexpr (Net::kCap) {
          if (__builtin_expect(draw >= dlim, 0)) {
            hit_cap(run, acc, true);
            stop = true;
          }
        }
      }
      emit();
    }
    if (!write) run.n_records[jl] = rec;
    else if (run.n_records[jl] != rec) acc.flags |= REBOP_FLAG_RANGE;
    acc.events += draw;
    acc.draws += draw;
    acc.trajectories += 1;
  }
  return acc;
}

// lane_events with K lanes per trajectory (K = 2 or 4; plain launches:
// trajectory j is group j), for runs too small to give every SIMD more than
// one wave: lane `sub` of a group computes the Philox block and exponential
// of draw (draw + sub), and the group runs up to K events of the loop above
// using block q for its q-th event (read from lane q by DPP) -- each event
// takes the next draw and an absorbing state takes none, so the blocks of a
// round are used in order or not at all (the argument of lane_loop_group).
// All lanes hold the same state; lane 0 of the group writes and counts.  As
// there, an iteration has one path for every trajectory: an absorbed one
// (total 0, quotient NaN) moves its time to infinity, and one that has ended
// takes no jump and keeps its time.  Straight rounds have no branch: an ended
// trajectory writes its last record again, and a round is done again step by
// step if a total in it was not a usual one.  A wave takes the step-by-step
// round while a trajectory has an absorbed state to report or records for
// less than a round left.  WRITE: run.rec_offsets is set.  10^4 SIR
// trajectories, both passes: 1152 us with branches, 940 us.
template <class Net, int K, bool WRITE>
__device__ __forceinline__ LaneTotals lane_events_group(Net &net, const rebop_dev_run &run, uint64_t gtid,
                                                        const double (*ln_tab)[4]) {
  LaneTotals acc;
  const uint64_t jl = gtid / K;
  if (jl >= run.n_traj) return acc;
  const uint32_t sub = __lane_id() % K;
  const bool lead = sub == 0;
  const uint32_t S = net.S();
  double x[Net::MS];
  double cum[Net::MR];
#pragma unroll
  for (int s = 0; s < Net::MS; ++s) x[s] = 0.0;
#pragma unroll
  for (int r = 0; r < Net::MR; ++r) cum[r] = 0.0;
  net.start(run, jl);
  net.load_x0(x, run.x0_div ? run.x0 + (jl / run.x0_div) * S : run.x0);
  if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
  const uint64_t base = WRITE ? run.rec_offsets[jl] : 0ull;
  // the caller's count bounds the writes (see lane_events)
  uint64_t room = WRITE ? run.n_records[jl] : 0ull; // records still to write
  double *rt = run.rec_times + base;
  int64_t *rs = run.rec_states + base * S;
  const double tmax = run.tmax;
  double t = 0.0, tot = 0.0;
  uint64_t draw = 0, rec = 0;
  const uint64_t dlim = cap_limit(run, 0ull);
  bool dead = false; // absorbed: tot is 0
  bool odd = false;  // some total of the wave was positive but not a usual one
  auto emit = [&]() {
    if (room != 0ull) {
      room -= 1;
      if (lead) {
        *rt = t;
        net.write_counts(x, rs, 1);
      }
      rt += 1;
      rs += S;
    }
  };
  auto unusual = [&]() {
    if (tot == __builtin_inf()) {
      acc.flags |= REBOP_FLAG_RANGE; // time would stop (E / tot == 0)
      tot = 0.0;
    }
    if (!(0.0 < tot)) {
      dead = true;
      tot = 0.0;
    }
  };
  bool more = t < tmax;
  if (more) {
    tot = net.props(x, cum);
    if (!usual_total(tot)) unusual();
  }
  odd = __ballot(more && !dead && !usual_total(tot)) != 0ull;
  emit();
  rec = 1;
  rebop_ln_pre pre;
  double u_next;
  auto fetch = [&](uint64_t d) {
    const rebop_u32x4 blk = rebop_draw_block(run.seed, run.traj_begin + jl, d + sub);
    pre = rebop_ln64_begin(rebop_u01_open_closed(blk.w[0], blk.w[1]), ln_tab);
    u_next = rebop_unif_of(blk);
  };
  fetch(0);
  uint64_t d0 = 0;
  while (__ballot(more) != 0ull) {
    double e_own = -rebop_ln64_finish(pre), u_own = u_next;
    fetch(d0 + K);
    if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
    // an ended trajectory has a record to write again, the first at least
    const bool careful = (more && (dead || (WRITE && room < (uint64_t)K))) ||
                         (WRITE && (!net.small(x) || run.n_records[jl] == 0ull));
    if (!Net::kCap && !odd && __ballot(careful) == 0ull) {
      double xs[Net::MS], ts = t, tots = tot;
#pragma unroll
      for (int s = 0; s < Net::MS; ++s) xs[s] = x[s];
      uint32_t fired = 0, worst = 0;
      double *wt = rt - 1; // the last record written
      int64_t *ws = rs - S;
#pragma unroll
      for (int q = 0; q < K; ++q) {
        const double e = group_read<K>(e_own, q);
        const double u = group_read<K>(u_own, q);
        const double tn = t + usual_quotient(e, tot);
        const uint32_t k = net.choose(x, cum, tot * u);
        const bool on = t < tmax;
        net.affect(x, on ? k : (uint32_t)Net::MR);
        t = on ? tn : t;
        tot = net.props(x, cum);
        const uint32_t step = on ? 1u : 0u, far = usual_distance(tot);
        fired += step;
        const uint32_t seen = t < tmax ? far : 0u;
        worst = worst > seen ? worst : seen;
        if constexpr (WRITE) {
          wt += step;
          ws += step * S;
          *wt = t;
          net.write_small(x, ws);
        }
      }
      if (__builtin_expect(__ballot(worst >= kUsualSpan) == 0ull, 1)) {
        draw += fired;
        rec += fired;
        more = t < tmax;
        if constexpr (WRITE) {
          room -= fired;
          rt = wt + 1;
          rs = ws + S;
        }
        d0 += K;
        continue;
      }
      // the round again, step by step (what it wrote is written again)
      t = ts;
      tot = tots;
#pragma unroll
      for (int s = 0; s < Net::MS; ++s) x[s] = xs[s];
      (void)net.props(x, cum);
      fetch(d0);
      e_own = -rebop_ln64_finish(pre);
      u_own = u_next;
      fetch(d0 + K);
    }
#pragma unroll
    for (int q = 0; q < K; ++q) {
      const double e = group_read<K>(e_own, q);
      const double u = group_read<K>(u_own, q);
      double dt = usual_quotient(e, tot);
      if (__builtin_expect(odd, 0))
        if (!dead && !usual_total(tot)) dt = e / tot;
      // the time of an absorbed trajectory: infinity in place of NaN
      const double tn = __builtin_fmin(t + dt, __builtin_inf());
      const bool fires = more && !dead;
      const uint32_t k = net.choose(x, cum, tot * u);
      net.affect(x, fires ? k : (uint32_t)Net::MR);
      t = more ? tn : t;
      draw += fires ? 1u : 0u;
      const double total = net.props(x, cum);
      tot = fires ? total : tot;
      rec += more ? 1u : 0u;
      const bool was = more;
      more = more && t < tmax;
      if constexpr (Net::kCap)
        if (__builtin_expect(fires && draw >= dlim, 0)) {
          hit_cap(run, acc, lead);
          more = false; // the draw cap was reached
        }
      // (a total that no event will use is not looked at)
      const bool strange = more && fires && !usual_total(total);
      if (__builtin_expect(__ballot(strange) != 0ull, 0)) {
        if (strange) unusual();
        odd = odd || __ballot(strange && !dead) != 0ull;
      }
      if (WRITE)
        if (was) emit();
    }
    d0 += K;
  }
  if (!net.in_range(x)) acc.flags |= Net::kRangeFlag;
  if (lead) {
    if (!WRITE) run.n_records[jl] = rec;
    else if (run.n_records[jl] != rec) acc.flags |= REBOP_FLAG_RANGE;
    acc.events += draw;
    acc.draws += draw;
    acc.trajectories += 1;
  }
  return acc;
}

// Sums lane totals over the workgroup in LDS (blk_ctr zeroed before use).
__device__ __forceinline__ void add_totals(const LaneTotals &acc, unsigned long long *blk_ctr) {
  atomicAdd(&blk_ctr[0], (unsigned long long)acc.events);
  atomicAdd(&blk_ctr[1], (unsigned long long)acc.draws);
  atomicAdd(&blk_ctr[2], (unsigned long long)acc.trajectories);
  if (acc.flags) atomicOr(&blk_ctr[3], (unsigned long long)acc.flags);
}

// After a workgroup barrier: one global update per workgroup.
__device__ __forceinline__ void flush_block_totals(unsigned long long *counters,
                                                   const unsigned long long *blk_ctr) {
  if (threadIdx.x == 0) {
    atomicAdd(&counters[REBOP_CTR_EVENTS], blk_ctr[0]);
    atomicAdd(&counters[REBOP_CTR_DRAWS], blk_ctr[1]);
    atomicAdd(&counters[REBOP_CTR_TRAJ], blk_ctr[2]);
    if (blk_ctr[3]) atomicOr(&counters[REBOP_CTR_FLAGS], blk_ctr[3]);
  }
}

// One global update per wave, reduced across the wave's lanes (no LDS): for
// kernels whose LDS is all spoken for.
__device__ __forceinline__ void flush_wave_totals(const LaneTotals &acc,
                                                  unsigned long long *counters) {
  unsigned long long ev = acc.events, dr = acc.draws, tr = acc.trajectories;
  uint32_t fl = acc.flags;
#pragma unroll
  for (int off = 32; off >= 1; off >>= 1) {
    ev += __shfl_xor(ev, off);
    dr += __shfl_xor(dr, off);
    tr += __shfl_xor(tr, off);
    fl |= __shfl_xor(fl, off);
  }
  if (__lane_id() == 0) {
    atomicAdd(&counters[REBOP_CTR_EVENTS], ev);
    atomicAdd(&counters[REBOP_CTR_DRAWS], dr);
    atomicAdd(&counters[REBOP_CTR_TRAJ], tr);
    if (fl) atomicOr(&counters[REBOP_CTR_FLAGS], (unsigned long long)fl);
  }
}

// The whole-launch epilogue of a single-network kernel.
__device__ __forceinline__ void flush_totals(const LaneTotals &acc, const rebop_dev_run &run,
                                             unsigned long long *blk_ctr) {
  add_totals(acc, blk_ctr);
  __syncthreads();
  flush_block_totals(run.counters, blk_ctr);
}

} // namespace rebop

#endif
