// jit.h -- the network-specialised kernels (jit.cpp): the per-reaction
// description the source generator takes, the loaded kernel handles, and the
// compile / occupancy / launch entry points used by the C ABI.
#ifndef REBOP_JIT_H
#define REBOP_JIT_H

#include <hip/hip_runtime.h>

#include <cstdint>
#include <string>
#include <utility>
#include <vector>

#include "ssa_layout.h"

namespace rebop {

struct JitReaction {
  double k;
  std::vector<std::pair<uint32_t, uint32_t>> factors; // (species, c): factor = x[s] - c
  std::vector<int64_t> diff;                          // dense [S]
  // Rate::Expr: postfix tokens (rebop_expr.h) and their constants; empty for LMA
  std::vector<uint32_t> expr;
  std::vector<double> consts;
  // define_system reaction: reactant terms (species, multiplicity) in written order
  std::vector<std::pair<uint32_t, uint32_t>> terms;
};

// The kernels of a network, each compiled when it is first launched or
// prepared: a run uses one or two of them, and compiling all of them for the
// first call made it wait 1.36 s (SIR) to 7.8 s (32 species, 64 reactions);
// the one it launches takes 0.40 s to 0.99 s.  (Each compilation also parses
// the headers, 0.35 s, so those prepared together are compiled together.)
enum JitVariant {
  kJitMain,     // one lane per trajectory
  kJitG2,       // 2 lanes per trajectory (plain launches), runs with group_straight
  kJitG4,       // 4 lanes per trajectory, also the tail of a persistent launch
  kJitG16,      // 16 lanes per trajectory (jit_sixteen)
  kJitG2Far,    // 2 and 4 lanes, runs without group_straight
  kJitG4Far,
  kJitSweep,    // one lane per trajectory, rate tables
  kJitEv2Count, // every event recorded with 2 lanes: counting the records, then writing them
  kJitEv2Write,
  kJitEv4Count, // the same with 4 lanes
  kJitEv4Write,
  kJitVariants
};
constexpr uint32_t jit_bit(int variant) { return 1u << variant; }
const char *jit_variant_name(int variant);

struct JitKernel {
  hipFunction_t fn[kJitVariants] = {};
  uint32_t have() const {
    uint32_t m = 0;
    for (int v = 0; v < kJitVariants; ++v) m |= fn[v] ? jit_bit(v) : 0u;
    return m;
  }
};

// Whether a network of R reactions has the kernel with 16 lanes, whose round
// of sixteen events is straight code.  The larger the network, the less of an
// event its draw is, and the longer the code: 12 species and 24 reactions, one
// trajectory 158 us with four lanes and 128 us with sixteen, 4096 178 and
// 153 us; 20 and 40 308 and 298 us, 371 and 360 us; 32 and 64 672 and 664 us,
// 746 and 769 us, with 6.6 s of compilation against 2.
inline bool jit_sixteen(uint32_t R, bool cap) { return R <= 32u && !cap; }
// The variants of a grid or target run of any size, which are prepared together.
uint32_t jit_prepare_set(uint32_t R, bool cap);

// Kernel source for a network of S species and the given reactions, without
// the entry points; with `system`, the define_system arithmetic (integer
// mass-action products over `terms`, first-match choice); with `cap`, the
// loops check the draw cap.
std::string jit_source(uint32_t S, const std::vector<JitReaction> &rx, bool system = false,
                       bool cap = false);
// Compiles (or finds in a cache) and loads variants on the current device.
int jit_get(const std::string &base, uint32_t mask, uint32_t all, JitKernel *out, std::string *err);
// Compiles for gfx950 without loading (no device needed).
int jit_compile_only(const std::string &base, uint32_t mask, std::string *err);
// Dynamic LDS bytes a launch of `run` takes (the LDS copy of the sample times).
size_t jit_dynamic_lds(const rebop_dev_run &run);
hipError_t jit_occupancy(const JitKernel &k, int variant, int threads, size_t lds, int *blocks_per_cu);
hipError_t jit_launch(const JitKernel &k, int variant, const rebop_dev_run &run, int blocks, int threads,
                      hipStream_t stream);

} // namespace rebop

#endif // REBOP_JIT_H
