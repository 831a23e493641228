// jit.cpp -- network-specialised SSA kernels, compiled at run time with hipRTC.
//
// For a given network the generated kernel has the rate constants, the
// propensity factor lists and the stoichiometry as compile-time constants:
// Rate::rate's multiplication sequence is unrolled with static species
// indices (no indexed register moves, no scalar loads), choose_cumrate_sum
// is an unrolled compare-and-count, and Jump::affect becomes, per species,
// a select of the integer difference by reaction index.  The lane engine is
// the same ssa_lane.h the ahead-of-time kernels use (its text is embedded in
// the library at build time), so both paths compute the same arithmetic in
// the same order; the device results are bit-identical.
//
// Compiled code objects are cached per (device, generated source).
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <algorithm>
#include <cmath>
#include <unistd.h>
#include <sys/stat.h>
#include <cstring>
#include <cstdlib>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>
#include <utility>
#include <vector>

#include "jit.h"
#include "rebop_expr.h"
#include "ssa_layout.h"

namespace rebop {

// text of rebop_rng.h, ssa_layout.h and ssa_lane.h (generated by build.py)
extern const int kEmbeddedHeaderCount;
extern const char *const kEmbeddedHeaderNames[];
extern const char *const kEmbeddedHeaderSources[];

static std::string f64_literal(double v) {
  if (std::isnan(v)) return "__builtin_nan(\"\")";
  char buf[64];
  std::snprintf(buf, sizeof buf, "%a", v);
  return std::string("(") + buf + ")";
}

// Straight-line code for a postfix expression: one temporary per token.
// Returns the name of the temporary holding the value.
static std::string expr_code(const JitReaction &r, uint32_t rid, std::string *s) {
  std::vector<std::string> st;
  uint32_t n = 0;
  for (uint32_t tok : r.expr) {
    const uint32_t op = REBOP_EXPR_OPCODE(tok), arg = REBOP_EXPR_ARG(tok);
    const std::string t = "e" + std::to_string(rid) + "_" + std::to_string(n++);
    std::string v;
    if (op == REBOP_OP_CONST) {
      v = f64_literal(r.consts[arg]);
    } else if (op == REBOP_OP_SPECIES) {
      v = "x[" + std::to_string(arg) + "]";
    } else if (op == REBOP_OP_NEG || op == REBOP_OP_EXP) {
      const std::string a = st.back();
      st.pop_back();
      v = op == REBOP_OP_NEG ? "-" + a : "rebop_exp64(" + a + ")";
    } else {
      const std::string b = st.back();
      st.pop_back();
      const std::string a = st.back();
      st.pop_back();
      switch (op) {
      case REBOP_OP_ADD: v = a + " + " + b; break;
      case REBOP_OP_SUB: v = a + " - " + b; break;
      case REBOP_OP_MUL: v = a + " * " + b; break;
      case REBOP_OP_DIV: v = a + " / " + b; break;
      case REBOP_OP_POW: v = "rebop_pow64(" + a + ", " + b + ")"; break;
      case REBOP_OP_MAX: v = "rebop_fmax64(" + a + ", " + b + ")"; break;
      default: v = "rebop_fmin64(" + a + ", " + b + ")"; break;
      }
    }
    *s += "    const double " + t + " = " + v + ";\n";
    st.push_back(t);
  }
  return st.back();
}

std::string jit_source(uint32_t S, const std::vector<JitReaction> &rx, bool system, bool cap) {
  const uint32_t R = (uint32_t)rx.size();
  const uint32_t MS = S ? S : 1, MR = R ? R : 1;
  std::string s;
  s.reserve(4096 + 256 * R);
  s += "#include \"ssa_lane.h\"\n#include \"rebop_expr.h\"\n";
  s += "#pragma clang fp contract(off)\n";
  const std::string Ss = std::to_string(S) + "u";
  const std::string MSs = std::to_string(MS);
  s += "template <bool SWEEP, bool GRID_LDS = false>\nstruct JitNet {\n";
  s += "  static constexpr int MS = " + MSs + ";\n";
  s += std::string("  static constexpr bool kCap = ") + (cap ? "true" : "false") + ";\n";
  s += "  static constexpr uint32_t kRangeFlag = REBOP_FLAG_EXACT;\n";
  s += "  static constexpr uint32_t kStopFlag = 0u;\n";
  s += "  static constexpr int MR = " + std::to_string(MR) + ";\n";
  s += "  using X = double[MS];\n  using C = double[MR];\n";
  s += "  double kr[MR];\n";
  s += "  const double *gl = nullptr; // GRID_LDS: the workgroup's LDS copy of the sample times\n";
  // the launch's parameters read again from the kernel's argument block: held
  // in scalar registers throughout, the pointers that only a trajectory's start
  // and end need push the Philox round keys out into vector-register lanes
  // (nine v_readlane an event for the dimer network)
  s += "  using Cold = const __attribute__((address_space(4))) rebop_dev_run;\n";
  s += "  __device__ __forceinline__ Cold &cold_run(const rebop_dev_run &) const {\n";
  s += "    Cold *p = (Cold *)__builtin_amdgcn_kernarg_segment_ptr();\n";
  s += "    asm volatile(\"\" : \"+s\"(p));\n    return *p;\n  }\n";
  s += "  __device__ __forceinline__ void start(const rebop_dev_run &run, uint64_t j) {\n";
  s += "    if (SWEEP) { const double *src = run.rates + (j / run.rates_div) * " + std::to_string(R) + "u;\n";
  s += "      for (int r = 0; r < MR; ++r) kr[r] = r < " + std::to_string(R) + " ? src[r] : 0.0; }\n";
  s += "  }\n";
  s += "  __device__ __forceinline__ uint32_t S() const { return " + Ss + "; }\n";
  s += "  __device__ __forceinline__ double grid_time(const rebop_dev_run &run, uint64_t i) const {\n";
  s += "    if constexpr (GRID_LDS) return gl[i]; else return rebop::table_time(run, i);\n  }\n";
  s += "  __device__ __forceinline__ void load_x0(X &x, const int64_t *src) const { rebop::reg_load_x0(x, src, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void load_state(X &x, const double *st, uint64_t stride) const { rebop::reg_load_state(x, st, stride, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void store_state(const X &x, double *st, uint64_t stride) const { rebop::reg_store_state(x, st, stride, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void write_counts(const X &x, int64_t *dst, uint64_t stride) const { rebop::reg_write_counts(x, dst, stride, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void write_raw(const X &x, int64_t *dst, uint64_t stride) const { rebop::reg_write_raw(x, dst, stride, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void write_raw_buffer(const X &x, rebop::ByteBuffer b, uint32_t at, uint32_t stride) const { rebop::reg_write_raw_buffer(x, b, at, stride, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ bool small(const X &x) const { return rebop::reg_small(x, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ void write_small(const X &x, int64_t *dst) const { rebop::reg_write_small(x, dst, " + Ss + "); }\n";
  s += "  __device__ __forceinline__ bool in_range(const X &x) const { return rebop::reg_in_range(x, " + Ss + "); }\n";
  // make_cumrates over Rate::rate
  s += "  __device__ __forceinline__ double props(X &x, C &cum) const {\n";
  s += "    double acc = 0.0;\n    double a;\n";
  for (uint32_t r = 0; r < R; ++r) {
    if (!rx[r].expr.empty()) {
      // Rate::Expr (expr.rs:24-38): the expression's value is the propensity
      s += "    {\n";
      const std::string v = expr_code(rx[r], r, &s);
      s += "    a = " + v + ";\n    }\n";
      s += "    acc = acc + a;\n    cum[" + std::to_string(r) + "] = acc;\n";
      continue;
    }
    s += "    a = SWEEP ? kr[" + std::to_string(r) + "] : " + f64_literal(rx[r].k) + ";\n";
    if (system) {
      // define_system (gillespie_macro.rs:108, _rate_lma! :128-142): per
      // reactant term, x (x-1) ... (x-m+1) as a wrapping 64-bit integer
      // product converted to f64 once; m <= 1 is the count itself
      for (auto &tm : rx[r].terms) {
        const std::string xs = "x[" + std::to_string(tm.first) + "]";
        if (tm.second <= 1u) {
          s += "    a = a * " + xs + ";\n";
          continue;
        }
        s += "    { const int64_t v = (int64_t)" + xs + "; uint64_t p = (uint64_t)v;";
        for (uint32_t i = 1; i < tm.second; ++i)
          s += " p = p * (uint64_t)(v - " + std::to_string(i) + ");";
        s += " a = a * (double)(int64_t)p; }\n";
      }
      s += "    acc = acc + a;\n    cum[" + std::to_string(r) + "] = acc;\n";
      continue;
    }
    for (auto &f : rx[r].factors) {
      const std::string xs = "x[" + std::to_string(f.first) + "]";
      if (f.second == 0)
        s += "    a = a * " + xs + ";\n";
      else
        s += "    a = a * (" + xs + " - " + std::to_string(f.second) + ".0);\n";
    }
    s += "    acc = acc + a;\n    cum[" + std::to_string(r) + "] = acc;\n";
  }
  s += "    return acc;\n  }\n";
  // choose_cumrate_sum
  s += "  __device__ __forceinline__ uint32_t choose(X &, C &cum, double chosen) const {\n";
  if (system) {
    // _choice! (gillespie_macro.rs:146-170): the first r with chosen < cum_r,
    // R (no reaction) when there is none
    s += "    uint32_t k = " + std::to_string(R) + "u;\n";
    for (uint32_t r = R; r-- > 0;)
      s += "    k = (chosen < cum[" + std::to_string(r) + "]) ? " + std::to_string(r) + "u : k;\n";
  } else {
    // the last sum is the total, which chosen = tot * U never exceeds
    s += "    uint32_t k = 0u;\n";
    for (uint32_t r = 0; r + 1u < R; ++r)
      s += "    k += (cum[" + std::to_string(r) + "] < chosen) ? 1u : 0u;\n";
  }
  s += "    return k;\n  }\n";
  // Jump::affect: per species, the integer difference selected by reaction
  s += "  __device__ __forceinline__ void affect(X &x, uint32_t k) const {\n";
  for (uint32_t sp = 0; sp < S; ++sp) {
    std::vector<std::pair<uint32_t, int64_t>> nz;
    for (uint32_t r = 0; r < R; ++r)
      if (rx[r].diff[sp] != 0) nz.emplace_back(r, rx[r].diff[sp]);
    if (nz.empty()) continue;
    const std::string xs = "x[" + std::to_string(sp) + "]";
    // The differences of every reaction (and of none, define_system's k = R)
    // as fields of one word, read by a shift and a field extract, where they
    // fit 32 bits: fewer instructions than a select per reaction once two
    // reactions change the species (10 of 27 fewer per event for the dimer
    // network's choice and jump).
    uint32_t w = 2;
    int64_t lo = 0, hi = 0;
    for (auto &e : nz) {
      lo = std::min(lo, e.second);
      hi = std::max(hi, e.second);
    }
    while (w <= 16u && (lo < -(1ll << (w - 1u)) || hi >= (1ll << (w - 1u)))) w *= 2u;
    if (nz.size() >= 2 && w <= 16u && w * (R + 1u) <= 32u) {
      uint32_t word = 0;
      for (auto &e : nz) word |= ((uint32_t)e.second & ((1u << w) - 1u)) << (w * e.first);
      s += "    " + xs + " = " + xs + " + (double)(int)__builtin_amdgcn_sbfe((int)" + std::to_string(word) +
           "u, k * " + std::to_string(w) + "u, " + std::to_string(w) + "u);\n";
      continue;
    }
    s += "    { int d = 0;";
    for (auto &e : nz)
      s += " d = (k == " + std::to_string(e.first) + "u) ? (" + std::to_string(e.second) + ") : d;";
    s += " " + xs + " = " + xs + " + (double)d; }\n";
  }
  s += "    (void)k; (void)x;\n  }\n";
  s += "};\n";
  // The ln table and (plain grid runs with nb_steps < REBOP_GRID_LDS) the
  // sample times are read from LDS copies, so that no event waits on vector
  // memory (such a wait also waits for the lane's earlier sample stores).
  s += "struct JitLds { unsigned long long ctr[4]; double ln[128][4]; };\n";
  s += "__device__ __forceinline__ void jit_begin(JitLds &l) {\n";
  s += "  if (threadIdx.x < 4) l.ctr[threadIdx.x] = 0ull;\n";
  s += "  for (uint32_t w = threadIdx.x; w < 512u; w += blockDim.x)\n";
  s += "    (&l.ln[0][0])[w] = (&rebop_ln_table[0][0])[w];\n}\n";
  s += "template <bool SWEEP>\n__device__ __forceinline__ void jit_body(const rebop_dev_run &run) {\n";
  s += "  __shared__ JitLds l;\n";
  s += "  extern __shared__ double grid_lds[];\n";
  s += "  jit_begin(l);\n";
  s += "  const bool lds_grid = !SWEEP && run.mode == REBOP_MODE_GRID && run.grid && run.nb_steps < REBOP_GRID_LDS;\n";
  s += "  if (lds_grid)\n";
  s += "    for (uint32_t w = threadIdx.x; w <= (uint32_t)run.nb_steps; w += blockDim.x) grid_lds[w] = run.grid[w];\n";
  s += "  __syncthreads();\n";
  s += "  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;\n";
  s += "  const uint64_t nthreads = (uint64_t)gridDim.x * blockDim.x;\n";
  s += "  rebop::LaneTotals acc;\n";
  s += "  if (lds_grid) {\n";
  s += "    JitNet<SWEEP, true> net;\n";
  s += "    net.gl = grid_lds;\n";
  s += "    acc = rebop::lane_loop(net, run, gtid, nthreads, l.ln);\n";
  s += "  } else {\n";
  s += "    JitNet<SWEEP> net;\n";
  s += "    acc = !SWEEP && run.mode == REBOP_MODE_EVENTS ? rebop::lane_events(net, run, gtid, nthreads, l.ln)\n";
  s += "                                                  : rebop::lane_loop(net, run, gtid, nthreads, l.ln);\n";
  s += "  }\n";
  s += "  rebop::flush_totals(acc, run, l.ctr);\n";
  s += "}\n";
  // every event recorded, K lanes per trajectory
  s += "template <int K, bool WRITE>\n__device__ __forceinline__ void jit_body_events(const rebop_dev_run &run) {\n";
  s += "  __shared__ JitLds l;\n";
  s += "  jit_begin(l);\n";
  s += "  __syncthreads();\n";
  s += "  JitNet<false> net;\n";
  s += "  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;\n";
  s += "  rebop::LaneTotals acc = rebop::lane_events_group<JitNet<false>, K, WRITE>(net, run, gtid, l.ln);\n";
  s += "  rebop::flush_totals(acc, run, l.ctr);\n";
  s += "}\n";
  // grouped kernels: the ln table and (GRID_LDS, a run with group_straight) the
  // sample times copied into LDS, so that the serial loop never waits on
  // vector memory (the launch sizes the dynamic LDS for the sample times)
  s += "template <int K, bool GRID_LDS>\n__device__ __forceinline__ void jit_body_group(const rebop_dev_run &run) {\n";
  s += "  __shared__ JitLds l;\n";
  s += "  extern __shared__ double grid_lds[];\n";
  s += "  jit_begin(l);\n";
  s += "  if constexpr (GRID_LDS) {\n";
  s += "    const uint64_t samples = rebop::run_samples(run);\n";
  s += "    for (uint32_t w = threadIdx.x; w < samples; w += blockDim.x) grid_lds[w] = run.grid[w];\n";
  s += "    if (threadIdx.x < REBOP_GRID_PAD) grid_lds[samples + threadIdx.x] = __builtin_nan(\"\");\n";
  s += "  }\n";
  s += "  __syncthreads();\n";
  s += "  JitNet<false> net;\n";
  s += "  const uint64_t gtid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;\n";
  s += "  rebop::LaneTotals acc = rebop::lane_loop_group<JitNet<false>, K, GRID_LDS>(net, run, gtid, l.ln, grid_lds);\n";
  s += "  rebop::flush_totals(acc, run, l.ctr);\n";
  s += "}\n";
  return s;
}

const char *jit_variant_name(int v) {
  static const char *const names[kJitVariants] = {"main", "g2", "g4", "g16", "g2_far", "g4_far", "sweep",
                                                  "ev2_count", "ev2_write", "ev4_count", "ev4_write"};
  return names[v];
}

uint32_t jit_prepare_set(uint32_t R, bool cap) {
  return jit_bit(kJitMain) | jit_bit(kJitG2) | jit_bit(kJitG4) | jit_bit(kJitG2Far) | jit_bit(kJitG4Far) |
         (jit_sixteen(R, cap) ? jit_bit(kJitG16) : 0u);
}

// The entry points of the variants in `mask`, after jit_source's text.
static std::string jit_kernels(uint32_t mask) {
  static const char *const body[kJitVariants] = {
      "jit_body<false>",           "jit_body_group<2, true>",   "jit_body_group<4, true>",
      "jit_body_group<16, true>",  "jit_body_group<2, false>",  "jit_body_group<4, false>",
      "jit_body<true>",            "jit_body_events<2, false>", "jit_body_events<2, true>",
      "jit_body_events<4, false>", "jit_body_events<4, true>"};
  // REBOP_JIT_WAVES_PER_EU=<n>: ask the compiler to fit n waves per SIMD in
  // the main kernel's registers (a tuning knob; unset: the compiler's choice)
  std::string occ;
  if (const char *v = std::getenv("REBOP_JIT_WAVES_PER_EU")) {
    const long n = std::strtol(v, nullptr, 10);
    if (n >= 1 && n <= 8) occ = " __attribute__((amdgpu_waves_per_eu(" + std::to_string(n) + ")))";
  }
  std::string s;
  for (int v = 0; v < kJitVariants; ++v)
    if (mask & jit_bit(v))
      s += "extern \"C\" __global__ void __launch_bounds__(256)" + (v == kJitMain ? occ : std::string()) +
           " rebop_ssa_jit_" + jit_variant_name(v) + "(rebop_dev_run run) { " + body[v] + "(run); }\n";
  return s;
}

namespace {
// hipRTC options of every specialised kernel (fp contraction off: the SSA's
// arithmetic must round as separate multiplies and adds)
const char *const kCompileOptions[] = {"--offload-arch=gfx950", "-O3", "-std=c++17",
                                       "-ffp-contract=off", "-fno-fast-math", "-Xclang",
                                       "-target-feature", "-Xclang", "-packed-fp32-ops"};
constexpr int kNumCompileOptions = (int)(sizeof kCompileOptions / sizeof kCompileOptions[0]);

std::mutex g_jit_mu;
std::map<std::pair<int, std::string>, JitKernel> g_jit_cache;

// On-disk cache of compiled code objects, so that a new process does not pay
// the run-time compilation again: <dir>/<hash>.co with the generated source
// beside it in <dir>/<hash>.src (checked on load, so a hash collision only
// costs a compile).  REBOP_JIT_CACHE names the directory (empty: no disk
// cache); default $XDG_CACHE_HOME/rebop_amd/jit or ~/.cache/rebop_amd/jit.
std::string jit_cache_dir() {
  if (const char *v = std::getenv("REBOP_JIT_CACHE")) return v;
  if (const char *x = std::getenv("XDG_CACHE_HOME"); x && *x) return std::string(x) + "/rebop_amd/jit";
  if (const char *h = std::getenv("HOME"); h && *h) return std::string(h) + "/.cache/rebop_amd/jit";
  return "";
}

uint64_t fnv1a(const std::string &s) {
  uint64_t h = 1469598103934665603ull;
  for (unsigned char c : s) {
    h ^= c;
    h *= 1099511628211ull;
  }
  return h;
}

bool read_file(const std::string &path, std::vector<char> *out) {
  FILE *f = std::fopen(path.c_str(), "rb");
  if (!f) return false;
  std::fseek(f, 0, SEEK_END);
  const long n = std::ftell(f);
  std::fseek(f, 0, SEEK_SET);
  out->resize(n > 0 ? (size_t)n : 0);
  const bool ok = n > 0 && std::fread(out->data(), 1, (size_t)n, f) == (size_t)n;
  std::fclose(f);
  return ok;
}

// writes via a temporary file and a rename, so readers never see a partial file
void write_file(const std::string &path, const char *data, size_t n) {
  const std::string tmp = path + ".tmp" + std::to_string((unsigned long long)getpid());
  FILE *f = std::fopen(tmp.c_str(), "wb");
  if (!f) return;
  const bool ok = std::fwrite(data, 1, n, f) == n;
  std::fclose(f);
  if (ok)
    (void)std::rename(tmp.c_str(), path.c_str());
  else
    (void)std::remove(tmp.c_str());
}

void make_dirs(const std::string &dir) {
  for (size_t i = 1; i <= dir.size(); ++i)
    if (i == dir.size() || dir[i] == '/') (void)mkdir(dir.substr(0, i).c_str(), 0755);
}

// What a code object depends on besides the generated source: the embedded
// headers' text, the compile options and the compiler's version.
const std::string &build_fingerprint() {
  static const std::string fp = [] {
    std::string all;
    for (int i = 0; i < kEmbeddedHeaderCount; ++i) all += kEmbeddedHeaderSources[i];
    for (const char *o : kCompileOptions) all += o;
    int major = 0, minor = 0;
    hiprtcVersion(&major, &minor);
    char buf[96];
    std::snprintf(buf, sizeof buf, "hiprtc %d.%d headers+options %016llx", major, minor,
                  (unsigned long long)fnv1a(all));
    return std::string(buf);
  }();
  return fp;
}

// The cached code object of `src`, if the disk cache holds it.
bool disk_cache_get(const std::string &src_only, std::vector<char> *code) {
  const std::string dir = jit_cache_dir();
  if (dir.empty()) return false;
  const std::string src = build_fingerprint() + "\n" + src_only;
  char name[32];
  std::snprintf(name, sizeof name, "%016llx", (unsigned long long)fnv1a(src));
  std::vector<char> stored;
  if (!read_file(dir + "/" + name + ".src", &stored)) return false;
  if (stored.size() != src.size() || std::memcmp(stored.data(), src.data(), src.size()) != 0)
    return false;
  return read_file(dir + "/" + name + ".co", code);
}

void disk_cache_put(const std::string &src_only, const std::vector<char> &code) {
  const std::string dir = jit_cache_dir();
  if (dir.empty()) return;
  const std::string src = build_fingerprint() + "\n" + src_only;
  make_dirs(dir);
  char name[32];
  std::snprintf(name, sizeof name, "%016llx", (unsigned long long)fnv1a(src));
  write_file(dir + "/" + name + ".co", code.data(), code.size());
  write_file(dir + "/" + name + ".src", src.data(), src.size());
}
} // namespace

// Compiles `src` for gfx950 into a code object (hipRTC).
static int compile(const std::string &src, std::vector<char> *code, std::string *err) {
  hiprtcProgram prog;
  hiprtcResult rr = hiprtcCreateProgram(&prog, src.c_str(), "rebop_ssa_jit.hip", kEmbeddedHeaderCount,
                                        kEmbeddedHeaderSources, kEmbeddedHeaderNames);
  if (rr != HIPRTC_SUCCESS) {
    *err = std::string("hiprtcCreateProgram: ") + hiprtcGetErrorString(rr);
    return -1;
  }
  rr = hiprtcCompileProgram(prog, kNumCompileOptions, const_cast<const char **>(kCompileOptions));
  if (rr != HIPRTC_SUCCESS) {
    size_t ls = 0;
    hiprtcGetProgramLogSize(prog, &ls);
    std::string log(ls, '\0');
    if (ls) hiprtcGetProgramLog(prog, &log[0]);
    hiprtcDestroyProgram(&prog);
    *err = std::string("hiprtcCompileProgram: ") + hiprtcGetErrorString(rr) + "\n" + log;
    return -1;
  }
  size_t cs = 0;
  hiprtcGetCodeSize(prog, &cs);
  code->resize(cs);
  hiprtcGetCode(prog, code->data());
  hiprtcDestroyProgram(&prog);
  return 0;
}

// The code object of `src` from the disk cache, or compiled.
static int code_object(const std::string &src, std::vector<char> *code, std::string *err) {
  // REBOP_DUMP_SPECIALIZED=<file>: write the generated kernel source there
  if (const char *path = std::getenv("REBOP_DUMP_SPECIALIZED")) write_file(path, src.data(), src.size());
  if (disk_cache_get(src, code)) return 0;
  if (int rc = compile(src, code, err)) return rc;
  disk_cache_put(src, *code);
  return 0;
}

// Loads the variants of `mask` that `out` does not hold for the network
// `base`: from one module, compiled (or found in a cache) for the current
// device.  `all`: the variants that are prepared together, whose module the
// disk cache may hold.
int jit_get(const std::string &base, uint32_t mask, uint32_t all, JitKernel *out, std::string *err) {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess) {
    *err = "hipGetDevice failed";
    return -1;
  }
  std::lock_guard<std::mutex> lock(g_jit_mu);
  JitKernel &k = g_jit_cache[std::make_pair(dev, base)];
  uint32_t missing = mask & ~k.have();
  if (missing) {
    std::vector<char> code;
    if (missing != all && (missing & ~all) == 0u && disk_cache_get(base + jit_kernels(all), &code))
      missing = all & ~k.have();
    else if (int rc = code_object(base + jit_kernels(missing), &code, err))
      return rc;
    hipModule_t mod = nullptr; // loaded until the process ends, as its functions may be in use
    hipError_t he = hipModuleLoadData(&mod, code.data());
    if (he != hipSuccess) {
      *err = std::string("hipModuleLoadData: ") + hipGetErrorString(he);
      return -1;
    }
    hipFunction_t fn[kJitVariants] = {};
    for (int v = 0; v < kJitVariants && he == hipSuccess; ++v)
      if (missing & jit_bit(v))
        he = hipModuleGetFunction(&fn[v], mod, (std::string("rebop_ssa_jit_") + jit_variant_name(v)).c_str());
    if (he != hipSuccess) {
      *err = std::string("hipModuleGetFunction: ") + hipGetErrorString(he);
      return -1;
    }
    for (int v = 0; v < kJitVariants; ++v)
      if (fn[v]) k.fn[v] = fn[v];
  }
  *out = k;
  return 0;
}

// Compiles the variants of `mask` for gfx950 without loading them (usable
// without a device).
int jit_compile_only(const std::string &base, uint32_t mask, std::string *err) {
  const std::string src = base + jit_kernels(mask);
  if (const char *path = std::getenv("REBOP_DUMP_SPECIALIZED")) write_file(path, src.data(), src.size());
  std::vector<char> code;
  return compile(src, &code, err);
}

size_t jit_dynamic_lds(const rebop_dev_run &run) {
  // the LDS copy of the sample times (jit_body, jit_body_group; a grid run
  // always has its table)
  if (run.rates || run.mode == REBOP_MODE_EVENTS) return 0u;
  const uint64_t samples = run_samples(run);
  return samples <= REBOP_GRID_LDS ? sizeof(double) * (size_t)(samples + REBOP_GRID_PAD) : 0u;
}

hipError_t jit_occupancy(const JitKernel &k, int variant, int threads, size_t lds, int *blocks_per_cu) {
  return hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, k.fn[variant], threads, lds);
}

hipError_t jit_launch(const JitKernel &k, int variant, const rebop_dev_run &run, int blocks, int threads,
                      hipStream_t stream) {
  rebop_dev_run arg = run;
  void *params[] = {&arg};
  return hipModuleLaunchKernel(k.fn[variant], (unsigned)blocks, 1, 1, (unsigned)threads, 1, 1,
                               (unsigned)jit_dynamic_lds(run), stream, params, nullptr);
}

} // namespace rebop
