// Host runtime of libsimplediffeq_hip: the C ABI declared in
// include/simplediffeq_hip.h.
//
// One sdeh_solve() is the whole ensemble loop that SciMLBase's EnsembleThreads
// would run over DiffEqBase.solve(prob_i, alg; kwargs...) (the six GPUSimple*
// methods of src/tsit5/gpuatsit5.jl and src/verner/gpuvern{7,9}.jl): it
// validates the request, stages host buffers through device memory when asked,
// builds the fixed-step grid with Julia's range rules, picks the integrator
// kernel (compiled ahead of time for the built-in right-hand sides, or by
// hipRTC for a registered RHS source), picks the launch shape (tuned or
// default), arms the persistent queue, launches, and gathers counters.
#include <hip/hip_runtime.h>
#include <hip/hiprtc.h>

#include <algorithm>
#include <cctype>
#include <chrono>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <map>
#include <set>
#include <string>
#include <tuple>
#include <vector>

#include "../../include/simplediffeq_hip.h"
#include "sdeh_kargs.h"
#include "sdeh_range.h"

#define SDEH_HIDDEN __attribute__((visibility("hidden")))

extern "C" {
SDEH_HIDDEN const void* sdeh_aot_Lorenz(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_GLV16(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_GLV16G(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_GLV16M(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_ExpDecay3(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_Affine1(int, int, int, int, int, int);
SDEH_HIDDEN const void* sdeh_aot_Linear2(int, int, int, int, int, int);
SDEH_HIDDEN hipError_t sdeh_util_fill_f64(double*, double, int64_t, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_transpose(const void*, void*, int64_t, int64_t, int, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_fill_f32(float*, float, int64_t, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_zero_u64(unsigned long long*, int, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_count(const int32_t*, const int32_t*, const int32_t*, int64_t,
                                       unsigned long long*, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_check_order(const int64_t*, int64_t, int32_t*, unsigned long long*,
                                             hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_span_order(const double*, int64_t, unsigned*, int64_t*,
                                            hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_resume_order(const double*, int64_t, unsigned*, int64_t*,
                                              unsigned long long*, hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_logkey_order(const float*, int64_t, unsigned*, int64_t*,
                                              hipStream_t);
SDEH_HIDDEN size_t sdeh_util_span_scratch_bytes();
SDEH_HIDDEN hipError_t sdeh_util_static_scratch(void**, size_t*);
SDEH_HIDDEN int sdeh_util_static_saveat_max();
SDEH_HIDDEN hipError_t sdeh_util_pack_offsets(const int32_t*, int32_t, int64_t, int64_t*, int64_t,
                                              int64_t*, int32_t*, unsigned long long*,
                                              hipStream_t);
SDEH_HIDDEN hipError_t sdeh_util_count_order(const int32_t*, const int32_t*, int64_t, unsigned*,
                                             int64_t*, hipStream_t);
SDEH_HIDDEN int sdeh_mlp_forward_impl(const float*, const float*, float*, int64_t, hipStream_t);
SDEH_HIDDEN int sdeh_mlp_plan_lorenz_impl(const float*, const double*, const double*,
                                          const double*, int64_t, const double*, float, float,
                                          float, float, float*, double*, float*, hipStream_t);
SDEH_HIDDEN int sdeh_mlp_loss_grad_impl(const float*, const float*, const float*, int64_t, float*,
                                        float*, float*, hipStream_t);
SDEH_HIDDEN size_t sdeh_mlp_grad_scratch_bytes(int64_t);
SDEH_HIDDEN int sdeh_mlp_adam_impl(float*, const float*, float*, float*, float, float, float, float,
                                   int32_t, hipStream_t);
}

#include "sdeh_embedded.inc"  // sdeh_embedded_names / sdeh_embedded_bodies / sdeh_embedded_count

namespace {

enum { SAVE_END = 0, SAVE_AT = 1, SAVE_STEPS = 2, SAVE_RUNS = 3 };
constexpr int64_t kUserBase = 1000;
constexpr int64_t kDefaultMaxiters = 10000000;
// Host-memory solves of at least kPipeMin trajectories run as kPipeChunks chunks:
// the inputs of one chunk travel to HBM while the previous chunk integrates, and
// its outputs travel back while the next one does.
constexpr int64_t kPipeMin = 1 << 17;
// Staged schedule: attempts of the first stage.  Its progress ranks the remaining
// work: on the 2^20-trajectory Lorenz ATsit5 ensemble the extrapolated remaining
// attempts after 32 attempts have a rank correlation of 0.98 with the true ones
// (0.95 after 16, 0.74 after 8).
constexpr int32_t kStageAttempts = 32;
constexpr int kPipeChunks = 4;
// Default refill batch with one lane per trajectory (see plan_solve).
constexpr int32_t kRefill = 4;
// Register-cap variants (waves per SIMD) the autotuner tries after the launch shape.
constexpr int kWaveVariants[] = {4, 6, 8};
static_assert(8 + kPipeChunks <= 16, "chunk queues live in counters[8..16)");

struct Builtin {
  int64_t id;
  const char* name;
  int32_t n, p;
  int64_t s;
  const void* (*lookup)(int, int, int, int, int, int);
  // Kernels of the group layout (`group` lanes per trajectory), if built.
  int32_t group;
  const void* (*group_lookup)(int, int, int, int, int, int);
  // Kernels of the matrix-core wave layout (`mgroup` lanes per trajectory), if built.
  int32_t mgroup;
  const void* (*mgroup_lookup)(int, int, int, int, int, int);
};

const Builtin kBuiltins[] = {
    {SDEH_RHS_LORENZ, "lorenz", 3, 3, 0, sdeh_aot_Lorenz, 1, nullptr, 0, nullptr},
    {SDEH_RHS_GLV16, "glv16", 16, 16, 256, sdeh_aot_GLV16, 16, sdeh_aot_GLV16G, 4,
     sdeh_aot_GLV16M},
    {SDEH_RHS_EXPDECAY3, "expdecay3", 3, 1, 0, sdeh_aot_ExpDecay3, 1, nullptr, 0, nullptr},
    {SDEH_RHS_AFFINE1, "affine1", 1, 2, 0, sdeh_aot_Affine1, 1, nullptr, 0, nullptr},
    {SDEH_RHS_LINEAR2, "linear2", 2, 4, 0, sdeh_aot_Linear2, 1, nullptr, 0, nullptr},
};

const Builtin* find_builtin(int64_t id) {
  for (const auto& b : kBuiltins)
    if (b.id == id) return &b;
  return nullptr;
}

struct UserRhs {
  std::string src, fn;
  int32_t n = 0, p = 0;
  int64_t s = 0;
};

struct KernelRef {
  const void* aot = nullptr;
  hipFunction_t fn = nullptr;
  int32_t lanes = 1;  // lanes per trajectory
  int32_t waves = 0;  // register-cap variant (0 = the default kernel)
  int32_t tpl = 1;    // trajectories per lane
};

struct Shape {
  int32_t schedule = SDEH_SCHED_ONE_LAUNCH, block = 256, grid = 0, chunk = 64, waves = 0,
          per_lane = 1, refill = 0;
  // a tuned packed solve's ranked passes (see run_plan) against its shape: 1 faster, 0 not,
  // -1 not timed (the tuned ensemble was too small for them)
  int32_t ranked = -1;
};

// Workgroups of a one-launch grid: every trajectory a lane (or TPL per lane).
int64_t one_launch_groups(int64_t n, const KernelRef& k, int block) {
  const int64_t lanes = (n + k.tpl - 1) / k.tpl * k.lanes;
  return (lanes + block - 1) / block;
}

// rhs, alg, dtype, save, kahan, lanes, packed
using TuneKey = std::tuple<int64_t, int, int, int, int, int, bool>;

struct GraphRec {
  hipGraph_t graph = nullptr;
  hipGraphExec_t exec = nullptr;
  void* mem = nullptr;  // queue counter + saveat copy owned by the graph
};

bool is_adaptive(int alg) {
  return alg == SDEH_ALG_ATSIT5 || alg == SDEH_ALG_AVERN7 || alg == SDEH_ALG_AVERN9;
}

uint64_t fnv1a(const std::string& s, uint64_t h = 1469598103934665603ull) {
  for (unsigned char ch : s) {
    h ^= ch;
    h *= 1099511628211ull;
  }
  return h;
}

}  // namespace

struct sdeh_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  hipStream_t s_in = nullptr, s_out = nullptr;  // host-memory pipeline copies
  hipStream_t s_k2 = nullptr;  // the pipeline's second kernel stream
  hipEvent_t ev0 = nullptr, ev1 = nullptr;
  hipEvent_t ev_pipe[2 * kPipeChunks] = {};  // per chunk: inputs landed, kernel done
  hipEvent_t ev_pipe_start = nullptr;         // the caller's stream at a pipeline's start
  std::string err;
  sdeh_stats stats{};
  int cus = 0;
  char* arena = nullptr;
  size_t arena_cap = 0;
  // [0] queue, [1..4] count_kernel outputs, [5] order check, [6] packed rows
  // offered (the offsets scan's total), [8..8+kPipeChunks) pipeline chunk queues
  unsigned long long* counters = nullptr;
  // The stream of the last call that may still be running and use the arena or
  // the counters (device-memory calls return once queued): a call on another
  // stream, or an arena reallocation, waits for it first.
  hipStream_t pending = nullptr;
  bool has_pending = false;
  std::vector<UserRhs> user;
  std::map<std::string, std::pair<hipModule_t, hipFunction_t>> rtc;
  std::map<TuneKey, Shape> tuned;
  // (rhs, alg, dtype, kahan) whose kernel of whole sectors could not be had
  std::set<std::tuple<int64_t, int, int, int>> no_runs;
  std::map<int64_t, GraphRec> graphs;
  int64_t next_graph = 1;
  // The device address of the library's static scratch on this context's device
  // (sdeh_solve_static), looked up at creation.
  unsigned long long* static_scratch = nullptr;
  size_t static_bytes = 0;
  // The order buffer sdeh_plan_order wrote last, and its length: a permutation by
  // construction, which a solve takes without the device permutation check.
  const int64_t* planned_order = nullptr;
  int64_t planned_n = 0;
};

namespace {

int fail(sdeh_ctx* c, int code, const char* fmt, ...) {
  char buf[1024];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  if (c) c->err = buf;
  return code;
}

#define HIPCHK(c, expr)                                                                    \
  do {                                                                                     \
    hipError_t e_ = (expr);                                                                \
    if (e_ != hipSuccess)                                                                  \
      return fail((c), SDEH_E_HIP, "%s failed: %s", #expr, hipGetErrorString(e_));         \
  } while (0)

int rhs_shape(sdeh_ctx* c, int64_t rhs, int32_t* n, int32_t* p, int64_t* s) {
  if (const Builtin* b = find_builtin(rhs)) {
    *n = b->n;
    *p = b->p;
    *s = b->s;
    return SDEH_OK;
  }
  const int64_t k = rhs - kUserBase;
  if (k >= 0 && k < (int64_t)c->user.size()) {
    *n = c->user[k].n;
    *p = c->user[k].p;
    *s = c->user[k].s;
    return SDEH_OK;
  }
  return fail(c, SDEH_E_INVALID, "unknown rhs %lld", (long long)rhs);
}

const std::vector<std::string>& rtc_options() {
  static const std::vector<std::string> o = {
      "--offload-arch=gfx950", "-O3", "-std=c++17", "-ffp-contract=off", "-mllvm",
      "-disable-machine-licm", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
      "-Xclang", "-target-feature", "-Xclang", "-fmacf64-inst"};
  return o;
}

// Compile (or fetch) the integrator kernel for a registered RHS.
int user_kernel(sdeh_ctx* c, int64_t rhs, int alg, int dtype, int save, int kahan,
                KernelRef* out, int waves = 0, int tpl = 1) {
  const UserRhs& u = c->user[rhs - kUserBase];
  if (waves && (!is_adaptive(alg) || save != SAVE_END))
    return fail(c, SDEH_E_UNSUPPORTED, "register-cap variants are adaptive endpoint kernels");
  if (tpl > 1 && (save != SAVE_END || waves || (alg != SDEH_ALG_ATSIT5 && alg != SDEH_ALG_AVERN7)))
    return fail(c, SDEH_E_UNSUPPORTED,
                "several trajectories per lane: ATsit5 and AVern7, endpoint output");
  char key[128];
  snprintf(key, sizeof key, "%lld/%d/%d/%d/%d/%d/%d", (long long)rhs, alg, dtype, save, kahan,
           waves, tpl);
  auto it = c->rtc.find(key);
  if (it != c->rtc.end()) {
    out->fn = it->second.second;
    out->waves = waves;
    out->tpl = tpl;
    return SDEH_OK;
  }
  const char* T = dtype == SDEH_F64 ? "double" : "float";
  std::string src = "#include \"sdeh_integrators.h\"\n";
  src += u.src;
  char wrap[2048];
  snprintf(wrap, sizeof wrap,
           "\nstruct sdeh_user_rhs {\n"
           "  static constexpr int N = %d, P = %d, S = %lld, G = 1;\n"
           "  template <class T>\n"
           "  __device__ static inline void f(T* du, const T* u, const T* p,\n"
           "                                  const T* __restrict__ ps, double t) {\n"
           "    %s<T>(du, u, p, ps, t);\n"
           "  }\n"
           "};\n",
           u.n, u.p, (long long)u.s, u.fn.c_str());
  src += wrap;
  if (tpl > 1)
    snprintf(wrap, sizeof wrap,
             "extern \"C\" __global__ void __launch_bounds__(256) sdeh_user_kernel(sdeh_kargs a) "
             "{ sdeh::adaptive_body_multi<%s, sdeh_user_rhs, %d, %s, %d>(a); }\n",
             T, alg, kahan ? "true" : "false", tpl);
  else if (is_adaptive(alg) && waves)
    snprintf(wrap, sizeof wrap,
             "extern \"C\" __global__ void __launch_bounds__(256) "
             "__attribute__((amdgpu_waves_per_eu(%d))) sdeh_user_kernel(sdeh_kargs a) "
             "{ sdeh::adaptive_body<%s, sdeh_user_rhs, %d, %d, %s, false, %d>(a); }\n",
             waves, T, alg, save, kahan ? "true" : "false", waves);
  else if (is_adaptive(alg))
    snprintf(wrap, sizeof wrap,
             "extern \"C\" __global__ void __launch_bounds__(256) "
             "__attribute__((amdgpu_waves_per_eu(sdeh::WavesHint<%s, sdeh_user_rhs, %d, %d>::value))) "
             "sdeh_user_kernel(sdeh_kargs a) "
             "{ sdeh::adaptive_body<%s, sdeh_user_rhs, %d, %d, %s>(a); }\n",
             T, alg, save, T, alg, save, kahan ? "true" : "false");
  else
    snprintf(wrap, sizeof wrap,
             "extern \"C\" __global__ void __launch_bounds__(256) sdeh_user_kernel(sdeh_kargs a) "
             "{ sdeh::fixed_body<%s, sdeh_user_rhs, %d, %d>(a); }\n",
             T, alg, save);
  src += wrap;

  std::string opts_key;
  for (const auto& o : rtc_options()) opts_key += o + " ";
  std::vector<char> code;
  const char* cache_dir = getenv("SDEH_CACHE_DIR");
  std::string cache_path;
  if (cache_dir && *cache_dir) {
    char hex[32];
    uint64_t h = fnv1a(src, fnv1a(opts_key));
    for (int i = 0; i < sdeh_embedded_count; ++i) h = fnv1a(sdeh_embedded_bodies[i], h);
    snprintf(hex, sizeof hex, "%016llx", (unsigned long long)h);
    cache_path = std::string(cache_dir) + "/sdeh_" + hex + ".co";
    if (FILE* f = fopen(cache_path.c_str(), "rb")) {
      fseek(f, 0, SEEK_END);
      const long sz = ftell(f);
      fseek(f, 0, SEEK_SET);
      if (sz > 0) {
        code.resize((size_t)sz);
        if (fread(code.data(), 1, (size_t)sz, f) != (size_t)sz) code.clear();
      }
      fclose(f);
    }
  }
  if (code.empty()) {
    hiprtcProgram prog;
    if (hiprtcCreateProgram(&prog, src.c_str(), "sdeh_user.hip", sdeh_embedded_count,
                            sdeh_embedded_bodies, sdeh_embedded_names) != HIPRTC_SUCCESS)
      return fail(c, SDEH_E_COMPILE, "hiprtcCreateProgram failed");
    std::vector<const char*> o;
    for (const auto& s : rtc_options()) o.push_back(s.c_str());
    const hiprtcResult r = hiprtcCompileProgram(prog, (int)o.size(), o.data());
    if (r != HIPRTC_SUCCESS) {
      size_t ls = 0;
      hiprtcGetProgramLogSize(prog, &ls);
      std::string log(ls, '\0');
      if (ls) hiprtcGetProgramLog(prog, &log[0]);
      hiprtcDestroyProgram(&prog);
      if (log.size() > 900) log.resize(900);
      return fail(c, SDEH_E_COMPILE, "hipRTC: %s\n%s", hiprtcGetErrorString(r), log.c_str());
    }
    size_t cs = 0;
    hiprtcGetCodeSize(prog, &cs);
    code.resize(cs);
    hiprtcGetCode(prog, code.data());
    hiprtcDestroyProgram(&prog);
    if (!cache_path.empty()) {
      const std::string tmp = cache_path + ".tmp";
      if (FILE* f = fopen(tmp.c_str(), "wb")) {
        const bool ok = fwrite(code.data(), 1, code.size(), f) == code.size();
        fclose(f);
        if (ok) rename(tmp.c_str(), cache_path.c_str());
      }
    }
  }
  hipModule_t mod;
  HIPCHK(c, hipModuleLoadData(&mod, code.data()));
  hipFunction_t fn;
  HIPCHK(c, hipModuleGetFunction(&fn, mod, "sdeh_user_kernel"));
  c->rtc[key] = {mod, fn};
  out->fn = fn;
  out->waves = waves;
  out->tpl = tpl;
  return SDEH_OK;
}

// lanes: 0 = for binary64, the matrix-core wave layout when the right-hand side has
// a kernel for the variant, else its group layout, else one lane per trajectory;
// 1 = one lane per trajectory; the group size = the group layout; the wave-layout
// size = that layout.  (Measured on GLV-16, 2^17 trajectories, AVern9 binary64 with
// 256 saveat points: 150.6 ms one lane per trajectory (the kernel spills), 18.0 ms
// in the 16-lane group layout, 10.8 ms in the 4-lane matrix-core layout; endpoint
// only 4.35 / 2.86 ms.  binary32 ATsit5 fits one lane's registers and runs 1.6x
// faster there than in the group layout, which repeats the controller on all 16
// lanes; auto_lanes says where it takes the matrix-core layout.)
int resolve_kernel(sdeh_ctx* c, int64_t rhs, int alg, int dtype, int save, int kahan,
                   int lanes, KernelRef* out, int waves = 0, int tpl = 1) {
  out->waves = 0;
  out->tpl = 1;
  if (waves && tpl > 1)
    return fail(c, SDEH_E_UNSUPPORTED,
                "register caps and several trajectories per lane do not combine");
  if (const Builtin* b = find_builtin(rhs)) {
    if (waves || tpl > 1) {  // the variants run one lane per trajectory state
      if (lanes > 1 || (lanes == 0 && dtype == SDEH_F64 && (b->mgroup > 1 || b->group > 1)))
        return fail(c, SDEH_E_UNSUPPORTED, waves ? "register-cap variants run one lane per "
                                                   "trajectory"
                                                 : "several trajectories per lane run one lane "
                                                   "per trajectory state");
      out->lanes = 1;
      out->aot = b->lookup(dtype, alg, save, kahan, waves, tpl);
      if (!out->aot)
        return fail(c, SDEH_E_UNSUPPORTED,
                    "no %s variant for rhs %s, alg %d, dtype %d, save mode %d, precision %d",
                    waves ? "register-cap" : "several-trajectories-per-lane", b->name, alg,
                    dtype, save, kahan);
      out->waves = waves;
      out->tpl = tpl;
      return SDEH_OK;
    }
    if (lanes != 0 && lanes != 1 && lanes != b->group && !(b->mgroup > 1 && lanes == b->mgroup)) {
      if (b->mgroup > 1)
        return fail(c, SDEH_E_INVALID,
                    "rhs %s runs with 1, %d or %d lanes per trajectory, not %d", b->name,
                    b->mgroup, b->group, lanes);
      if (b->group > 1)
        return fail(c, SDEH_E_INVALID, "rhs %s runs with 1 or %d lanes per trajectory, not %d",
                    b->name, b->group, lanes);
      return fail(c, SDEH_E_INVALID, "rhs %s runs with 1 lane per trajectory, not %d", b->name,
                  lanes);
    }
    if (b->mgroup > 1 && (lanes == b->mgroup || (lanes == 0 && dtype == SDEH_F64))) {
      out->aot = b->mgroup_lookup(dtype, alg, save, kahan, 0, 1);
      out->lanes = b->mgroup;
      if (out->aot) return SDEH_OK;
      if (lanes == b->mgroup)
        return fail(c, SDEH_E_UNSUPPORTED,
                    "no matrix-core kernel for rhs %s, alg %d, dtype %d, save mode %d, "
                    "precision %d", b->name, alg, dtype, save, kahan);
    }
    if ((lanes == b->group || (lanes == 0 && dtype == SDEH_F64)) && b->group > 1 &&
        b->group_lookup) {
      out->aot = b->group_lookup(dtype, alg, save, kahan, 0, 1);
      out->lanes = b->group;
      if (out->aot || lanes == b->group) {
        if (!out->aot)
          return fail(c, SDEH_E_UNSUPPORTED,
                      "no group-layout kernel for rhs %s, alg %d, dtype %d, save mode %d, "
                      "precision %d", b->name, alg, dtype, save, kahan);
        return SDEH_OK;
      }
    }
    out->lanes = 1;
    out->aot = b->lookup(dtype, alg, save, kahan, 0, 1);
    if (!out->aot)
      return fail(c, SDEH_E_UNSUPPORTED,
                  "no built-in kernel for rhs %s, alg %d, dtype %d, save mode %d, precision %d",
                  b->name, alg, dtype, save, kahan);
    return SDEH_OK;
  }
  if (lanes > 1)
    return fail(c, SDEH_E_INVALID, "registered right-hand sides run one lane per trajectory");
  out->lanes = 1;
  return user_kernel(c, rhs, alg, dtype, save, kahan, out, waves, tpl);
}

// The lanes that `lanes` = 0 stands for: in binary32 the matrix-core layout too, where it has
// a kernel and nothing that only one lane per trajectory offers is asked for.  Both layouts
// give the same bits.  One lane | matrix-core layout, GLV-16 ATsit5, tolerances 1e-6 (us):
//   n             endpoint        11 points       256 points, trajectory-major
//      1,024     367 |   115     400 |   144     570 |   236
//    131,072     650 |   450     648 |   528     955 |   880
//    524,288   1,840 | 1,400   2,037 | 1,733
// (f32 matrix products run at twice the vector rate and beside it, a wave holds a quarter of
// the trajectories, and the kernel's 107 registers leave four waves per SIMD instead of two.)
// A caller that asks for the queue keeps one lane: a grid, chunk or batch is made for the
// layout it has had, and a chunk of 64 is four of this layout's waves (120,001 trajectories
// over 20 time units 264 | 329; with the chunk left open 259 | 229).  An ensemble of at most 64
// keeps one lane too, although the layout is the faster one there as well (1 trajectory 396 |
// 90, 64 trajectories 390 | 97): callers of `lanes` = 0 have been promised it; lanes = 4 asks.
int auto_lanes(const sdeh_solve_desc* d, int save, int kahan) {
  const bool queue = d->schedule == SDEH_SCHED_PERSISTENT || d->schedule == SDEH_SCHED_STAGED ||
                     (d->schedule == SDEH_SCHED_AUTO && (d->grid || d->chunk || d->refill));
  if (d->lanes != 0 || d->dtype != SDEH_F32 || d->n_traj <= 64 || d->waves || d->per_lane || queue)
    return d->lanes;
  const Builtin* b = find_builtin(d->rhs);
  return b && b->mgroup > 1 && b->mgroup_lookup(d->dtype, d->alg, save, kahan, 0, 1) ? b->mgroup
                                                                                     : 0;
}

hipError_t launch(const KernelRef& k, int grid, int block, sdeh_kargs* a, hipStream_t s) {
  void* args[] = {a};
  if (k.aot) return hipLaunchKernel(k.aot, dim3(grid), dim3(block), args, 0, s);
  return hipModuleLaunchKernel(k.fn, grid, 1, 1, block, 1, 1, 0, s, args, nullptr);
}

int blocks_per_cu(sdeh_ctx* c, const KernelRef& k, int block) {
  int nb = 0;
  hipError_t e = k.aot ? hipOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k.aot, block, 0)
                       : hipModuleOccupancyMaxActiveBlocksPerMultiprocessor(&nb, k.fn, block, 0);
  if (e != hipSuccess || nb < 1) nb = 1;
  return nb;
}

// Device-pointer check: the range [p, p + bytes) must lie in one device
// allocation.  Refusing here is what keeps a bad caller buffer from becoming a
// GPU memory fault.
int check_dev(sdeh_ctx* c, const void* p, size_t bytes, const char* what) {
  if (bytes == 0) return SDEH_OK;
  if (!p) return fail(c, SDEH_E_INVALID, "%s is NULL", what);
  hipDeviceptr_t base = nullptr;
  size_t size = 0;
  if (hipMemGetAddressRange(&base, &size, (hipDeviceptr_t)p) != hipSuccess || !base) {
    (void)hipGetLastError();
    return fail(c, SDEH_E_INVALID, "%s is not a device allocation", what);
  }
  const char* b = (const char*)base;
  const char* q = (const char*)p;
  if (q < b || q + bytes > b + size)
    return fail(c, SDEH_E_INVALID, "%s: %zu bytes do not fit its allocation", what, bytes);
  return SDEH_OK;
}

struct Arena {
  char* base;
  size_t off = 0;
  void* take(size_t bytes) {
    if (bytes == 0) return nullptr;
    void* p = base + off;
    off += (bytes + 255) & ~size_t(255);
    return p;
  }
};

size_t round256(size_t b) { return (b + 255) & ~size_t(255); }

// Order this call's use of the context's scratch after the last call's.
int after_pending(sdeh_ctx* c, hipStream_t s) {
  if (c->has_pending && c->pending != s) {
    HIPCHK(c, hipStreamSynchronize(c->pending));
    c->has_pending = false;
  }
  return SDEH_OK;
}

void note_pending(sdeh_ctx* c, hipStream_t s, bool done) {
  c->pending = s;
  c->has_pending = !done;
}

int ensure_arena(sdeh_ctx* c, size_t need) {
  if (need <= c->arena_cap) return SDEH_OK;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (c->has_pending) HIPCHK(c, hipStreamSynchronize(c->pending));
  c->has_pending = false;
  HIPCHK(c, hipStreamSynchronize(c->s_in));  // pipeline work on the old arena
  HIPCHK(c, hipStreamSynchronize(c->s_k2));
  HIPCHK(c, hipStreamSynchronize(c->s_out));
  if (c->arena) HIPCHK(c, hipFree(c->arena));
  c->arena = nullptr;
  c->arena_cap = 0;
  size_t cap = need + need / 4 + 4096;
  if (hipMalloc((void**)&c->arena, cap) != hipSuccess) {
    (void)hipGetLastError();
    return fail(c, SDEH_E_NOMEM, "device allocation of %zu bytes failed", cap);
  }
  c->arena_cap = cap;
  return SDEH_OK;
}

struct Plan {
  int32_t n_state = 0, n_param = 0;
  int64_t n_shared = 0;
  int save = SAVE_END;
  int kahan = 0;
  size_t es = 8;  // element size of the state type
  // packed save_everystep: a counting pass (k_count, the endpoint kernel; adaptive
  // solvers only), the offsets scan, then the saving kernel
  bool packed = false;
  // the counting pass runs staged and the saving kernel takes the trajectories by
  // decreasing attempts, as counted, in one launch (see run_plan)
  bool pk_ranked = false;
  KernelRef k_runs;  // its kernel where it is not k
  // point-major saveat output by way of trajectory-major rows in scratch (see row_scratch)
  bool by_rows = false;
  void* rows_out = nullptr;
  int64_t pk_cap = 0;
  int64_t* pk_off = nullptr;
  int64_t* pk_tiles = nullptr;
  // longest-span-first hand-out order computed on the device (see span_order);
  // the pipeline's chunks alternate between two histograms
  bool span = false;
  int64_t* span_ord = nullptr;
  unsigned* span_hist[2] = {nullptr, nullptr};
  // staged schedule (see run_plan): hand-out order of the second launch and its
  // sort scratch; the parked state lives in the kargs' st_* buffers
  bool staged = false;
  bool default_staged = false;  // the library's choice: persistent where scratch is short
  int64_t* st_order = nullptr;
  unsigned* st_hist = nullptr;
  bool unchecked_order = false;  // io->order taken without the permutation check
  KernelRef k_count;
  KernelRef k;
  Shape shape;
  sdeh_kargs a{};
};

// Whether the staged schedule applies: an adaptive solve with endpoint output, one lane
// and one trajectory per lane, in the library's own order.
bool stageable(const sdeh_solve_desc* d, const sdeh_io* io, const Plan& pl) {
  return is_adaptive(d->alg) && pl.save == SAVE_END && !pl.packed && pl.k.lanes == 1 &&
         pl.k.tpl == 1 && !io->order && d->n_traj > 1 && d->n_traj < (1ll << 32);
}

// Bytes from one parked record of a staged solve to the next (whole 64-byte sectors).
size_t staged_stride(const sdeh_solve_desc* d, const Plan& pl) {
  const size_t rec = SDEH_PARK_BYTES((size_t)pl.n_state, (size_t)pl.n_param, pl.es,
                                     d->alg == SDEH_ALG_ATSIT5 ? 1 : 0, pl.kahan ? 1 : 0);
  return (rec + 63) & ~size_t(63);
}

// The launch shape of an adaptive solve that names none and has not been tuned, for `n`
// trajectories of which `sorted` says whether they are handed out longest span first,
// `ordered` whether in a caller's order, `can_stage` whether the staged schedule is open to the
// solve and `dense` whether its output is dense (see dense_output).  `resident` = lanes that fit the GPU at once.
//   one launch   up to 1 x resident lanes (endpoint output: 3 x in the span order, 1.5 x in
//                a caller's order; 2 x in binary32 with several lanes per trajectory, 4 x
//                for dense output).
//                While every wave is resident the queue only costs: its atomics, its
//                reset, and waves that take 64 slots each while others get none.
//   staged       binary64, one tspan, endpoint output, from there to 4 x: its first pass
//                ranks the trajectories (scratch bounded by kStagedBytes; no visit
//                counters, which would count a resumed trajectory twice).
//   persistent   the rest.
// Beyond resident one launch gains while a wave's trajectories are about as long as each
// other and loses once they are not, which only the solve itself shows, so the line is where
// an ensemble of unlike lengths is not slower than on the queue by more than one of like
// lengths gains.  Queue | one launch (us):
//   resident x                          1             2             3 or 4
//   Lorenz saveat 31 points AVern7, one tspan (196,608 trajectories resident)
//     rho log-uniform in 0.5 .. 200     3,523 | 3,471   4,892 | 6,161   5,888 | 8,835
//   Lorenz ATsit5 binary64, own spans, in the span order (327,680)
//     spans 0.5 .. 10                     592 |   503     815 |   757   1,070 | 1,063
//     the same, rho in 0.5 .. 200                         931 |   851   1,063 | 1,167
//     spans 9 .. 10, rho in 0.5 .. 200  (1.3 x: 1,547 | 1,702)          2,231 | 3,355
//   Lorenz ATsit5, spans 0.5 .. 10, in the order of a caller's keys, at 1.25, 1.5 and 2 x
//   binary32 compensated (458,752)
//     keys 10 % off the lengths           652 |   376     745 |   416     851 |   503
//     40 % off                            655 |   511     794 |   572     808 |   707
//     keys at random                      700 |   662     762 |   744     832 |   955
//     at random, rho in 0.5 .. 200      2,074 | 2,316   2,231 | 2,758   2,488 | 3,433
//   binary64
//     keys 10 % off the lengths           938 |   655   1,159 |   730   1,080 |   839
//     keys at random                    1,102 | 1,170   1,153 | 1,343   1,268 | 1,637
//   and 2^22 in binary32 (8 x): true lengths 1,614 | 1,373, at random 2,038 | 3,484.  A key that
//   predicts nothing costs the more the larger the ensemble, and the library cannot tell it
//   from a good one; an order that sdeh_plan_order made counts as any other.
//   GLV-16, 256 points, AVern9 binary64 on the matrix cores (32,768)
//     like growth rates                 2,224 | 2,157   4,362 | 3,987   7,247 | 6,492
//     rates over two decades            6,406 | 6,252   8,668 | 11,213 10,967 | 16,735
//   the same, ATsit5 binary32 (65,536)
//     like growth rates                   547 |   480     911 |   780   1,740 | 1,513
//     rates over two decades            2,146 | 2,039   2,358 | 2,735   4,104 | 5,780
// Parking a trajectory and resuming it costs most where it was nearly done, at mean attempts
// about the first pass's kStageAttempts, the more the further the records outgrow the caches.
// Queue | staged (us), Lorenz ATsit5 (n = 2 x, 4 x, 6.4 x resident):
//   binary64  16 attempts   286 |   268
//             31            405 |   417     673 |   727     946 | 1,108
//             44            532 |   490     923 |   874   1,301 | 1,339
//             161         2,016 | 1,525                   (5 x: 4,667 | 3,302)
//   binary32  31            366 |   383     584 |   654     814 |   993
//             56            512 |   501     814 |   877   1,153 | 1,272
//             161         1,218 |   991           (5 x: 2,808 | 2,173)
//   binary32, affine, 50    399 |   449     605 |   727     848 | 1,079
// (binary32 attempts are half as dear and their records not half as large.)
// One-lane kernels launch blocks of 64 (small ensembles spread over more CUs: 487
// against 538 us at n = 1,024; the same beyond 65,536), the others blocks of 256 (their
// LDS exchange buffers are sized for four waves: 12.9 against 7.9 ms in blocks of 64).
// Persistent layouts with several lanes per trajectory claim one wave's slots at a time,
// asked for or by default: claiming 64, a wave takes the work of several, others get none,
// and which ones get it decides the time (GLV-16 ATsit5 binary64, 500,000: 2,972 against 3,491
// us; 40,001 over 20 time units 203 against 360-436).
constexpr size_t kStagedBytes = size_t(1) << 30;

Shape default_shape(sdeh_ctx* c, const Plan& pl, int dtype, int64_t n, bool sorted,
                    bool can_stage, bool dense, bool ordered) {
  Shape sh;
  const int lanes = pl.k.lanes > 0 ? pl.k.lanes : 1;
  const int64_t work = (n + pl.k.tpl - 1) / pl.k.tpl * lanes;
  const int64_t resident = (int64_t)c->cus * blocks_per_cu(c, pl.k, 256) * 256;
  const bool end = pl.save == SAVE_END;
  const double times = dense       ? 4.0
                       : lanes > 1 ? (dtype == SDEH_F32 ? 2.0 : 1.0)
                                   : (end && sorted ? 3.0 : end && ordered ? 1.5 : 1.0);
  sh.chunk = 64 / lanes;
  if (can_stage && !sorted && dtype == SDEH_F64 && work > resident && work <= 4 * resident) {
    sh.schedule = SDEH_SCHED_STAGED;
  } else if (work <= (int64_t)(times * (double)resident)) {
    sh.schedule = SDEH_SCHED_ONE_LAUNCH;
    if (lanes == 1) sh.block = 64;
  } else {
    sh.schedule = SDEH_SCHED_PERSISTENT;
  }
  return sh;
}

// Whether point-major saveat output goes by way of trajectory-major rows in scratch and a
// transpose.  The lanes of a wave reach a save point at different times, the further apart
// the more points there are, so in the point-major layout each stores single elements,
// lines apart; the memory-side cache (256 MB) still joins them into whole lines where the
// output about fits it, and beyond that each goes to memory by itself.  The costlier a step,
// the more of that hides behind it.  Stored in place | by way of rows (us):
//   ATsit5  Lorenz binary64  150,001 x 101 points    679 |   677     524,288 x  50  1,126 | 1,154
//                            262,144 x  80           917 |   814     524,288 x  30    898 |   953
//                            262,144 x 101         1,166 |   928   1,048,576 x  30  1,551 | 1,745
//                            262,144 x 200         2,857 | 1,561
//           Lorenz binary32  262,144 x 101           845 |   607
//           GLV-16 binary32  131,072 x 256         4,942 | 1,806     131,072 x  50    578 |   702
//                  binary64   65,536 x 128         1,379 | 1,133     131,072 x  50  1,054 | 1,283
//   AVern7  Lorenz           262,144 x 200         3,942 | 3,326     262,144 x 101  2,151 | 2,272
//                            524,288 x 160         5,671 | 5,392
//   AVern9  Lorenz           524,288 x 160         9,968 | 10,125
//           GLV-16           131,072 x 120         5,535 | 5,806
// Where only some of the save times lie in the span, the copy and the transpose move the rest
// for nothing, so they are not counted, and the half has to be reached (ATsit5 Lorenz, of how
// many points reached; in place, filled beforehand):
//   262,144 x 200   100: 1,370 | 1,397   50:   818 | 1,236     700,001 x 101  50: 1,876 | 2,268
//   131,072 x 400   200: 1,442 | 1,311  100:   811 | 1,157     150,001 x 101  50:   417 |   567
// In an order (the caller's, or the longest span first) a wave's lanes hold trajectories far
// apart, no store shares a line with another lane's, and rows win from fewer points on, once
// the output is clear of that cache; with spans of their own nobody knows what is reached:
//   ATsit5 Lorenz   random order | spans of 0.2 to 3 (us, in place | by way of rows)
//     binary64  600,001 x  50 (90 M values)  3,180 | 1,430    1,190 |   980
//               300,001 x  70 (63 M)         1,660 |   910      680 |   710
//               150,001 x 101 (45 M)             not run        382 |   533
//     binary32  600,001 x 100 (180 M)        5,700 | 1,330    1,800 | 1,020
//   AVern7      300,001 x 100 (90 M)         3,020 | 1,750    1,110 | 1,100
//     binary32  300,001 x 100 (90 M)         1,510 |   930      640 |   630
//   AVern9      600,001 x  50 (90 M)         3,530 | 2,970    1,210 | 1,370  (in place, then)
// (Fixed-step solvers reach a point with all lanes at once.)
constexpr size_t kRowsFrom = size_t(300) << 20, kRowsTo = size_t(2) << 30;
constexpr size_t kOrderedRowsFrom = 75'000'000;  // values

// Save times in the common span; with spans of their own, all.
int64_t reached_points(const sdeh_solve_desc* d, const sdeh_io* io) {
  if (io->tspan) return d->n_saveat;
  return std::upper_bound(d->saveat, d->saveat + d->n_saveat, d->tf) - d->saveat;
}

bool row_scratch(const sdeh_solve_desc* d, const sdeh_io* io, const Plan& pl, size_t bytes) {
  if (pl.save != SAVE_AT || d->save_layout != SDEH_SAVE_POINT_MAJOR || bytes > kRowsTo ||
      (d->alg != SDEH_ALG_ATSIT5 && d->alg != SDEH_ALG_AVERN7))
    return false;
  const int64_t reached = reached_points(d, io);
  if (2 * reached < d->n_saveat) return false;
  if (pl.span || io->order) return reached >= 32 && bytes / pl.es > kOrderedRowsFrom;
  return reached >= (d->alg == SDEH_ALG_ATSIT5 ? 80 : 160) && bytes > kRowsFrom;
}

// Whether an adaptive solve of `n` trajectories over one span, in index order, stores in
// place point-major output so dense that one launch is the faster up to 4 x the lanes that
// fit the GPU at once, also for trajectories of unlike lengths: the lanes of a wave then stay
// near the same save times, where refilled ones do not, and such a solve waits for its stores,
// each a piece of a line.  Queue | one launch (us), like lengths and unlike ones:
//   GLV-16, 131,072, binary64 (rates over two decades)
//     AVern9  256 points  9,119 | 6,554  21,262 | 16,346     64  3,327 | 3,507   6,660 | 9,382
//     ATsit5  256 points  6,854 | 5,913  18,214 | 14,855     64  1,272 | 1,132   3,243 | 2,609
//                                                            32    836 |   781   1,579 | 2,213
//   Lorenz, 800,000, binary64 (rho log-uniform in 0.5 .. 200)
//     ATsit5   64 points  2,040 | 1,877   3,234 |  2,612     16    892 |   871   1,367 | 1,923
//     AVern7  150 points  6,829 | 5,305  10,923 |  8,953     64  2,693 | 2,570   4,229 | 5,281
//     AVern9  150 points  7,196 | 7,142   9,979 | 12,153
bool dense_output(const sdeh_solve_desc* d, const sdeh_io* io, const Plan& pl, int64_t n,
                  bool rows_open) {
  if (pl.save != SAVE_AT || d->save_layout != SDEH_SAVE_POINT_MAJOR || io->tspan || io->order ||
      (pl.k.lanes > 1 && d->dtype == SDEH_F32))
    return false;
  const size_t bytes = (size_t)d->n_saveat * pl.n_state * n * pl.es;
  const int64_t from = d->alg == SDEH_ALG_ATSIT5   ? 64
                       : d->alg == SDEH_ALG_AVERN7 ? 150
                       : pl.k.lanes > 1            ? 256
                                                   : INT64_MAX;
  return reached_points(d, io) >= from && bytes > kRowsFrom &&
         !(rows_open && row_scratch(d, io, pl, bytes));
}

// Whether u_saveat is filled with NaN before the launch, or each trajectory writes NaN to
// the rows it ended before.  The fill moves every byte of the output once more.  The kernel's
// own rows cost nothing where the save times end with the span, and more than the fill once
// there are some: a lane at a time, lines apart.  In the kernel | beforehand (us, point-major,
// by how many of the save times lie beyond the end):
//                                               none          3 %         25 %        90 %
//   Lorenz ATsit5 binary64    1,024 x 101    209 | 213    217 | 207    239 | 185    314 | 116
//                            20,001 x 101    215 | 223    222 | 219    250 | 195    356 | 129
//   and with spans of 0.2 to 3 against save times up to 3: 234 | 205, 246 | 229;
//   GLV-16 ATsit5 binary64  131,072 x 128, spans of 2 to 20: 10,657 | 3,940.
// The kernels with several lanes per trajectory write whole rows in the trajectory-major
// layout and have no need of the fill there (the same spans: 1,435), and a fixed-step
// ensemble ends all at once.
bool nan_beforehand(const sdeh_solve_desc* d, const sdeh_io* io, const Plan& pl) {
  if (pl.save != SAVE_AT || !is_adaptive(d->alg)) return false;
  if (pl.k.lanes > 1 && d->save_layout != SDEH_SAVE_POINT_MAJOR) return false;
  const double* end = d->saveat + d->n_saveat;
  return io->tspan || 16 * (end - std::upper_bound(d->saveat, end, d->tf)) > d->n_saveat;
}

// Validate the descriptor and fill everything except the device pointers.
// `path`: which entry point runs the plan (the default launch shape depends on it).
enum class Path { kDevice, kHost, kStatic, kGraph };
int plan_solve(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, Plan* pl,
               Path path = Path::kDevice) {
  if (!d || !io) return fail(c, SDEH_E_INVALID, "desc and io must not be NULL");
  if (d->alg < SDEH_ALG_TSIT5 || d->alg > SDEH_ALG_EULER)
    return fail(c, SDEH_E_INVALID, "alg %d out of range", d->alg);
  if (d->dtype != SDEH_F64 && d->dtype != SDEH_F32)
    return fail(c, SDEH_E_INVALID, "dtype %d out of range", d->dtype);
  if (d->n_traj < 0) return fail(c, SDEH_E_INVALID, "n_traj < 0");
  int r = rhs_shape(c, d->rhs, &pl->n_state, &pl->n_param, &pl->n_shared);
  if (r) return r;
  if (pl->n_shared > 0 && io->n_shared != pl->n_shared)
    return fail(c, SDEH_E_INVALID, "rhs needs %lld shared elements, io->n_shared = %lld",
                (long long)pl->n_shared, (long long)io->n_shared);
  pl->es = d->dtype == SDEH_F64 ? 8 : 4;
  const bool adaptive = is_adaptive(d->alg);
  if ((d->alg == SDEH_ALG_RK4 || d->alg == SDEH_ALG_EULER) && d->saveat && d->n_saveat > 0)
    return fail(c, SDEH_E_UNSUPPORTED,
                "GPUSimpleRK4 and GPUSimpleEuler have no dense output (saveat); the reference "
                "returns every grid point (gpurk4.jl:68-86): use save_everystep");
  if (d->saveat && d->n_saveat > 0) {
    pl->save = SAVE_AT;
    for (int64_t j = 1; j < d->n_saveat; ++j)
      if (!(d->saveat[j] >= d->saveat[j - 1]))
        return fail(c, SDEH_E_INVALID, "saveat must be ascending (entry %lld)", (long long)j);
  } else if (d->save_everystep) {
    pl->save = SAVE_STEPS;
    if (d->save_layout != SDEH_SAVE_PACKED && d->max_saves < 1)
      return fail(c, SDEH_E_INVALID,
                  "save_everystep needs max_saves >= 1 and u_steps/t_steps/n_steps buffers "
                  "(set save_everystep = 0 for endpoint-only output)");
  } else {
    pl->save = SAVE_END;
  }
  if (d->precision == SDEH_PREC_KAHAN) {
    if (d->dtype != SDEH_F32 || !adaptive)
      return fail(c, SDEH_E_UNSUPPORTED, "the compensated update is a binary32 adaptive mode");
    pl->kahan = 1;
  } else if (d->precision != SDEH_PREC_PLAIN) {
    return fail(c, SDEH_E_INVALID, "precision %d out of range", d->precision);
  }
  if (!adaptive && io->tspan)
    return fail(c, SDEH_E_UNSUPPORTED, "fixed-step solvers take one common tspan");
  if (d->block != 0 && (d->block < 64 || d->block > 256 || d->block % 64 != 0))
    return fail(c, SDEH_E_INVALID, "block must be 64, 128, 192 or 256");
  if (d->grid < 0 || d->chunk < 0) return fail(c, SDEH_E_INVALID, "grid/chunk must be >= 0");
  if (d->save_layout != SDEH_SAVE_POINT_MAJOR && d->save_layout != SDEH_SAVE_TRAJ_MAJOR &&
      d->save_layout != SDEH_SAVE_PACKED)
    return fail(c, SDEH_E_INVALID, "save_layout %d out of range", d->save_layout);
  pl->packed = d->save_layout == SDEH_SAVE_PACKED;
  if (pl->packed && pl->save != SAVE_STEPS)
    return fail(c, SDEH_E_INVALID,
                "the packed layout holds save_everystep output (save_everystep = 1, no saveat)");
  if (pl->packed && io->steps_capacity < 0)
    return fail(c, SDEH_E_INVALID, "steps_capacity < 0");

  sdeh_kargs& a = pl->a;
  a.n = d->n_traj;
  a.n_saveat = pl->save == SAVE_AT ? d->n_saveat : 0;
  a.maxiters = d->maxiters > 0 ? d->maxiters : kDefaultMaxiters;
  a.t0 = d->t0;
  a.tf = d->tf;
  a.dt = d->dt;
  a.abstol = d->abstol;
  a.reltol = d->reltol;
  // Error-norm scales m * reltol + abstol in [2^-420, 2^1022) for every finite m.
  a.err_bare = d->abstol >= 0x1p-420 && d->abstol <= 0x1p1020 && d->reltol >= 0.0 &&
               d->reltol <= 0x1p-3;
  a.max_saves = pl->save == SAVE_STEPS && !pl->packed ? d->max_saves : 0;
  a.quirks = d->quirks;
  a.traj_major = d->save_layout == SDEH_SAVE_TRAJ_MAJOR;
  if (pl->packed) {
    pl->pk_cap = io->steps_capacity;
    a.packed = 1;
  }
  if (d->schedule < SDEH_SCHED_AUTO || d->schedule > SDEH_SCHED_STAGED)
    return fail(c, SDEH_E_INVALID, "schedule %d out of range", d->schedule);
  if (d->span_order != 0 && d->span_order != 1)
    return fail(c, SDEH_E_INVALID, "span_order %d out of range", d->span_order);
  pl->span = d->span_order == 0 && adaptive && io->tspan && !io->order && d->n_traj > 1 &&
             d->n_traj < (1ll << 32);
  if (!adaptive) {
    if (d->dt == 0.0) return fail(c, SDEH_E_INVALID, "range step cannot be zero");
    const sdeh_range::Grid g = sdeh_range::make(d->t0, d->dt, d->tf);
    a.g_len = g.len;
    a.g_rational = g.rational;
    a.g_start_n = g.start_n;
    a.g_step_n = g.step_n;
    a.g_den = g.den;
    a.g_start = g.start;
    a.g_step = g.step;
  }
  r = resolve_kernel(c, d->rhs, d->alg, d->dtype, pl->save, pl->kahan,
                     auto_lanes(d, pl->save, pl->kahan), &pl->k);
  if (r) return r;
  a.filled = nan_beforehand(d, io, *pl);
  if (pl->packed && adaptive) {  // the counting pass: the endpoint kernel, same layout
    r = resolve_kernel(c, d->rhs, d->alg, d->dtype, SAVE_END, pl->kahan, pl->k.lanes,
                       &pl->k_count);
    if (r) return r;
  }

  // launch shape
  Shape sh;
  if (d->waves != 0 && d->waves != 4 && d->waves != 6 && d->waves != 8)
    return fail(c, SDEH_E_INVALID, "waves must be 0, 4, 6 or 8");
  if (d->per_lane < 0 || d->per_lane > 2)
    return fail(c, SDEH_E_INVALID, "per_lane must be 0, 1 or 2");
  if (d->refill < 0) return fail(c, SDEH_E_INVALID, "refill must be >= 0");
  if ((d->waves || d->per_lane == 2) && !adaptive)
    return fail(c, SDEH_E_UNSUPPORTED,
                "register-cap and several-trajectories-per-lane variants are adaptive endpoint "
                "kernels");
  if (adaptive) {
    auto it = c->tuned.find(TuneKey(d->rhs, d->alg, d->dtype, pl->save, pl->kahan, pl->k.lanes,
                                     pl->packed));
    if (it != c->tuned.end()) {
      sh = it->second;
    } else {
      sh.schedule = SDEH_SCHED_PERSISTENT;
      if (pl->k.lanes > 1) sh.chunk = 64 / pl->k.lanes;  // one wave's slots
    }
    // the kernel variant: the caller's register cap or trajectories per lane, else
    // the tuned ones (where they exist for this solve), else the default kernel
    const bool mine = d->waves || d->per_lane;
    const int waves = mine ? d->waves : sh.waves;
    const int tpl = mine ? (d->per_lane ? d->per_lane : 1) : sh.per_lane;
    sh.waves = 0;
    sh.per_lane = 1;
    if (waves || tpl > 1) {
      KernelRef kv;
      r = resolve_kernel(c, d->rhs, d->alg, d->dtype, pl->save, pl->kahan, pl->k.lanes, &kv,
                         waves, tpl);
      if (r && mine) return r;
      if (!r) {
        pl->k = kv;
        sh.waves = waves;
        sh.per_lane = tpl;
      }
    }
    // (a caller that sets the queue's grid, chunk or refill batch gets the queue)
    const bool open = d->schedule == SDEH_SCHED_AUTO && !d->grid && !d->chunk && !d->refill &&
                      d->n_traj > 0;
    if (it == c->tuned.end() && open) {
      const bool piped =
          path == Path::kHost && d->n_traj >= kPipeMin && !io->order && !pl->packed;
      const int64_t n = piped ? (d->n_traj + kPipeChunks - 1) / kPipeChunks : d->n_traj;
      const bool can_stage = (path == Path::kDevice || (path == Path::kHost && !piped)) &&
                             stageable(d, io, *pl) && !io->visits &&
                             (size_t)n * (staged_stride(d, *pl) + 16) <= kStagedBytes;
      const int32_t w = sh.waves, tp = sh.per_lane;
      sh = default_shape(c, *pl, d->dtype, n, pl->span && path != Path::kStatic, can_stage,
                         dense_output(d, io, *pl, n, path == Path::kDevice), io->order != nullptr);
      sh.waves = w;
      sh.per_lane = tp;
      pl->default_staged = sh.schedule == SDEH_SCHED_STAGED;
    }
    // Packed output beyond resident: rank the saving pass by the counting pass, unless the
    // tuner has found this solve's shape to be faster.
    const int64_t n = d->n_traj;
    if (open && (it == c->tuned.end() || it->second.ranked != 0) && pl->packed &&
        pl->k.lanes == 1 && !io->order && !io->visits && n > 1 && n < (1ll << 32) &&
        n > (int64_t)c->cus * blocks_per_cu(c, pl->k, 256) * 256 &&
        (size_t)n * (staged_stride(d, *pl) + 16) <= kStagedBytes) {
      pl->pk_ranked = true;
      sh.schedule = SDEH_SCHED_ONE_LAUNCH;
      sh.block = 256;
      pl->span = false;
      // the kernel that writes its rows by whole sectors, for states of at most 32 bytes
      const auto id = std::make_tuple(d->rhs, d->alg, d->dtype, pl->kahan);
      if ((size_t)pl->n_state * pl->es <= 32 && !c->no_runs.count(id)) {
        KernelRef kr;
        const std::string err = c->err;
        if (!resolve_kernel(c, d->rhs, d->alg, d->dtype, SAVE_RUNS, pl->kahan, 1, &kr)) {
          pl->k_runs = kr;
        } else {  // row by row, then: no error of this call, and not tried again
          c->err = err;
          c->no_runs.insert(id);
        }
      }
    }
    if (d->schedule != SDEH_SCHED_AUTO) sh.schedule = d->schedule;
    if (d->block) sh.block = d->block;
    if (d->chunk) sh.chunk = d->chunk;
    if (sh.schedule == SDEH_SCHED_PERSISTENT || sh.schedule == SDEH_SCHED_STAGED) {
      if (d->grid) sh.grid = d->grid;
      else if (it == c->tuned.end() || d->block || it->second.schedule != sh.schedule ||
               it->second.waves != sh.waves || it->second.per_lane != sh.per_lane)
        sh.grid = c->cus * blocks_per_cu(c, pl->k, sh.block);
      if (sh.grid < 1) sh.grid = 1;
    }
  } else {
    sh.schedule = SDEH_SCHED_ONE_LAUNCH;
    if (d->block) sh.block = d->block;
  }
  // The kernel that keeps its constants in registers, for ensembles of a wave or two
  // per SIMD (AVern9: one, its 302 registers allow no second).  Lorenz, the default
  // kernel | this one (us; ATsit5, AVern7, AVern9):
  //      1,024    89 | 81     197 | 162     391 | 354
  //     65,536    95 | 86     204 | 165     412 | 370
  //    131,072   127 | 122    274 | 250     561 | 782
  //    262,144   205 | 242    467 | 474     951 | 1,252
  // with 11 saved points
  //      1,024   122 | 110    366 | 345     762 | 836 (AVern9: not built)
  //    131,072   166 | 157    489 | 473
  // every step in packed rows (AVern9's counting pass only)
  //      1,024   202 | 186    419 | 361     793 | 751
  //    131,072   290 | 280    605 | 580   1,147 | 1,146
  const int64_t simds = 4 * (int64_t)c->cus;
  if (sh.schedule == SDEH_SCHED_ONE_LAUNCH && d->dtype == SDEH_F64 && adaptive &&
      pl->k.lanes == 1 && !sh.waves && sh.per_lane <= 1 &&
      d->n_traj <= simds * 64 * (d->alg == SDEH_ALG_AVERN9 ? 1 : 2)) {
    const Builtin* b = find_builtin(d->rhs);
    const void* lone = b ? b->lookup(d->dtype, d->alg, pl->save, 0, 1, 1) : nullptr;
    if (lone) pl->k.aot = lone;
    lone = b && pl->packed ? b->lookup(d->dtype, d->alg, SAVE_END, 0, 1, 1) : nullptr;
    if (lone) pl->k_count.aot = lone;
  }
  if (sh.schedule == SDEH_SCHED_ONE_LAUNCH) {
    const int64_t g = one_launch_groups(d->n_traj, pl->k, sh.block);
    if (g > 0x7fffffff) return fail(c, SDEH_E_INVALID, "ensemble too large for one launch");
    sh.grid = (int)g;
  }
  if (sh.schedule == SDEH_SCHED_STAGED) {
    // endpoint output, one lane per trajectory, the library's own order; the
    // second launch is the persistent one, so a staged shape falls back to it
    pl->staged = stageable(d, io, *pl);
    if (!pl->staged) sh.schedule = SDEH_SCHED_PERSISTENT;
    // (a staged solve orders its second launch itself; pl->span stays for the paths
    // that run the shape as persistent: graph capture, the host pipeline)
  }
  a.persistent = sh.schedule == SDEH_SCHED_PERSISTENT || sh.schedule == SDEH_SCHED_STAGED;
  a.chunk = sh.chunk;
  // refill batch: the caller's, else the tuned one, else 4 slots with one lane per
  // trajectory (measured on the 2^22 Lorenz ensemble: 4.5% faster binary64, 7%
  // binary32, than claiming for each free slot) and 1 with several lanes
  if (a.persistent && pl->k.tpl > 1) {
    sh.refill = 1;  // the two-per-lane kernels claim for each free slot
  } else if (a.persistent) {
    const int slots = 64 / (pl->k.lanes > 0 ? pl->k.lanes : 1);
    int rf = d->refill ? d->refill : sh.refill;
    if (!rf) rf = pl->k.lanes == 1 ? kRefill : 1;
    sh.refill = rf < slots ? rf : slots;
  } else {
    sh.refill = 0;
  }
  a.refill_min = sh.refill;
  pl->shape = sh;
  return SDEH_OK;
}

// Bytes of each io buffer for a plan.
struct Sizes {
  size_t u0, p, ps, tspan, dt0, order, u_end, t_end, i32, u_saveat, u_steps, t_steps, saveat;
  // packed layout: offsets output and scan scratch; span order and its histogram
  size_t pk_off, pk_tiles, span_order, span_hist;
  // staged schedule: parked records (st_stride bytes each), key and order ([n]),
  // sort scratch
  size_t st_rec, st_stride, st_key, st_order, st_hist;
};

Sizes sizes_of(const sdeh_solve_desc* d, const sdeh_io* io, const Plan& pl) {
  const size_t n = (size_t)d->n_traj;
  Sizes s{};
  s.u0 = (size_t)pl.n_state * n * pl.es;
  s.p = (size_t)pl.n_param * n * pl.es;
  s.ps = (size_t)pl.n_shared * pl.es;
  s.tspan = io->tspan ? 2 * n * 8 : 0;
  s.dt0 = io->dt0 ? n * 8 : 0;
  s.order = io->order ? n * 8 : 0;
  s.u_end = s.u0;
  s.t_end = n * 8;
  s.i32 = n * 4;
  s.u_saveat = pl.save == SAVE_AT ? (size_t)d->n_saveat * pl.n_state * n * pl.es : 0;
  s.u_steps = pl.save == SAVE_STEPS ? (size_t)d->max_saves * pl.n_state * n * pl.es : 0;
  s.t_steps = pl.save == SAVE_STEPS ? (size_t)d->max_saves * n * 8 : 0;
  s.saveat = pl.save == SAVE_AT ? (size_t)d->n_saveat * 8 : 0;
  if (pl.span) {
    s.span_order = n * 8;
    s.span_hist = sdeh_util_span_scratch_bytes();
  }
  if (pl.staged || pl.pk_ranked) {
    s.st_stride = staged_stride(d, pl);
    s.st_rec = n * s.st_stride;
    s.st_key = n * 8;
    s.st_order = n * 8;
    s.st_hist = sdeh_util_span_scratch_bytes();
  }
  if (pl.packed) {
    const size_t cap = (size_t)pl.pk_cap;
    s.u_steps = cap * pl.n_state * pl.es;
    s.t_steps = cap * 8;
    s.pk_off = (n + 1) * 8;
    s.pk_tiles = ((n + 1023) / 1024 + 1) * 8;
  }
  return s;
}

int check_order_host(sdeh_ctx* c, const int64_t* order, int64_t n) {
  std::vector<unsigned char> seen((size_t)n, 0);
  for (int64_t i = 0; i < n; ++i) {
    const int64_t v = order[i];
    if (v < 0 || v >= n || seen[(size_t)v])
      return fail(c, SDEH_E_INVALID, "order is not a permutation of 0..n_traj-1 (entry %lld)",
                  (long long)i);
    seen[(size_t)v] = 1;
  }
  return SDEH_OK;
}

// The staged launches of kernel `k` (`grid` persistent blocks of `block`): every
// trajectory runs its first kStageAttempts attempts in a one-launch pass; those still
// running park their state and an estimate of the attempts they still need, the
// estimates are counting-sorted (largest first), and a persistent launch resumes the
// parked trajectories in that order, so the longest start first and the end of the
// launch drains less.  Its queue starts behind the trajectories that have ended, which
// the order does not name: with them in it, an ensemble of short trajectories paid for
// a queue of ended ones (linear decay, 14 attempts each, 2.6 M trajectories 1,090 us, now 561).
// Parking stores the whole per-trajectory state (one record each, so the resumed pass
// reads one or two cache lines per trajectory whatever the order), and every trajectory
// takes the same steps as in one launch.
int launch_staged(sdeh_ctx* c, const Plan& pl, const KernelRef& k, int grid, int block,
                  unsigned long long* queue, hipStream_t s) {
  sdeh_kargs a1 = pl.a;
  a1.persistent = 0;
  a1.order = nullptr;
  a1.stage_cap = kStageAttempts;
  a1.resume = 0;
  const int64_t g1 = (a1.n * k.lanes + block - 1) / block;
  HIPCHK(c, launch(k, (int)g1, block, &a1, s));
  HIPCHK(c, sdeh_util_resume_order(a1.st_key, a1.n, pl.st_hist, pl.st_order, queue, s));
  sdeh_kargs a2 = pl.a;
  a2.persistent = 1;
  a2.order = pl.st_order;
  a2.stage_cap = 0;
  a2.resume = 1;
  if (a2.refill_min == 0) a2.refill_min = kRefill;  // the plan's own launch has no queue
  HIPCHK(c, launch(k, grid, block, &a2, s));
  return SDEH_OK;
}

// Launch the prepared plan on `s` (kernel bracketed by the context events).
int run_plan(sdeh_ctx* c, Plan& pl, hipStream_t s, unsigned long long* queue, bool timed) {
  sdeh_kargs& a = pl.a;
  // NaN for the rows not reached, unless the kernel writes it (see nan_beforehand); and for
  // those of trajectories that an order not checked to be a permutation may leave out.
  if (pl.save == SAVE_AT && (a.filled || pl.unchecked_order)) {
    const int64_t cnt = a.n_saveat * pl.n_state * a.n;
    if (pl.es == 8) HIPCHK(c, sdeh_util_fill_f64((double*)a.u_saveat, __builtin_nan(""), cnt, s));
    else HIPCHK(c, sdeh_util_fill_f32((float*)a.u_saveat, __builtin_nanf(""), cnt, s));
  }
  a.queue = queue;
  if (a.n > 0) {
    if (timed) HIPCHK(c, hipEventRecord(c->ev0, s));
    if (pl.packed) {
      // rows per trajectory: naccept + 1 from an endpoint pass (the same arithmetic,
      // so the same steps), or the grid length of a fixed-step solver
      const bool counted = pl.k_count.aot || pl.k_count.fn;
      if (pl.pk_ranked) {
        const int grid = c->cus * blocks_per_cu(c, pl.k_count, 256);
        const int st = launch_staged(c, pl, pl.k_count, grid, 256, queue, s);
        if (st) return st;
      } else if (counted) {
        if (a.persistent) HIPCHK(c, sdeh_util_zero_u64(queue, 1, s));
        HIPCHK(c, launch(pl.k_count, pl.shape.grid, pl.shape.block, &a, s));
      }
      const int32_t add = counted ? 1 : (int32_t)std::max<int64_t>(a.g_len, 1);
      HIPCHK(c, sdeh_util_pack_offsets(counted ? a.naccept : nullptr, add, a.n, pl.pk_tiles,
                                       pl.pk_cap, pl.pk_off, a.n_steps, c->counters + 6, s));
      // The counts rank the saving pass exactly: waves of equal lengths, longest first.
      // (Lorenz ATsit5, 2^20 trajectories, 67 M rows: 3,120 us with both passes persistent;
      // 2,820 with the staged endpoint pass and the ranked saving pass; 2,220 with the
      // latter writing whole sectors and the controller's tables in LDS.)
      if (pl.pk_ranked) {
        HIPCHK(c, sdeh_util_count_order(a.naccept, a.nreject, a.n, pl.st_hist, pl.st_order, s));
        a.order = pl.st_order;
      }
    }
    if (pl.staged) {
      const int st = launch_staged(c, pl, pl.k, pl.shape.grid, pl.shape.block, queue, s);
      if (st) return st;
    } else {
      if (a.persistent) HIPCHK(c, sdeh_util_zero_u64(queue, 1, s));
      // (its kernel finds whole elements in the outputs' 64-byte sectors)
      const bool runs = pl.pk_ranked && (pl.k_runs.aot || pl.k_runs.fn) &&
                        (uintptr_t)a.u_steps % pl.es == 0 && (uintptr_t)a.t_steps % 8 == 0;
      HIPCHK(c, launch(runs ? pl.k_runs : pl.k, pl.shape.grid, pl.shape.block, &a, s));
    }
    if (pl.by_rows)
      HIPCHK(c, sdeh_util_transpose(a.u_saveat, pl.rows_out, a.n, a.n_saveat * pl.n_state,
                                    (int)pl.es, s));
    if (timed) HIPCHK(c, hipEventRecord(c->ev1, s));
  }
  return SDEH_OK;
}

// Trajectories [a, a + m) of a host array with `rows` rows per trajectory, to or
// from its device copy.  Host: [row][n] (element (r, i) at r * n + i), or, with
// traj_major, [n][row].  Device: the chunk-blocked copy, in which chunk [a, a+m)
// is a standalone [row][m] (or [m][row]) array starting at element rows * a.
hipError_t chunk_copy(char* dev, const void* host_in, void* host_out, size_t es, int64_t rows,
                      int64_t n, int64_t a, int64_t m, bool traj_major, hipStream_t st) {
  const bool h2d = host_in != nullptr;
  char* host = h2d ? (char*)host_in : (char*)host_out;
  if (!host || rows == 0 || m == 0) return hipSuccess;
  char* dblk = dev + (size_t)rows * a * es;
  if (traj_major || rows == 1) {
    char* hblk = host + (size_t)rows * a * es;
    const size_t bytes = (size_t)rows * m * es;
    return h2d ? hipMemcpyAsync(dblk, hblk, bytes, hipMemcpyHostToDevice, st)
               : hipMemcpyAsync(hblk, dblk, bytes, hipMemcpyDeviceToHost, st);
  }
  char* hcol = host + (size_t)a * es;
  const size_t w = (size_t)m * es, hp = (size_t)n * es;
  return h2d ? hipMemcpy2DAsync(dblk, w, hcol, hp, w, (size_t)rows, hipMemcpyHostToDevice, st)
             : hipMemcpy2DAsync(hcol, hp, dblk, w, w, (size_t)rows, hipMemcpyDeviceToHost, st);
}

// Host-memory solve in kPipeChunks chunks of trajectories: inputs go up on s_in,
// each chunk integrates as a standalone ensemble once its inputs have landed
// (chunks alternate between `s` and s_k2, so one chunk's end-of-launch drain
// overlaps the next one's start; each has its own work-queue counter), and its
// outputs come back on s_out once its kernel is done.  The device buffers in
// pl.a are chunk-blocked (chunk_copy).  ev0/ev1 bracket the kernels, and `s`
// finishes after all of them.  Per-trajectory results do not depend on the
// chunking.
int run_host_pipeline(sdeh_ctx* c, Plan& pl, const sdeh_io* io, hipStream_t s) {
  const sdeh_kargs base = pl.a;
  const int64_t n = base.n, N = pl.n_state, P = pl.n_param;
  const int64_t ns = base.n_saveat, ms = base.max_saves;
  const size_t es = pl.es;
  const bool tm = base.traj_major != 0;
  const int K = kPipeChunks;
  // Everything already queued on `s` comes first: an earlier device-memory solve on
  // `s` that may still be running (its arena scratch is what the chunk uploads
  // overwrite) and this call's own uploads of the saveat times and p_shared, which
  // the chunks on s_k2 read.  The three pipeline streams wait for that point.
  HIPCHK(c, hipEventRecord(c->ev_pipe_start, s));
  HIPCHK(c, hipStreamWaitEvent(c->s_in, c->ev_pipe_start, 0));
  HIPCHK(c, hipStreamWaitEvent(c->s_k2, c->ev_pipe_start, 0));
  HIPCHK(c, hipStreamWaitEvent(c->s_out, c->ev_pipe_start, 0));
  auto offs = [](const void* p, int64_t rows, int64_t a, size_t e) -> void* {
    return p ? (void*)((char*)p + (size_t)rows * a * e) : nullptr;
  };
  auto down = [&](int k) -> int {
    const int64_t a0 = n * k / K, m = n * (k + 1) / K - a0;
    HIPCHK(c, hipStreamWaitEvent(c->s_out, c->ev_pipe[K + k], 0));
    const hipStream_t so = c->s_out;
    HIPCHK(c, chunk_copy((char*)base.u_end, nullptr, io->u_end, es, N, n, a0, m, false, so));
    HIPCHK(c, chunk_copy((char*)base.t_end, nullptr, io->t_end, 8, 1, n, a0, m, false, so));
    HIPCHK(c, chunk_copy((char*)base.retcode, nullptr, io->retcode, 4, 1, n, a0, m, false, so));
    HIPCHK(c, chunk_copy((char*)base.naccept, nullptr, io->naccept, 4, 1, n, a0, m, false, so));
    HIPCHK(c, chunk_copy((char*)base.nreject, nullptr, io->nreject, 4, 1, n, a0, m, false, so));
    if (pl.save == SAVE_AT)
      HIPCHK(c, chunk_copy((char*)base.u_saveat, nullptr, io->u_saveat, es, ns * N, n, a0, m, tm,
                           so));
    if (pl.save == SAVE_STEPS) {
      HIPCHK(c, chunk_copy((char*)base.u_steps, nullptr, io->u_steps, es, ms * N, n, a0, m, tm,
                           so));
      HIPCHK(c, chunk_copy((char*)base.t_steps, nullptr, io->t_steps, 8, ms, n, a0, m, tm, so));
      HIPCHK(c, chunk_copy((char*)base.n_steps, nullptr, io->n_steps, 4, 1, n, a0, m, false, so));
    }
    return SDEH_OK;
  };
  for (int k = 0; k < K; ++k) {
    const int64_t a0 = n * k / K, m = n * (k + 1) / K - a0;
    const hipStream_t si = c->s_in;
    HIPCHK(c, chunk_copy((char*)base.u0, io->u0, nullptr, es, N, n, a0, m, false, si));
    HIPCHK(c, chunk_copy((char*)base.p, io->p, nullptr, es, P, n, a0, m, false, si));
    if (io->tspan)
      HIPCHK(c, chunk_copy((char*)base.tspan, io->tspan, nullptr, 8, 2, n, a0, m, false, si));
    if (io->dt0)
      HIPCHK(c, chunk_copy((char*)base.dt0, io->dt0, nullptr, 8, 1, n, a0, m, false, si));
    const hipStream_t sk = (k & 1) ? c->s_k2 : s;
    HIPCHK(c, hipEventRecord(c->ev_pipe[k], si));
    HIPCHK(c, hipStreamWaitEvent(sk, c->ev_pipe[k], 0));
    Plan cp = pl;
    sdeh_kargs& ka = cp.a;
    ka.n = m;
    if (cp.shape.schedule == SDEH_SCHED_ONE_LAUNCH)
      cp.shape.grid = (int)one_launch_groups(m, cp.k, cp.shape.block);
    ka.order = nullptr;
    ka.u0 = offs(base.u0, N, a0, es);
    ka.p = offs(base.p, P, a0, es);
    ka.tspan = (const double*)offs(base.tspan, 2, a0, 8);
    ka.dt0 = (const double*)offs(base.dt0, 1, a0, 8);
    ka.u_end = offs(base.u_end, N, a0, es);
    ka.t_end = (double*)offs(base.t_end, 1, a0, 8);
    ka.retcode = (int32_t*)offs(base.retcode, 1, a0, 4);
    ka.naccept = (int32_t*)offs(base.naccept, 1, a0, 4);
    ka.nreject = (int32_t*)offs(base.nreject, 1, a0, 4);
    ka.u_saveat = offs(base.u_saveat, ns * N, a0, es);
    ka.u_steps = offs(base.u_steps, ms * N, a0, es);
    ka.t_steps = (double*)offs(base.t_steps, ms, a0, 8);
    ka.n_steps = (int32_t*)offs(base.n_steps, 1, a0, 4);
    if (pl.span && m > 1) {
      HIPCHK(c, sdeh_util_span_order(ka.tspan, m, pl.span_hist[k & 1], pl.span_ord + a0, sk));
      ka.order = pl.span_ord + a0;
    }
    if (k == 0) HIPCHK(c, hipEventRecord(c->ev0, s));
    int r = run_plan(c, cp, sk, c->counters + 8 + k, false);
    if (r) return r;
    HIPCHK(c, hipEventRecord(c->ev_pipe[K + k], sk));
    // the previous chunk's outputs go back now: its kernel is done or nearly so,
    // and this chunk's kernel is already queued behind it
    if (k > 0) {
      r = down(k - 1);
      if (r) return r;
    }
  }
  int r = down(K - 1);
  if (r) return r;
  for (int k = 1; k < K; k += 2) HIPCHK(c, hipStreamWaitEvent(s, c->ev_pipe[K + k], 0));
  HIPCHK(c, hipEventRecord(c->ev1, s));
  return SDEH_OK;
}

int solve_impl(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, int32_t memory,
               hipStream_t s, int32_t sync) {
  const auto t_start = std::chrono::steady_clock::now();
  Plan pl;
  int r = plan_solve(c, d, io, &pl, memory == SDEH_MEM_HOST ? Path::kHost : Path::kDevice);
  if (r) return r;
  r = after_pending(c, s);
  if (r) return r;
  Sizes sz = sizes_of(d, io, pl);
  const int64_t n = d->n_traj;
  if (n > 0) {
    if (!io->u0 || !io->u_end || !io->t_end || !io->retcode)
      return fail(c, SDEH_E_INVALID, "u0, u_end, t_end and retcode are required");
    if (pl.n_param > 0 && !io->p) return fail(c, SDEH_E_INVALID, "p is required (n_param > 0)");
    if (pl.n_shared > 0 && !io->p_shared)
      return fail(c, SDEH_E_INVALID, "p_shared is required for this rhs");
    if (pl.save == SAVE_AT && !io->u_saveat)
      return fail(c, SDEH_E_INVALID, "u_saveat is required with saveat");
    // (a packed call with steps_capacity 0 stores no rows: it reports steps_needed)
    const bool rows = !(pl.packed && pl.pk_cap == 0);
    if (pl.save == SAVE_STEPS && ((rows && (!io->u_steps || !io->t_steps)) || !io->n_steps))
      return fail(c, SDEH_E_INVALID, "u_steps, t_steps and n_steps are required");
    if (pl.packed && !io->steps_offset)
      return fail(c, SDEH_E_INVALID, "steps_offset is required with the packed layout");
  }
  sdeh_kargs& a = pl.a;
  const bool host = memory == SDEH_MEM_HOST;
  if (!host && memory != SDEH_MEM_DEVICE) return fail(c, SDEH_E_INVALID, "memory mode");
  if (host && io->visits)
    return fail(c, SDEH_E_INVALID, "visits counters take device memory (SDEH_MEM_DEVICE)");
  if (host && io->order && n > 0) {
    r = check_order_host(c, io->order, n);
    if (r) return r;
  }
  if (pl.staged && host && n >= kPipeMin && !pl.packed) {  // the pipeline's chunks run persistent
    pl.staged = false;
    pl.shape.schedule = SDEH_SCHED_PERSISTENT;
  }

  pl.by_rows = !host && row_scratch(d, io, pl, sz.u_saveat);
  // Device layout: saveat copy + (host mode) all buffers + counters always.
  const bool own_counts = !io->naccept || !io->nreject || host;
  auto scratch_need = [&]() {
    size_t need = round256(sz.saveat);
    if (host) {
      need += round256(sz.u0) + round256(sz.p) + round256(sz.ps) + round256(sz.tspan) +
              round256(sz.dt0) + round256(sz.order) + round256(sz.u_end) + round256(sz.t_end) +
              round256(sz.i32) + round256(sz.u_saveat) + round256(sz.u_steps) +
              round256(sz.t_steps) + round256(sz.i32);
    }
    if (own_counts) need += 2 * round256(sz.i32);
    if (!host && io->order) need += round256(sz.i32);
    if (pl.packed) {
      need += round256(sz.pk_tiles);
      if (host) need += round256(sz.pk_off);
    }
    if (pl.span) need += round256(sz.span_order) + 2 * round256(sz.span_hist);
    if (pl.by_rows) need += round256(sz.u_saveat);
    if (pl.staged || pl.pk_ranked)
      need += round256(sz.st_rec) + round256(sz.st_key) + round256(sz.st_order) +
              round256(sz.st_hist);
    return need;
  };
  // the persistent schedule instead of the parked records
  auto drop_records = [&]() {
    if (pl.pk_ranked) {
      pl.shape.block = d->block ? d->block : 256;
      pl.shape.grid = c->cus * blocks_per_cu(c, pl.k, pl.shape.block);
      a.persistent = 1;
    }
    pl.staged = pl.default_staged = pl.pk_ranked = false;
    pl.shape.schedule = SDEH_SCHED_PERSISTENT;
    sz = sizes_of(d, io, pl);
  };
  // A caller's capture of `s` records the launches for later replays.  The records and rows
  // live in the arena, which cannot be allocated during a capture and which a later, larger
  // solve frees while the graph still writes to it, so a captured solve does without them.
  if (!host && (pl.default_staged || pl.pk_ranked || pl.by_rows)) {
    hipStreamCaptureStatus cs = hipStreamCaptureStatusNone;
    HIPCHK(c, hipStreamIsCapturing(s, &cs));
    if (cs != hipStreamCaptureStatusNone) {
      if (pl.default_staged || pl.pk_ranked) drop_records();
      pl.by_rows = false;
    }
  }
  r = ensure_arena(c, scratch_need());
  if (r == SDEH_E_NOMEM && (pl.default_staged || pl.pk_ranked)) {
    // no room for the parked records
    drop_records();
    c->err.clear();
    r = ensure_arena(c, scratch_need());
  }
  if (r == SDEH_E_NOMEM && pl.by_rows) {  // no room for the rows: stored where they belong
    pl.by_rows = false;
    c->err.clear();
    r = ensure_arena(c, scratch_need());
  }
  if (r) return r;
  Arena ar{c->arena};
  double* d_saveat = (double*)ar.take(sz.saveat);
  if (sz.saveat) HIPCHK(c, hipMemcpyAsync(d_saveat, d->saveat, sz.saveat, hipMemcpyHostToDevice, s));
  a.saveat = d_saveat;
  // host memory: the pipeline moves per-trajectory inputs and outputs chunk by
  // chunk; shared inputs (p_shared, order) go up once
  const bool piped = host && n >= kPipeMin && !io->order && !pl.packed;
  if (host) {
    auto up = [&](const void* src, size_t b, bool per_traj) -> void* {
      void* p = ar.take(b);
      if (b && src && !(piped && per_traj))
        (void)hipMemcpyAsync(p, src, b, hipMemcpyHostToDevice, s);
      return p;
    };
    a.u0 = up(io->u0, sz.u0, true);
    a.p = up(io->p, sz.p, true);
    a.ps = up(io->p_shared, sz.ps, false);
    a.tspan = (const double*)up(io->tspan, sz.tspan, true);
    a.dt0 = (const double*)up(io->dt0, sz.dt0, true);
    a.order = (const int64_t*)up(io->order, sz.order, false);
    HIPCHK(c, hipGetLastError());
    a.u_end = ar.take(sz.u_end);
    a.t_end = (double*)ar.take(sz.t_end);
    a.retcode = (int32_t*)ar.take(sz.i32);
    a.u_saveat = ar.take(sz.u_saveat);
    a.u_steps = ar.take(sz.u_steps);
    a.t_steps = (double*)ar.take(sz.t_steps);
    a.n_steps = (int32_t*)ar.take(pl.save == SAVE_STEPS ? sz.i32 : 0);
  } else if (n > 0) {
    r = check_dev(c, io->u0, sz.u0, "u0");
    if (!r) r = check_dev(c, io->p, sz.p, "p");
    if (!r) r = check_dev(c, io->p_shared, sz.ps, "p_shared");
    if (!r && io->tspan) r = check_dev(c, io->tspan, sz.tspan, "tspan");
    if (!r && io->dt0) r = check_dev(c, io->dt0, sz.dt0, "dt0");
    if (!r && io->order) r = check_dev(c, io->order, sz.order, "order");
    if (!r) r = check_dev(c, io->u_end, sz.u_end, "u_end");
    if (!r) r = check_dev(c, io->t_end, sz.t_end, "t_end");
    if (!r) r = check_dev(c, io->retcode, sz.i32, "retcode");
    if (!r && io->naccept) r = check_dev(c, io->naccept, sz.i32, "naccept");
    if (!r && io->nreject) r = check_dev(c, io->nreject, sz.i32, "nreject");
    if (!r && io->visits) r = check_dev(c, io->visits, sz.i32, "visits");
    if (!r && pl.save == SAVE_AT) r = check_dev(c, io->u_saveat, sz.u_saveat, "u_saveat");
    if (!r && pl.save == SAVE_STEPS) {
      r = check_dev(c, io->u_steps, sz.u_steps, "u_steps");
      if (!r) r = check_dev(c, io->t_steps, sz.t_steps, "t_steps");
      if (!r) r = check_dev(c, io->n_steps, sz.i32, "n_steps");
      if (!r && pl.packed) r = check_dev(c, io->steps_offset, sz.pk_off, "steps_offset");
    }
    if (r) return r;
    a.visits = io->visits;
    a.u0 = io->u0;
    a.p = io->p;
    a.ps = io->p_shared;
    a.tspan = io->tspan;
    a.dt0 = io->dt0;
    a.order = io->order;
    a.u_end = io->u_end;
    a.t_end = io->t_end;
    a.retcode = io->retcode;
    a.u_saveat = io->u_saveat;
    a.u_steps = io->u_steps;
    a.t_steps = io->t_steps;
    a.n_steps = io->n_steps;
  }
  if (pl.by_rows && n > 0) {
    pl.rows_out = a.u_saveat;
    if (pl.k.lanes > 1) a.filled = 0;  // whole rows now
    a.u_saveat = ar.take(sz.u_saveat);
    a.traj_major = 1;
  }
  a.naccept = (!host && io->naccept) ? io->naccept : nullptr;
  a.nreject = (!host && io->nreject) ? io->nreject : nullptr;
  if (!a.naccept) a.naccept = (int32_t*)ar.take(sz.i32);
  if (!a.nreject) a.nreject = (int32_t*)ar.take(sz.i32);
  if (pl.packed) {
    pl.pk_off = host ? (int64_t*)ar.take(sz.pk_off) : io->steps_offset;
    pl.pk_tiles = (int64_t*)ar.take(sz.pk_tiles);
    a.steps_off = pl.pk_off;
    if (n == 0 && io->steps_offset) {
      if (host) {
        io->steps_offset[0] = 0;
      } else {
        r = check_dev(c, io->steps_offset, 8, "steps_offset");
        if (r) return r;
        HIPCHK(c, hipMemsetAsync(io->steps_offset, 0, 8, s));
      }
    }
  }
  if (pl.span && !pl.staged) {  // longest span first (the pipeline orders each chunk itself)
    pl.span_ord = (int64_t*)ar.take(sz.span_order);
    pl.span_hist[0] = (unsigned*)ar.take(sz.span_hist);
    pl.span_hist[1] = (unsigned*)ar.take(sz.span_hist);
    if (!piped) {
      HIPCHK(c, sdeh_util_span_order(a.tspan, n, pl.span_hist[0], pl.span_ord, s));
      a.order = pl.span_ord;
    }
  }
  if (pl.staged || pl.pk_ranked) {
    a.st_rec = ar.take(sz.st_rec);
    a.st_stride = (int64_t)sz.st_stride;
    a.st_key = (double*)ar.take(sz.st_key);
    pl.st_order = (int64_t*)ar.take(sz.st_order);
    pl.st_hist = (unsigned*)ar.take(sz.st_hist);
  }

  // Permutation check on the device, except for the order sdeh_plan_order wrote last
  // (the kernels still never read an entry outside [0, n)).
  const bool planned = io->order == c->planned_order && n == c->planned_n;
  pl.unchecked_order = !host && io->order && planned;
  if (!host && io->order && n > 0 && !planned) {
    int32_t* seen = (int32_t*)ar.take(sz.i32);
    HIPCHK(c, sdeh_util_zero_u64(c->counters + 5, 1, s));
    HIPCHK(c, sdeh_util_check_order(io->order, n, seen, c->counters + 5, s));
    unsigned long long bad = 0;
    HIPCHK(c, hipMemcpyAsync(&bad, c->counters + 5, 8, hipMemcpyDeviceToHost, s));
    HIPCHK(c, hipStreamSynchronize(s));
    if (bad) return fail(c, SDEH_E_INVALID, "order is not a permutation of 0..n_traj-1");
  }

  // the events' times are only read by synchronous calls, and each event is a barrier
  // packet of its own between the kernels of back-to-back solves
  const bool do_sync = host || sync;
  if (piped) {
    // p_shared and the saveat times went up on `s`; the kernels queue behind them
    r = run_host_pipeline(c, pl, io, s);
  } else {
    r = run_plan(c, pl, s, c->counters, do_sync);
  }
  if (r) return r;
  note_pending(c, s, false);
  unsigned long long cnt[6] = {0, 0, 0, 0, 0, 0};  // counters [1..6]
  if (do_sync) {  // counters are only read back by synchronous calls
    HIPCHK(c, sdeh_util_zero_u64(c->counters + 1, 4, s));
    HIPCHK(c, sdeh_util_count(a.naccept, a.nreject, a.retcode, n, c->counters + 1, s));
  }
  if (do_sync) HIPCHK(c, hipMemcpyAsync(cnt, c->counters + 1, sizeof cnt, hipMemcpyDeviceToHost, s));
  if (host && n > 0 && !piped) {
    auto down = [&](void* dst, const void* src, size_t b) {
      if (dst && b) (void)hipMemcpyAsync(dst, src, b, hipMemcpyDeviceToHost, s);
    };
    down(io->u_end, a.u_end, sz.u_end);
    down(io->t_end, a.t_end, sz.t_end);
    down(io->retcode, a.retcode, sz.i32);
    down(io->naccept, a.naccept, sz.i32);
    down(io->nreject, a.nreject, sz.i32);
    down(io->u_saveat, a.u_saveat, sz.u_saveat);
    if (pl.packed) {  // only the rows used travel back
      int64_t used = 0;
      HIPCHK(c, hipMemcpyAsync(&used, pl.pk_off + n, 8, hipMemcpyDeviceToHost, s));
      HIPCHK(c, hipStreamSynchronize(s));
      down(io->u_steps, a.u_steps, (size_t)used * pl.n_state * pl.es);
      down(io->t_steps, a.t_steps, (size_t)used * 8);
      down(io->steps_offset, pl.pk_off, sz.pk_off);
    } else {
      down(io->u_steps, a.u_steps, sz.u_steps);
      down(io->t_steps, a.t_steps, sz.t_steps);
    }
    down(io->n_steps, a.n_steps, pl.save == SAVE_STEPS ? sz.i32 : 0);
    HIPCHK(c, hipGetLastError());
  }
  c->stats = sdeh_stats{};
  c->stats.block = pl.shape.block;
  c->stats.grid = pl.shape.grid;
  c->stats.chunk = pl.shape.chunk;
  c->stats.schedule = pl.shape.schedule;
  c->stats.lanes = pl.k.lanes;
  c->stats.waves = pl.k.waves;
  c->stats.per_lane = pl.k.tpl;
  c->stats.refill = pl.shape.refill;
  if (do_sync) {
    if (piped) HIPCHK(c, hipStreamSynchronize(c->s_out));
    HIPCHK(c, hipStreamSynchronize(s));
    note_pending(c, s, true);
    float ms = 0.f;
    if (n > 0) HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
    c->stats.kernel_ms = ms;
    c->stats.attempts = (int64_t)cnt[0];
    c->stats.accepts = (int64_t)cnt[1];
    c->stats.steps_needed = pl.packed && n > 0 ? (int64_t)cnt[5] : 0;
    c->stats.total_ms =
        std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start)
            .count();
    if (cnt[2]) return fail(c, SDEH_E_DTMIN, "%llu trajectories stopped at dt < dtmin", cnt[2]);
    if (cnt[3] && pl.packed)
      return fail(c, SDEH_E_SAVE_OVERFLOW,
                  "%llu trajectories lost points: %llu points offered, steps_capacity %lld",
                  cnt[3], cnt[5], (long long)pl.pk_cap);
    if (cnt[3])
      return fail(c, SDEH_E_SAVE_OVERFLOW, "%llu trajectories had more than max_saves steps",
                  cnt[3]);
  }
  return SDEH_OK;
}

// The allocation-free solve (sdeh_solve_static): device buffers, endpoint or saveat
// output, one-launch or persistent schedule.  Its only scratch is the library's
// static device array: words 0..5 (queue counter, counts), then the saveat times.
// No arena, no hipMalloc: what would need per-ensemble scratch (span order, staged
// records, the permutation check of io->order, internal count arrays, packed
// save_everystep) is refused or left out.
int solve_static_impl(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, hipStream_t s,
                      int32_t sync) {
  const auto t_start = std::chrono::steady_clock::now();
  Plan pl;
  int r = plan_solve(c, d, io, &pl, Path::kStatic);
  if (r) return r;
  if (pl.save == SAVE_STEPS)
    return fail(c, SDEH_E_UNSUPPORTED,
                "the allocation-free solve writes endpoint or saveat output (set "
                "save_everystep = 0 or give saveat)");
  const int64_t max_saveat = sdeh_util_static_saveat_max();
  if (pl.save == SAVE_AT && d->n_saveat > max_saveat)
    return fail(c, SDEH_E_INVALID,
                "the allocation-free solve holds at most %lld saveat times (got %lld)",
                (long long)max_saveat, (long long)d->n_saveat);
  if (io->order)
    return fail(c, SDEH_E_UNSUPPORTED,
                "the allocation-free solve takes no order (its check needs per-trajectory "
                "scratch); use sdeh_solve");
  const int64_t n = d->n_traj;
  if (n > 0 && (!io->naccept || !io->nreject))
    return fail(c, SDEH_E_INVALID, "the allocation-free solve needs naccept and nreject buffers");
  // index order (the span order needs per-trajectory scratch); a staged shape runs
  // as the persistent launch
  pl.span = false;
  if (pl.staged || pl.shape.schedule == SDEH_SCHED_STAGED) {
    pl.staged = false;
    pl.shape.schedule = SDEH_SCHED_PERSISTENT;
  }
  const Sizes sz = sizes_of(d, io, pl);
  if (n > 0) {
    if (!io->u0 || !io->u_end || !io->t_end || !io->retcode)
      return fail(c, SDEH_E_INVALID, "u0, u_end, t_end and retcode are required");
    if (pl.n_param > 0 && !io->p) return fail(c, SDEH_E_INVALID, "p is required (n_param > 0)");
    if (pl.n_shared > 0 && !io->p_shared)
      return fail(c, SDEH_E_INVALID, "p_shared is required for this rhs");
    if (pl.save == SAVE_AT && !io->u_saveat)
      return fail(c, SDEH_E_INVALID, "u_saveat is required with saveat");
    r = check_dev(c, io->u0, sz.u0, "u0");
    if (!r) r = check_dev(c, io->p, sz.p, "p");
    if (!r) r = check_dev(c, io->p_shared, sz.ps, "p_shared");
    if (!r && io->tspan) r = check_dev(c, io->tspan, sz.tspan, "tspan");
    if (!r && io->dt0) r = check_dev(c, io->dt0, sz.dt0, "dt0");
    if (!r) r = check_dev(c, io->u_end, sz.u_end, "u_end");
    if (!r) r = check_dev(c, io->t_end, sz.t_end, "t_end");
    if (!r) r = check_dev(c, io->retcode, sz.i32, "retcode");
    if (!r) r = check_dev(c, io->naccept, sz.i32, "naccept");
    if (!r) r = check_dev(c, io->nreject, sz.i32, "nreject");
    if (!r && io->visits) r = check_dev(c, io->visits, sz.i32, "visits");
    if (!r && pl.save == SAVE_AT) r = check_dev(c, io->u_saveat, sz.u_saveat, "u_saveat");
    if (r) return r;
  }
  // this call's stream follows the context's earlier ones (their kernels may still
  // read the context's events and the static scratch)
  r = after_pending(c, s);
  if (r) return r;
  unsigned long long* const words = c->static_scratch;  // the device address, never the symbol
  double* const d_saveat = (double*)(words + 8);
  sdeh_kargs& a = pl.a;
  if (sz.saveat) HIPCHK(c, hipMemcpyAsync(d_saveat, d->saveat, sz.saveat, hipMemcpyHostToDevice, s));
  a.saveat = d_saveat;
  a.u0 = io->u0;
  a.p = io->p;
  a.ps = io->p_shared;
  a.tspan = io->tspan;
  a.dt0 = io->dt0;
  a.order = nullptr;
  a.u_end = io->u_end;
  a.t_end = io->t_end;
  a.retcode = io->retcode;
  a.naccept = io->naccept;
  a.nreject = io->nreject;
  a.u_saveat = io->u_saveat;
  a.visits = io->visits;
  r = run_plan(c, pl, s, words, sync != 0);  // run_plan clears the queue word before a persistent launch
  if (r) return r;
  note_pending(c, s, false);
  c->stats = sdeh_stats{};
  c->stats.block = pl.shape.block;
  c->stats.grid = pl.shape.grid;
  c->stats.chunk = pl.shape.chunk;
  c->stats.schedule = pl.shape.schedule;
  c->stats.lanes = pl.k.lanes;
  c->stats.waves = pl.k.waves;
  c->stats.per_lane = pl.k.tpl;
  c->stats.refill = pl.shape.refill;
  if (!sync) return SDEH_OK;
  unsigned long long cnt[4] = {0, 0, 0, 0};
  if (n > 0) {
    HIPCHK(c, sdeh_util_zero_u64(words + 1, 4, s));
    HIPCHK(c, sdeh_util_count(a.naccept, a.nreject, a.retcode, n, words + 1, s));
    HIPCHK(c, hipMemcpyAsync(cnt, words + 1, sizeof cnt, hipMemcpyDeviceToHost, s));
  }
  HIPCHK(c, hipStreamSynchronize(s));
  note_pending(c, s, true);
  float ms = 0.f;
  if (n > 0) HIPCHK(c, hipEventElapsedTime(&ms, c->ev0, c->ev1));
  c->stats.kernel_ms = ms;
  c->stats.attempts = (int64_t)cnt[0];
  c->stats.accepts = (int64_t)cnt[1];
  c->stats.total_ms =
      std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start).count();
  if (cnt[2]) return fail(c, SDEH_E_DTMIN, "%llu trajectories stopped at dt < dtmin", cnt[2]);
  return SDEH_OK;
}

}  // namespace

extern "C" {

void sdeh_desc_init(sdeh_solve_desc* d) {
  if (!d) return;
  memset(d, 0, sizeof *d);
  d->alg = SDEH_ALG_ATSIT5;
  d->dtype = SDEH_F64;
  d->rhs = SDEH_RHS_LORENZ;
  d->t0 = 0.0;
  d->tf = 1.0;
  d->dt = (double)0.1f;       // gpuatsit5.jl:208 dt = 0.1f0
  d->abstol = (double)1.0e-6f;  // gpuatsit5.jl:210 abstol = 1.0f-6
  d->reltol = (double)1.0e-3f;  // reltol = 1.0f-3
  d->save_everystep = 1;      // gpuatsit5.jl:209
  d->quirks = 1;
  d->schedule = SDEH_SCHED_AUTO;
  d->precision = SDEH_PREC_PLAIN;
}

int sdeh_abi_version(void) { return SDEH_ABI_VERSION; }

int sdeh_create(sdeh_ctx** out, int device) {
  if (!out) return SDEH_E_INVALID;
  *out = nullptr;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev == 0) return SDEH_E_HIP;
  if (device < 0 || device >= ndev) return SDEH_E_INVALID;
  sdeh_ctx* c = new sdeh_ctx;
  c->device = device;
  if (hipSetDevice(device) != hipSuccess ||
      hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&c->s_in, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&c->s_out, hipStreamNonBlocking) != hipSuccess ||
      hipStreamCreateWithFlags(&c->s_k2, hipStreamNonBlocking) != hipSuccess ||
      hipEventCreate(&c->ev0) != hipSuccess || hipEventCreate(&c->ev1) != hipSuccess ||
      hipMalloc((void**)&c->counters, 16 * sizeof(unsigned long long)) != hipSuccess) {
    sdeh_destroy(c);
    return SDEH_E_HIP;
  }
  for (hipEvent_t& e : c->ev_pipe)
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      sdeh_destroy(c);
      return SDEH_E_HIP;
    }
  if (hipEventCreateWithFlags(&c->ev_pipe_start, hipEventDisableTiming) != hipSuccess) {
    sdeh_destroy(c);
    return SDEH_E_HIP;
  }
  {
    void* q = nullptr;
    size_t b = 0;
    if (sdeh_util_static_scratch(&q, &b) != hipSuccess || !q) {
      sdeh_destroy(c);
      return SDEH_E_HIP;
    }
    c->static_scratch = (unsigned long long*)q;
    c->static_bytes = b;
  }
  hipDeviceProp_t prop;
  if (hipGetDeviceProperties(&prop, device) == hipSuccess) c->cus = prop.multiProcessorCount;
  if (c->cus <= 0) c->cus = 256;
  *out = c;
  return SDEH_OK;
}

void sdeh_destroy(sdeh_ctx* c) {
  if (!c) return;
  if (c->stream) (void)hipStreamSynchronize(c->stream);
  for (auto& g : c->graphs) {
    if (g.second.exec) (void)hipGraphExecDestroy(g.second.exec);
    if (g.second.graph) (void)hipGraphDestroy(g.second.graph);
    if (g.second.mem) (void)hipFree(g.second.mem);
  }
  for (auto& m : c->rtc) (void)hipModuleUnload(m.second.first);
  if (c->arena) (void)hipFree(c->arena);
  if (c->counters) (void)hipFree(c->counters);
  if (c->ev0) (void)hipEventDestroy(c->ev0);
  if (c->ev1) (void)hipEventDestroy(c->ev1);
  for (hipEvent_t e : c->ev_pipe)
    if (e) (void)hipEventDestroy(e);
  if (c->ev_pipe_start) (void)hipEventDestroy(c->ev_pipe_start);
  if (c->s_in) {
    (void)hipStreamSynchronize(c->s_in);
    (void)hipStreamDestroy(c->s_in);
  }
  if (c->s_out) {
    (void)hipStreamSynchronize(c->s_out);
    (void)hipStreamDestroy(c->s_out);
  }
  if (c->s_k2) {
    (void)hipStreamSynchronize(c->s_k2);
    (void)hipStreamDestroy(c->s_k2);
  }
  if (c->stream) (void)hipStreamDestroy(c->stream);
  delete c;
}

const char* sdeh_last_error(const sdeh_ctx* c) { return c ? c->err.c_str() : "null context"; }

int sdeh_rhs_info(sdeh_ctx* c, int64_t rhs, int32_t* n_state, int32_t* n_param,
                  int64_t* n_shared) {
  if (!c || !n_state || !n_param || !n_shared) return SDEH_E_INVALID;
  return rhs_shape(c, rhs, n_state, n_param, n_shared);
}

int sdeh_compile_rhs(sdeh_ctx* c, const char* src, const char* fn_name, int32_t n_state,
                     int32_t n_param, int64_t n_shared, int64_t* handle) {
  if (!c || !src || !fn_name || !handle) return SDEH_E_INVALID;
  if (n_state < 1 || n_state > 64 || n_param < 0 || n_param > 256 || n_shared < 0)
    return fail(c, SDEH_E_INVALID, "rhs shape out of range (1 <= n_state <= 64)");
  const size_t len = strlen(fn_name);
  bool ident = len > 0 && len <= 200 && !isdigit((unsigned char)fn_name[0]);
  for (const char* q = fn_name; *q && ident; ++q)
    ident = isalnum((unsigned char)*q) || *q == '_';
  if (!ident)
    return fail(c, SDEH_E_INVALID, "fn_name must be a C identifier of at most 200 characters");
  UserRhs u;
  u.src = src;
  u.fn = fn_name;
  u.n = n_state;
  u.p = n_param;
  u.s = n_shared;
  c->user.push_back(u);
  const int64_t h = kUserBase + (int64_t)c->user.size() - 1;
  // Compile the default kernel now so source errors surface at registration.
  KernelRef k;
  const int r = user_kernel(c, h, SDEH_ALG_ATSIT5, SDEH_F64, SAVE_END, 0, &k);
  if (r) {
    c->user.pop_back();
    return r;
  }
  *handle = h;
  return SDEH_OK;
}

int sdeh_solve(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, int32_t memory,
               void* stream, int32_t sync) {
  if (!c) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  return solve_impl(c, d, io, memory, stream ? (hipStream_t)stream : c->stream, sync);
}

int sdeh_solve_static(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, void* stream,
                      int32_t sync) {
  if (!c || !d || !io) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  return solve_static_impl(c, d, io, stream ? (hipStream_t)stream : c->stream, sync);
}

int sdeh_get_stats(const sdeh_ctx* c, sdeh_stats* out) {
  if (!c || !out) return SDEH_E_INVALID;
  *out = c->stats;
  return SDEH_OK;
}

int sdeh_synchronize(sdeh_ctx* c) {
  if (!c) return SDEH_E_INVALID;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  if (c->has_pending) HIPCHK(c, hipStreamSynchronize(c->pending));
  c->has_pending = false;
  return SDEH_OK;
}

int64_t sdeh_fixed_grid(double t0, double dt, double tf, double* elems, int64_t cap) {
  if (dt == 0.0) return -1;
  const sdeh_range::Grid g = sdeh_range::make(t0, dt, tf);
  if (elems)
    for (int64_t i = 0; i < std::min(cap, g.len); ++i) elems[i] = sdeh_range::elem(g, i);
  return g.len;
}

int sdeh_graph_capture(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io,
                       int64_t* graph_handle) {
  if (!c || !graph_handle) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  Plan pl;
  int r = plan_solve(c, d, io, &pl, Path::kGraph);
  if (r) return r;
  if (io->order) return fail(c, SDEH_E_UNSUPPORTED, "graph capture takes no order permutation");
  if (pl.staged) {  // a captured solve runs the staged shape as its persistent launch
    pl.staged = false;
    pl.shape.schedule = SDEH_SCHED_PERSISTENT;
  }
  if (pl.packed)
    return fail(c, SDEH_E_UNSUPPORTED, "graph capture of the packed save layout is not built");
  const Sizes sz = sizes_of(d, io, pl);
  const int64_t n = d->n_traj;
  r = check_dev(c, io->u0, sz.u0, "u0");
  if (!r) r = check_dev(c, io->p, sz.p, "p");
  if (!r) r = check_dev(c, io->p_shared, sz.ps, "p_shared");
  if (!r && io->tspan) r = check_dev(c, io->tspan, sz.tspan, "tspan");
  if (!r && io->dt0) r = check_dev(c, io->dt0, sz.dt0, "dt0");
  if (!r) r = check_dev(c, io->u_end, sz.u_end, "u_end");
  if (!r) r = check_dev(c, io->t_end, sz.t_end, "t_end");
  if (!r) r = check_dev(c, io->retcode, sz.i32, "retcode");
  if (!r) r = check_dev(c, io->naccept, sz.i32, "naccept");
  if (!r) r = check_dev(c, io->nreject, sz.i32, "nreject");
  if (!r && pl.save == SAVE_AT) r = check_dev(c, io->u_saveat, sz.u_saveat, "u_saveat");
  if (!r && pl.save == SAVE_STEPS) {
    r = check_dev(c, io->u_steps, sz.u_steps, "u_steps");
    if (!r) r = check_dev(c, io->t_steps, sz.t_steps, "t_steps");
    if (!r) r = check_dev(c, io->n_steps, sz.i32, "n_steps");
  }
  if (!r && io->visits) r = check_dev(c, io->visits, sz.i32, "visits");
  if (r) return r;
  if (n == 0) return fail(c, SDEH_E_INVALID, "empty ensemble");
  GraphRec g;
  HIPCHK(c, hipMalloc(&g.mem, 256 + round256(sz.saveat) + round256(sz.span_order) +
                                  round256(sz.span_hist)));
  double* d_saveat = (double*)((char*)g.mem + 256);
  if (sz.saveat) {
    HIPCHK(c, hipMemcpy(d_saveat, d->saveat, sz.saveat, hipMemcpyHostToDevice));
  }
  sdeh_kargs& a = pl.a;
  a.saveat = d_saveat;
  a.u0 = io->u0;
  a.p = io->p;
  a.ps = io->p_shared;
  a.tspan = io->tspan;
  a.dt0 = io->dt0;
  a.order = nullptr;
  a.u_end = io->u_end;
  a.t_end = io->t_end;
  a.retcode = io->retcode;
  a.naccept = io->naccept;
  a.nreject = io->nreject;
  a.u_saveat = io->u_saveat;
  a.u_steps = io->u_steps;
  a.t_steps = io->t_steps;
  a.n_steps = io->n_steps;
  a.visits = io->visits;
  HIPCHK(c, hipStreamSynchronize(c->stream));
  HIPCHK(c, hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
  if (pl.span) {  // the hand-out order is recomputed on every replay
    char* q = (char*)g.mem + 256 + round256(sz.saveat);
    pl.span_ord = (int64_t*)q;
    pl.span_hist[0] = (unsigned*)(q + round256(sz.span_order));
    a.order = pl.span_ord;
  }
  r = pl.span ? (sdeh_util_span_order(a.tspan, n, pl.span_hist[0], pl.span_ord, c->stream) ==
                         hipSuccess
                     ? SDEH_OK
                     : fail(c, SDEH_E_HIP, "span order launch failed"))
              : SDEH_OK;
  if (!r) r = run_plan(c, pl, c->stream, (unsigned long long*)g.mem, false);
  hipGraph_t graph = nullptr;
  const hipError_t e = hipStreamEndCapture(c->stream, &graph);
  if (r) {
    if (graph) (void)hipGraphDestroy(graph);
    (void)hipFree(g.mem);
    return r;
  }
  if (e != hipSuccess) {
    (void)hipFree(g.mem);
    return fail(c, SDEH_E_HIP, "hipStreamEndCapture: %s", hipGetErrorString(e));
  }
  g.graph = graph;
  if (hipGraphInstantiate(&g.exec, graph, nullptr, nullptr, 0) != hipSuccess) {
    (void)hipGraphDestroy(graph);
    (void)hipFree(g.mem);
    return fail(c, SDEH_E_HIP, "hipGraphInstantiate failed");
  }
  const int64_t h = c->next_graph++;
  c->graphs[h] = g;
  *graph_handle = h;
  return SDEH_OK;
}

int sdeh_graph_launch(sdeh_ctx* c, int64_t h, void* stream) {
  if (!c) return SDEH_E_INVALID;
  auto it = c->graphs.find(h);
  if (it == c->graphs.end()) return fail(c, SDEH_E_INVALID, "unknown graph %lld", (long long)h);
  HIPCHK(c, hipGraphLaunch(it->second.exec, stream ? (hipStream_t)stream : c->stream));
  return SDEH_OK;
}

int sdeh_graph_destroy(sdeh_ctx* c, int64_t h) {
  if (!c) return SDEH_E_INVALID;
  auto it = c->graphs.find(h);
  if (it == c->graphs.end()) return fail(c, SDEH_E_INVALID, "unknown graph %lld", (long long)h);
  HIPCHK(c, hipStreamSynchronize(c->stream));
  (void)hipGraphExecDestroy(it->second.exec);
  (void)hipGraphDestroy(it->second.graph);
  (void)hipFree(it->second.mem);
  c->graphs.erase(it);
  return SDEH_OK;
}

int sdeh_autotune(sdeh_ctx* c, const sdeh_solve_desc* d, const sdeh_io* io, sdeh_stats* best) {
  if (!c || !d || !io) return SDEH_E_INVALID;
  if (!is_adaptive(d->alg))
    return fail(c, SDEH_E_INVALID, "autotune applies to the adaptive solvers");
  HIPCHK(c, hipSetDevice(c->device));
  struct Cand {
    int sched, block, chunk, occ_div;
  };
  std::vector<Cand> cands;
  for (int b : {64, 128, 256}) cands.push_back({SDEH_SCHED_ONE_LAUNCH, b, 0, 1});
  for (int b : {64, 128, 256})
    for (int ch : {16, 64, 256}) cands.push_back({SDEH_SCHED_PERSISTENT, b, ch, 1});
  for (int ch : {64}) cands.push_back({SDEH_SCHED_PERSISTENT, 256, ch, 2});
  for (int ch : {16, 64}) cands.push_back({SDEH_SCHED_STAGED, 256, ch, 1});
  double best_ms = 1e300;
  Shape best_shape;
  sdeh_stats best_stats{};
  TuneKey key;
  // The layout is resolved once, from the caller's descriptor: every candidate runs on it, and
  // so does the solve that takes the winner (its schedule is not the candidate's, and lanes = 0
  // may stand for another layout there).
  sdeh_solve_desc base_desc = *d;
  {  // the shape search runs the caller's kernel choice, not an earlier tuning's
    Plan pl;
    int r = plan_solve(c, d, io, &pl);
    if (r) return r;
    key = TuneKey(d->rhs, d->alg, d->dtype, pl.save, pl.kahan, pl.k.lanes, pl.packed);
    c->tuned.erase(key);
    base_desc.lanes = pl.k.lanes;
  }
  d = &base_desc;
  for (const Cand& k : cands) {
    sdeh_solve_desc dd = *d;
    dd.schedule = k.sched;
    dd.block = k.block;
    dd.chunk = k.chunk;
    dd.grid = 0;
    if (k.sched != SDEH_SCHED_ONE_LAUNCH) {
      Plan pl;
      int r = plan_solve(c, &dd, io, &pl);
      if (r) return r;
      if (pl.shape.schedule != k.sched) continue;  // staged does not apply to this solve
      dd.grid = std::max(1, pl.shape.grid / k.occ_div);
    }
    double ms = 1e300;
    for (int rep = 0; rep < 2; ++rep) {  // first run warms caches and modules
      int r = sdeh_solve(c, &dd, io, SDEH_MEM_DEVICE, nullptr, 1);
      if (r && r != SDEH_E_DTMIN) return r;
      ms = c->stats.kernel_ms;
    }
    if (ms < best_ms) {
      best_ms = ms;
      best_shape.schedule = k.sched;
      best_shape.block = k.block;
      best_shape.chunk = c->stats.chunk;
      best_shape.grid = c->stats.grid;
      best_shape.waves = c->stats.waves;
      best_shape.per_lane = c->stats.per_lane;
      best_shape.refill = c->stats.refill;
      best_stats = c->stats;
    }
  }
  // Then the register cap: the best shape's schedule, block and chunk with each
  // register-cap variant built for this solve (its own resident grid).
  if (!d->waves) {
    const Shape base = best_shape;
    for (int w : kWaveVariants) {
      sdeh_solve_desc dd = *d;
      dd.schedule = base.schedule;
      dd.block = base.block;
      dd.chunk = base.chunk;
      dd.grid = 0;
      dd.waves = w;
      Plan pl;
      int r = plan_solve(c, &dd, io, &pl);
      if (r == SDEH_E_UNSUPPORTED) continue;  // no such variant for this solve
      if (r) return r;
      double ms = 1e300;
      for (int rep = 0; rep < 2; ++rep) {
        r = sdeh_solve(c, &dd, io, SDEH_MEM_DEVICE, nullptr, 1);
        if (r && r != SDEH_E_DTMIN) return r;
        ms = c->stats.kernel_ms;
      }
      if (ms < best_ms) {
        best_ms = ms;
        best_shape = base;
        best_shape.grid = c->stats.grid;
        best_shape.waves = w;
        best_shape.refill = c->stats.refill;
        best_stats = c->stats;
      }
    }
  }
  // Then the refill batch of a persistent or staged shape with one lane per
  // trajectory: claim for each free slot, or for batches of 4 or 8.
  if (!d->refill && best_shape.schedule != SDEH_SCHED_ONE_LAUNCH && best_shape.per_lane == 1 &&
      best_stats.lanes == 1) {
    const Shape base = best_shape;
    for (int rf : {1, 4, 8}) {
      if (rf == base.refill) continue;  // the shape search ran this one
      sdeh_solve_desc dd = *d;
      dd.schedule = base.schedule;
      dd.block = base.block;
      dd.chunk = base.chunk;
      dd.grid = base.grid;
      dd.waves = base.waves;
      dd.refill = rf;
      double ms = 1e300;
      for (int rep = 0; rep < 2; ++rep) {
        int r = sdeh_solve(c, &dd, io, SDEH_MEM_DEVICE, nullptr, 1);
        if (r && r != SDEH_E_DTMIN) return r;
        ms = c->stats.kernel_ms;
      }
      if (ms < best_ms) {
        best_ms = ms;
        best_shape = base;
        best_shape.refill = rf;
        best_stats = c->stats;
      }
    }
  }
  // And two trajectories per lane, one launch and persistent, where built.
  if (!d->waves && !d->per_lane) {
    struct Multi {
      int sched, block, chunk;
    };
    const Multi mc[] = {{SDEH_SCHED_ONE_LAUNCH, 64, 0},   {SDEH_SCHED_ONE_LAUNCH, 128, 0},
                        {SDEH_SCHED_ONE_LAUNCH, 256, 0},  {SDEH_SCHED_PERSISTENT, 128, 64},
                        {SDEH_SCHED_PERSISTENT, 256, 64}, {SDEH_SCHED_PERSISTENT, 256, 16}};
    for (const Multi& k : mc) {
      sdeh_solve_desc dd = *d;
      dd.schedule = k.sched;
      dd.block = k.block;
      dd.chunk = k.chunk;
      dd.grid = 0;
      dd.per_lane = 2;
      Plan pl;
      int r = plan_solve(c, &dd, io, &pl);
      if (r == SDEH_E_UNSUPPORTED) break;  // no such variant for this solve
      if (r) return r;
      double ms = 1e300;
      for (int rep = 0; rep < 2; ++rep) {
        r = sdeh_solve(c, &dd, io, SDEH_MEM_DEVICE, nullptr, 1);
        if (r && r != SDEH_E_DTMIN) return r;
        ms = c->stats.kernel_ms;
      }
      if (ms < best_ms) {
        best_ms = ms;
        best_shape = Shape{};
        best_shape.schedule = k.sched;
        best_shape.block = k.block;
        best_shape.chunk = c->stats.chunk;
        best_shape.grid = c->stats.grid;
        best_shape.per_lane = 2;
        best_stats = c->stats;
      }
    }
  }
  // Packed output: the ranked passes, which no schedule names, where they are open to this solve.
  if (!d->grid && !d->chunk && !d->refill) {
    sdeh_solve_desc dd = *d;
    dd.schedule = SDEH_SCHED_AUTO;
    dd.block = 0;
    Plan pl;
    int r = plan_solve(c, &dd, io, &pl);
    if (r) return r;
    if (pl.pk_ranked) {
      double ms = 1e300;
      for (int rep = 0; rep < 2; ++rep) {
        r = sdeh_solve(c, &dd, io, SDEH_MEM_DEVICE, nullptr, 1);
        if (r && r != SDEH_E_DTMIN) return r;
        ms = c->stats.kernel_ms;
      }
      best_shape.ranked = ms < best_ms ? 1 : 0;
      if (best_shape.ranked) best_stats = c->stats;
    }
  }
  c->err.clear();
  c->tuned[key] = best_shape;
  if (best) *best = best_stats;
  return SDEH_OK;
}

int sdeh_mlp_forward(sdeh_ctx* c, const float* params, const float* x, float* y, int64_t n,
                     void* stream) {
  if (!c || !params || !x || !y || n < 0) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  int r = check_dev(c, params, SDEH_MLP_NPARAM * 4, "params");
  if (!r) r = check_dev(c, x, (size_t)n * SDEH_MLP_NIN * 4, "x");
  if (!r) r = check_dev(c, y, (size_t)n * SDEH_MLP_NOUT * 4, "y");
  if (r) return r;
  r = sdeh_mlp_forward_impl(params, x, y, n, stream ? (hipStream_t)stream : c->stream);
  if (r) return fail(c, r, "mlp forward launch failed");
  return SDEH_OK;
}

int sdeh_mlp_plan_lorenz(sdeh_ctx* c, const float* params, const double* p, const double* u0,
                         const double* tspan, int64_t n, const double* feat, const float* y_norm,
                         float* key, double* dt0, float* pred, void* stream) {
  if (!c || !params || !p || !u0 || !tspan || !feat || !y_norm || !key || !dt0 || n < 0)
    return SDEH_E_INVALID;
  for (int k = 0; k < 8; k += 2)
    if (!(feat[k + 1] != 0.0)) return fail(c, SDEH_E_INVALID, "feature scale %d is zero", k / 2);
  HIPCHK(c, hipSetDevice(c->device));
  int r = check_dev(c, params, SDEH_MLP_NPARAM * 4, "params");
  if (!r) r = check_dev(c, p, (size_t)n * 3 * 8, "p");
  if (!r) r = check_dev(c, u0, (size_t)n * 3 * 8, "u0");
  if (!r) r = check_dev(c, tspan, (size_t)n * 2 * 8, "tspan");
  if (!r) r = check_dev(c, key, (size_t)n * 4, "key");
  if (!r) r = check_dev(c, dt0, (size_t)n * 8, "dt0");
  if (!r && pred) r = check_dev(c, pred, (size_t)n * SDEH_MLP_NOUT * 4, "pred");
  if (r) return r;
  r = sdeh_mlp_plan_lorenz_impl(params, p, u0, tspan, n, feat, y_norm[0], y_norm[1], y_norm[2],
                                y_norm[3], key, dt0, pred,
                                stream ? (hipStream_t)stream : c->stream);
  if (r) return fail(c, r, "mlp plan launch failed");
  return SDEH_OK;
}

int sdeh_plan_order(sdeh_ctx* c, const float* key, int64_t n, int64_t* order, void* stream) {
  if (!c || !key || !order || n < 0) return SDEH_E_INVALID;
  if (n >= (1ll << 32)) return fail(c, SDEH_E_INVALID, "n must be below 2^32");
  if (n == 0) return SDEH_OK;
  HIPCHK(c, hipSetDevice(c->device));
  int r = check_dev(c, key, (size_t)n * 4, "key");
  if (!r) r = check_dev(c, order, (size_t)n * 8, "order");
  if (r) return r;
  // the bucket counts live in the arena, which an earlier call may still be using
  const hipStream_t s = stream ? (hipStream_t)stream : c->stream;
  r = after_pending(c, s);
  if (!r) r = ensure_arena(c, sdeh_util_span_scratch_bytes());
  if (r) return r;
  c->planned_order = nullptr;
  HIPCHK(c, sdeh_util_logkey_order(key, n, (unsigned*)c->arena, order, s));
  note_pending(c, s, false);
  c->planned_order = order;
  c->planned_n = n;
  return SDEH_OK;
}

int sdeh_mlp_loss_grad(sdeh_ctx* c, const float* params, const float* x, const float* y,
                       int64_t n, float* loss, float* grad, void* stream) {
  if (!c || !params || !x || !y || !loss || !grad || n < 1) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  int r = check_dev(c, params, SDEH_MLP_NPARAM * 4, "params");
  if (!r) r = check_dev(c, x, (size_t)n * SDEH_MLP_NIN * 4, "x");
  if (!r) r = check_dev(c, y, (size_t)n * SDEH_MLP_NOUT * 4, "y");
  if (!r) r = check_dev(c, loss, 4, "loss");
  if (!r) r = check_dev(c, grad, SDEH_MLP_NPARAM * 4, "grad");
  if (r) return r;
  // scratch for per-block partial gradients lives in the arena; its size comes
  // from the MLP unit, which owns the launch shape
  const hipStream_t s = stream ? (hipStream_t)stream : c->stream;
  r = after_pending(c, s);
  if (!r) r = ensure_arena(c, sdeh_mlp_grad_scratch_bytes(n));
  if (r) return r;
  r = sdeh_mlp_loss_grad_impl(params, x, y, n, loss, grad, (float*)c->arena, s);
  note_pending(c, s, false);
  if (r) return fail(c, r, "mlp loss/grad launch failed");
  return SDEH_OK;
}

int sdeh_mlp_adam(sdeh_ctx* c, float* params, const float* grad, float* m, float* v, float lr,
                  float beta1, float beta2, float eps, int32_t t, void* stream) {
  if (!c || !params || !grad || !m || !v || t < 1) return SDEH_E_INVALID;
  HIPCHK(c, hipSetDevice(c->device));
  int r = check_dev(c, params, SDEH_MLP_NPARAM * 4, "params");
  if (!r) r = check_dev(c, grad, SDEH_MLP_NPARAM * 4, "grad");
  if (!r) r = check_dev(c, m, SDEH_MLP_NPARAM * 4, "m");
  if (!r) r = check_dev(c, v, SDEH_MLP_NPARAM * 4, "v");
  if (r) return r;
  r = sdeh_mlp_adam_impl(params, grad, m, v, lr, beta1, beta2, eps, t,
                         stream ? (hipStream_t)stream : c->stream);
  if (r) return fail(c, r, "mlp adam launch failed");
  return SDEH_OK;
}

}  // extern "C"
