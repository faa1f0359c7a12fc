// rkx host runtime: the C ABI of include/rkx.h over HIP.
//
// The step loop of the reference's solver() (src/impl/seq/D.c:58-78) runs on
// the device: every step's kernels read t, h and the current-buffer index from
// a device-resident state, and the step control (accept/reject and the next
// h) runs on the device as well.  The host follows t, h and the counts in
// pinned memory and keeps a few steps launched ahead, long solves from a graph
// captured while the first steps run (run_steps); launches past the end of the
// integration return at once.
#include "rkx_internal.hpp"

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <atomic>
#include <mutex>
#include <thread>
#include <string>
#include <vector>

namespace rkx {

namespace {
thread_local std::string g_last_error;
}

int fail(int code, const std::string &msg)
{
  g_last_error = msg;
  return code;
}

dev_ode make_dev_ode(const rkx_ode &p)
{
  dev_ode d{};
  d.kind = p.kind;
  d.n = p.n;
  d.cells = p.n / 2;
  d.N = (p.kind == RKX_BRUSS2D) ? p.grid : 0;
  if (p.kind == RKX_BRUSS2D) {
    const double N1 = static_cast<double>(p.grid) - 1.0;
    d.coef = p.alpha * N1 * N1;   // ((alpha*N1)*N1), bruss2d-mix.c:77
  }
  d.c0 = p.c0;
  d.d0 = p.d0;
  d.d1 = p.d1;
  d.c1 = p.c1;
  d.diff = p.diff;
  return d;
}

namespace {
hipStream_t g_stream = nullptr;
std::mutex g_init_mu;
}  // namespace

int default_stream(hipStream_t *out)
{
  std::lock_guard<std::mutex> lk(g_init_mu);
  if (!g_stream) {
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
      return fail(RKX_EDEVICE, "no HIP device available");
    RKX_HIP(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
  }
  *out = g_stream;
  return RKX_OK;
}

int check_ode(const rkx_ode *p)
{
  if (!p)
    return fail(RKX_EINVAL, "null problem descriptor");
  switch (p->kind) {
  case RKX_BRUSS2D:
    if (p->grid < 2 || p->n != 2 * p->grid * p->grid)
      return fail(RKX_EINVAL, "BRUSS2D needs N >= 2 and n = 2*N*N");
    if (p->grid > 32767)
      return fail(RKX_ELIMIT, "BRUSS2D grid above 32767 (n = 2N^2 must fit in int)");
    break;
  case RKX_LV:
    if (p->grid < 1 || p->n != 2 * p->grid)
      return fail(RKX_EINVAL, "LV needs pairs >= 1 and n = 2*pairs");
    break;
  case RKX_LV_CHAIN:
    if (p->grid < 3 || p->n != 2 * p->grid)
      return fail(RKX_EINVAL, "LV chain needs cells >= 3 and n = 2*cells");
    break;
  default:
    return fail(RKX_EINVAL, "unknown problem kind");
  }
  return RKX_OK;
}

int check_method(const rkx_method *m)
{
  if (!m || m->s < 2 || m->s > RKX_MAX_STAGES)
    return fail(RKX_EINVAL, "method needs 2 <= s <= 16 stages");
  for (int i = 0; i < m->s; ++i)
    for (int j = i; j < m->s; ++j)
      if (m->A[i][j] != 0.0)
        return fail(RKX_EINVAL, "method is not explicit (A[i][j] != 0 for j >= i)");
  return RKX_OK;
}

void fill_dev_method(const rkx_method &m, dev_method &d)
{
  std::memset(&d, 0, sizeof(d));
  for (int i = 0; i < m.s; ++i) {
    for (int j = 0; j < i; ++j)
      d.A[i * RKX_MAX_STAGES + j] = m.A[i][j];
    d.b[i] = m.b[i];
    d.e[i] = m.b[i] - m.b_hat[i];      // seq/D.c:40-41
    d.c[i] = m.c[i];
  }
  for (int i = 0; i < m.s; ++i) {
    for (int l = i + 1; l < m.s; ++l)
      d.col[i][l - i - 1] = d.A[l * RKX_MAX_STAGES + i];
    d.col[i][m.s - i - 1] = d.b[i];
    d.col[i][m.s - i] = d.e[i];
  }
}

// initial_stepsize (src/tools.c:25-36)
double initial_h(double H, double tol, int limit, double h0)
{
  if (h0 > 0.0)
    return h0;
  return tol > 0.0 ? std::fmin(10.0 * tol, H / static_cast<double>(limit))
                   : H / static_cast<double>(limit);
}

namespace {

struct graph_holder {
  hipGraph_t g = nullptr;
  hipGraphExec_t ge = nullptr;
  ~graph_holder()
  {
    if (ge)
      (void) hipGraphExecDestroy(ge);
    if (g)
      (void) hipGraphDestroy(g);
  }
};

// What the launches of one solve use: its device memory, returned to the pool
// on scope exit, its view and its step graph.  All of it outlives the work on
// the solve's stream (if any), which goes on behind the loop's last attempt.
struct solve_mem {
  // Pinned: the view, and what the host's step control passes to and fro.
  struct pinned {
    host_view view;
    step_slot slot;
    err_line err[kErrLines];
    state st;
    dev_coef coef;
  };
  struct held {
    void *p;
    size_t bytes;
  };
  std::vector<held> blocks;
  hipStream_t stream = nullptr;
  pinned *host = nullptr;
  graph_holder steps;                // destroyed after the wait below
  ~solve_mem()
  {
    const bool ok = !stream || hipStreamSynchronize(stream) == hipSuccess;
    for (const held &b : blocks) {
      if (ok)
        pool_give(b.p, b.bytes);
      else
        (void) hipFree(b.p);
    }
    if (host)
      give_pinned(host, ok);
  }
  int alloc(void **out, size_t bytes)
  {
    held b{};
    if (int rc = pool_take(&b.p, bytes, &b.bytes))
      return rc;
    blocks.push_back(b);
    *out = b.p;
    return RKX_OK;
  }
  // Up to kPinned of these (8 KB each) are kept.
  static constexpr size_t kPinned = 64;
  static std::mutex &pinned_mu()
  {
    static std::mutex *m = new std::mutex;
    return *m;
  }
  static std::vector<pinned *> &pinned_kept()
  {
    static auto *v = new std::vector<pinned *>;
    return *v;
  }
  int take_pinned()
  {
    {
      std::lock_guard<std::mutex> lk(pinned_mu());
      if (!pinned_kept().empty()) {
        host = pinned_kept().back();
        pinned_kept().pop_back();
      }
    }
    // coherent: the host reads the view while kernels write it
    if (!host)
      RKX_HIP(hipHostMalloc(reinterpret_cast<void **>(&host), sizeof(pinned),
                            hipHostMallocPortable | hipHostMallocMapped | hipHostMallocCoherent));
    return RKX_OK;
  }
  static void release_pinned()
  {
    std::vector<pinned *> drop;
    {
      std::lock_guard<std::mutex> lk(pinned_mu());
      drop.swap(pinned_kept());
    }
    for (pinned *w : drop)
      (void) hipHostFree(w);
  }
  static void give_pinned(pinned *w, bool ok)
  {
    std::lock_guard<std::mutex> lk(pinned_mu());
    if (ok && pinned_kept().size() < kPinned)
      pinned_kept().push_back(w);
    else
      (void) hipHostFree(w);
  }
};

}  // namespace

// The step control on the host: ctrl_decide/ctrl_finish with the C library's pow.
void host_finish(step_vars &v, double err)
{
  double px = 0.0, py = 0.0;
  const bool need = ctrl_decide(v, err, px, py);
  ctrl_finish(v, need, need ? std::pow(px, py) : 0.0);
}

step_ring make_ring(const step_vars &v, bool traced)
{
  step_ring g{};
  g.slot[0].v = v;
  g.slot[0].traced = traced;
  return g;
}

hipError_t fused_plan::launch(int r, hipStream_t stream)
{
  switch (kind) {
  case kPairs:
    return launch_lv_step(dp, s, ref, coef, y0, y1, r, stream);
  case kChain:
    chain.r = r;
    return launch_chain(pattern, shape, chain, stream);
  case kTile:
    return launch_tile_step(pattern, shape, tile, r, stream);
  case kGroups:
    groups.r = r;
    return launch_groups(form, groups, nz, stream);
  default:
    sweep.r = r;
    return launch_sweep(pattern, waves, general, sweep, stream);
  }
}

namespace {
// Attempts a launch of one workgroup makes: its start and end (4 us) are
// spread over them, and a launch is short enough for the host to follow.
constexpr int kRunSteps = 32;
}  // namespace

hipError_t fused_plan::launch_many(int r, hipStream_t stream)
{
  return launch_run(pattern, run, r, many, stream);
}

int make_fused_plan(const rkx_ode &p, const rkx_method &m, int rows, int waves,
                    const step_refs &ref, dev_coef *coef, double *y0, double *y1, fused_plan *out)
{
  fused_plan f;
  f.dp = make_dev_ode(p);
  f.ref = ref;
  f.coef = coef;
  f.y0 = y0;
  f.y1 = y1;
  f.s = m.s;
  f.pattern = sweep_pattern(m);
  if (chain_supported(f.dp, m)) {
    f.kind = fused_plan::kChain;
    f.shape = chain_default_cells(f.dp, m);
    f.chain.one = make_chain_inst(f.dp, m, f.shape, ref, y0, y1);
    f.chain.ntiles = f.chain.one.nwg;
  } else if (pairs_supported(f.dp, m)) {
    f.kind = fused_plan::kPairs;
  } else {
    // the tile kernel moves a cell's (u, v) in one 16-byte access: a caller's
    // buffer that is not aligned for it stays with the row sweep
    const bool aligned = ((reinterpret_cast<uintptr_t>(y0) | reinterpret_cast<uintptr_t>(y1)) &
                          15u) == 0;
    const bool free_tile = rows <= 0 && waves <= 0 && aligned;
    f.shape = free_tile ? tile_default_shape(f.dp, m) : -1;
    if (free_tile && run_supported(f.pattern, f.dp.N)) {
      f.many = kRunSteps;
      f.run.N = f.dp.N;
      f.run.coef = f.dp.coef;
      f.run.y0 = y0;
      f.run.y1 = y1;
      f.run.ref = ref;
    }
    if (f.shape >= 0) {
      f.kind = fused_plan::kTile;
      f.tile = make_tile_inst(f.dp, m, f.shape, ref, y0, y1);
    } else {
      sweep_cfg cfg = sweep_default_cfg(f.dp, m);
      if (rows > 0)
        cfg.rows = rows;
      if (waves > 0)
        cfg.waves = waves;
      if (cfg.waves < 1 || cfg.waves > 4 || cfg.rows < 1 || 64 * cfg.waves <= 2 * m.s)
        return fail(RKX_EINVAL, "tile_waves must be 1..4 (and wider than 2s), tile_rows >= 1");
      if (sweep_resident_blocks(f.pattern, cfg.waves) < 1)
        return fail(RKX_EINVAL, "tile_waves wider than this table's fused kernel "
                                "(DOPRI87: at most 2)");
      f.kind = fused_plan::kSweep;
      f.waves = cfg.waves;
      f.sweep.one = make_sweep_inst(f.dp, m, cfg, ref, y0, y1);
      f.sweep.ntiles = f.sweep.one.ntiles;
      f.general = !sweep_inst_single_reflect(f.pattern, m.s, f.sweep.one);
    }
  }
  *out = f;
  return RKX_OK;
}

// The control block of a solve: everything small that its kernels read, in
// one allocation and one copy.
struct solve_ctl {
  state st;
  step_ring ring;
  dev_method meth;
  dev_coef coef;
};

// DUMP output (include/tools.h:239-256): one line per attempted step, t and
// h then every component of the step's new y, "%.20e" separated by tabs.  The
// reference creates the file at the first attempt and appends afterwards.
struct dump_file {
  FILE *f = nullptr;
  ~dump_file()
  {
    if (f)
      std::fclose(f);
  }
  int append(const char *path, double t, double h, const std::vector<double> &y)
  {
    if (!f && !(f = std::fopen(path, "w")))
      return fail(RKX_EINVAL, std::string("rkx_solve: cannot open dump file ") + path);
    std::fprintf(f, "%.20e\t%.20e", t, h);
    for (double v : y)
      std::fprintf(f, "\t%.20e", v);
    std::fputc('\n', f);
    if (std::ferror(f))
      return fail(RKX_EINVAL, std::string("rkx_solve: write to dump file failed: ") + path);
    return RKX_OK;
  }
};

}  // namespace rkx

using namespace rkx;

namespace {

// Keeps the GPU supplied with steps until the device's step control ends the
// loop.  Steps past the end return at once but still cost a launch each, so
// the host follows the solve through its view and launches no more than it
// expects: the steps left at the current step size (most are limited by
// stability and change little) or to the step limit, and the one launch whose
// control ends the loop.  Long solves replay a graph of 32 kernels or more (1.7 us
// of launch a step, 2.6 us launched one by one), captured while the first
// steps run; it takes 85 us, so short solves do without.  The caller keeps the
// graph (gh) until the stream is done: replays are still queued when the view
// shows the end.
//
// enqueue(r, report): the last of the steps launched together reports the state
// it starts from, and in a graph every fourth does.
//
// per_step: kernels of a step.  The graph then has fewer steps and pays after
// fewer (chain of 100 cells, 13 stages, 27 kernels a step: 60 attempts 5907 us
// launched one by one, 5049 from graphs).
//
// many > 0: a launch makes up to that many attempts (and none pending: the
// host sees the state after the last of them).  Two launches are kept in
// flight then, the second covering the host's reaction to the first.
template <class STEP>
int run_steps(STEP &&enqueue, int per_step, int many, const host_view &view, double te,
              int step_limit, graph_holder &gh, hipStream_t stream)
{
  constexpr int kLow = 12;            // steps in flight below which more are launched
  constexpr int kGraphFrom = 160;     // expected kernels worth a graph
  // steps of the graph, and launched at a time without it
  const int chunk = std::max(32 / per_step / kRing, 1) * kRing;
  const int group = std::max(8 / per_step, kRing / 2);
  const volatile host_view &w = view;
  long long launched = 0;
  auto capture = [&]() -> int {
    RKX_HIP(hipStreamBeginCapture(stream, hipStreamCaptureModeThreadLocal));
    hipError_t cap = hipSuccess;
    for (int k = 0; k < chunk && cap == hipSuccess; ++k)
      cap = enqueue(k & (kRing - 1), (k & 3) == 3);
    const hipError_t end = hipStreamEndCapture(stream, &gh.g);
    if (cap != hipSuccess)
      return fail(RKX_EDEVICE, std::string("kernel launch during capture failed: ") +
                                   hipGetErrorString(cap));
    RKX_HIP(end);
    RKX_HIP(hipGraphInstantiate(&gh.ge, gh.g, nullptr, nullptr, 0));
    return RKX_OK;
  };
  for (unsigned spin = 1;; ++spin) {
    if (__atomic_load_n(&view.done, __ATOMIC_ACQUIRE))
      return RKX_OK;
    const long long made = static_cast<long long>(w.acc) + w.rej;
    const double t = w.t, h = w.h;
    double left = std::ceil((te - t) / h);
    if (!(left >= 1.0))
      left = 1.0;
    if (step_limit > 0)
      left = std::fmin(left, static_cast<double>(step_limit) - static_cast<double>(made));
    const double want = std::fmin(left + 1.0, 1e9) - static_cast<double>(launched - made);
    if (many > 0) {
      if (want >= 1.0 && launched - made <= many) {
        RKX_HIP(enqueue(static_cast<int>(launched / many) & (kRing - 1), true));
        launched += many;
        spin = 0;
        continue;
      }
    } else if (want >= 1.0 && launched - made < kLow) {
      const bool chunks = want >= chunk && launched % kRing == 0;
      const bool graph = chunks && gh.ge;
      const bool make = chunks && !gh.ge && launched > 0 && left * per_step >= kGraphFrom;
      if (graph) {
        RKX_HIP(hipGraphLaunch(gh.ge, stream));
        launched += chunk;
      } else {
        // twice as many before a graph is captured, to bridge that time
        const double most = make ? 2 * group : group;
        const int n = static_cast<int>(std::fmin(want, most));
        for (int k = 0; k < n; ++k, ++launched)
          RKX_HIP(enqueue(static_cast<int>(launched & (kRing - 1)), k == n - 1));
        if (make)
          if (int rc = capture())
            return rc;
      }
      spin = 0;
      continue;
    }
    if (spin % 64 == 0) {
      // every launch has run and the loop has not moved past the last but
      // one: the device-side control is not running -- stop, do not spin
      const hipError_t q = hipStreamQuery(stream);
      if (q == hipSuccess) {
        const long long now = static_cast<long long>(w.acc) + w.rej;
        if (!__atomic_load_n(&view.done, __ATOMIC_ACQUIRE) && now + 1 < launched && now == made)
          return fail(RKX_EDEVICE, "device step control made no progress");
      } else if (q != hipErrorNotReady) {
        return fail(RKX_EDEVICE, std::string("a step failed: ") + hipGetErrorString(q));
      } else {
        (void) hipGetLastError();
      }
      std::this_thread::yield();
    }
  }
}

}  // namespace

extern "C" {

const char *rkx_last_error(void) { return g_last_error.c_str(); }

int rkx_release_workspaces(void)
{
  pool_release();
  solve_mem::release_pinned();
  return RKX_OK;
}

int rkx_device_sync(void)
{
  RKX_HIP(hipDeviceSynchronize());
  return RKX_OK;
}

void rkx_opts_default(rkx_opts *o)
{
  if (!o)
    return;
  std::memset(o, 0, sizeof(*o));
  o->impl = RKX_IMPL_PIPEDLS;
  o->ctrl = RKX_CTRL_DEVICE;
}

int rkx_ode_bruss2d(rkx_ode *p, int N, double alpha)
{
  if (!p || N < 2 || N > 32767)
    return fail(RKX_EINVAL, "rkx_ode_bruss2d: need 2 <= N <= 32767 (n = 2N^2 fits in int)");
  std::memset(p, 0, sizeof(*p));
  p->kind = RKX_BRUSS2D;
  p->grid = N;
  p->n = 2 * N * N;
  p->alpha = alpha;
  return RKX_OK;
}

int rkx_ode_lv(rkx_ode *p, int pairs, double c0, double d0, double d1, double c1)
{
  if (!p || pairs < 1 || pairs > (1 << 29))
    return fail(RKX_EINVAL, "rkx_ode_lv: bad pair count");
  std::memset(p, 0, sizeof(*p));
  p->kind = RKX_LV;
  p->grid = pairs;
  p->n = 2 * pairs;
  p->c0 = c0;
  p->d0 = d0;
  p->d1 = d1;
  p->c1 = c1;
  return RKX_OK;
}

int rkx_ode_lv_chain(rkx_ode *p, int cells, double c0, double d0, double d1, double c1,
                     double diff)
{
  if (!p || cells < 3 || cells > (1 << 29))
    return fail(RKX_EINVAL, "rkx_ode_lv_chain: need 3 <= cells");
  std::memset(p, 0, sizeof(*p));
  p->kind = RKX_LV_CHAIN;
  p->grid = cells;
  p->n = 2 * cells;
  p->c0 = c0;
  p->d0 = d0;
  p->d1 = d1;
  p->c1 = c1;
  p->diff = diff;
  return RKX_OK;
}

int rkx_ode_acc_dist(const rkx_ode *p)
{
  if (check_ode(p))
    return RKX_EINVAL;
  switch (p->kind) {
  case RKX_BRUSS2D: return 2 * p->grid;
  case RKX_LV: return 1;
  default: return 2;
  }
}

int rkx_ode_start(const rkx_ode *p, double t, double *y0)
{
  (void) t;
  if (int rc = check_ode(p))
    return rc;
  if (!y0)
    return fail(RKX_EINVAL, "rkx_ode_start: null y0");
  if (p->kind == RKX_BRUSS2D) {
    const int N = p->grid;
    for (int i = 0; i < N; ++i)
      for (int j = 0; j < N; ++j) {
        y0[2 * N * i + 2 * j] = 0.5 + static_cast<double>(j) / static_cast<double>(N - 1);
        y0[2 * N * i + 2 * j + 1] =
            1.0 + (5.0 * static_cast<double>(i)) / static_cast<double>(N - 1);
      }
  } else {
    for (int i = 0; i < p->n; i += 2) {   // lv.c:58-62
      y0[i] = 0.2;
      y0[i + 1] = 1.1;
    }
  }
  return RKX_OK;
}

// splitmix64 finaliser over (seed, instance, index): a counter-based generator,
// so every value is reproducible independently of generation order.
static inline unsigned long long rkx_mix(unsigned long long z)
{
  z += 0x9E3779B97F4A7C15ull;
  z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
  z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
  return z ^ (z >> 31);
}

static inline double rkx_unit(unsigned long long seed, int inst, long long idx)
{
  const unsigned long long k =
      rkx_mix(seed ^ rkx_mix(static_cast<unsigned long long>(inst) * 0x100000001B3ull) ^
              rkx_mix(static_cast<unsigned long long>(idx) + 0x632BE59BD9B4E019ull));
  return static_cast<double>(k >> 11) * 0x1.0p-53;   // [0, 1)
}

int rkx_ode_start_seeded(const rkx_ode *p, unsigned long long seed, int instance, double amp,
                         double *y0)
{
  if (int rc = rkx_ode_start(p, 0.0, y0))
    return rc;
  if (p->kind == RKX_BRUSS2D) {
    const int N = p->grid;
    for (long long c = 0; c < static_cast<long long>(N) * N; ++c)
      y0[2 * c] = y0[2 * c] + amp * (2.0 * rkx_unit(seed, instance, c) - 1.0);
  } else {
    for (int c = 0; c < p->n / 2; ++c) {
      y0[2 * c] = 0.2 + 0.1 * rkx_unit(seed, instance, 2 * c);
      y0[2 * c + 1] = 1.1 + 0.1 * rkx_unit(seed, instance, 2 * c + 1);
    }
  }
  return RKX_OK;
}

int rkx_eval_rng_device(const rkx_ode *p, int i, int j, double t, const double *y_dev,
                        double *f_dev, void *stream)
{
  (void) t;
  if (int rc = check_ode(p))
    return rc;
  if (i < 0 || j >= p->n || j < i || !y_dev || !f_dev)
    return fail(RKX_EINVAL, "rkx_eval_rng_device: bad range or pointer");
  hipStream_t s = static_cast<hipStream_t>(stream);
  if (!s)
    if (int rc = default_stream(&s))
      return rc;
  const dev_ode d = make_dev_ode(*p);
  RKX_HIP(launch_eval_rng(d, i, j, y_dev, f_dev, s));
  RKX_HIP(hipStreamSynchronize(s));
  return RKX_OK;
}

int rkx_eval_rng_host(const rkx_ode *p, int i, int j, double t, const double *y, double *f)
{
  (void) t;
  if (int rc = check_ode(p))
    return rc;
  if (i < 0 || j >= p->n || j < i || !y || !f)
    return fail(RKX_EINVAL, "rkx_eval_rng_host: bad range or pointer");
  // Only the components the stencils of f[i..j] read travel to the device:
  // [i - d - 1, j + d + 1] clipped to the vector (the periodic chain reads
  // across its ends, so it sends everything).  The kernel indexes absolutely,
  // so it gets the window's base shifted back by lo, as the reference's tiled
  // stages pass v - first to ode_eval_rng (include/block-inline.h:338).
  const int d = rkx_ode_acc_dist(p);
  int lo = 0, hi = p->n - 1;
  if (p->kind != RKX_LV_CHAIN) {
    lo = std::max(0, (i & ~1) - d);
    hi = std::min(p->n - 1, (j | 1) + d);
  }
  const size_t win = static_cast<size_t>(hi - lo + 1);
  // per-thread device staging, grown on demand and kept for the thread's
  // later calls (a problem object's callbacks are called many times)
  thread_local double *yd = nullptr, *fd = nullptr;
  thread_local size_t cap = 0;
  if (win > cap) {
    if (yd)
      (void) hipFree(yd);
    if (fd)
      (void) hipFree(fd);
    yd = fd = nullptr;
    cap = 0;
    if (int rc = device_alloc(reinterpret_cast<void **>(&yd), win * sizeof(double)))
      return rc;
    if (int rc = device_alloc(reinterpret_cast<void **>(&fd), win * sizeof(double)))
      return rc;
    cap = win;
  }
  hipStream_t s = nullptr;
  if (int rc = default_stream(&s))
    return rc;
  RKX_HIP(hipMemcpyAsync(yd, y + lo, win * sizeof(double), hipMemcpyHostToDevice, s));
  const dev_ode dp = make_dev_ode(*p);
  RKX_HIP(launch_eval_rng(dp, i, j, yd - lo, fd - lo, s));
  RKX_HIP(hipMemcpyAsync(f + i, fd + (i - lo), static_cast<size_t>(j - i + 1) * sizeof(double),
                         hipMemcpyDeviceToHost, s));
  RKX_HIP(hipStreamSynchronize(s));
  return RKX_OK;
}

int rkx_eval_comp_host(const rkx_ode *p, int i, double t, const double *y, double *out)
{
  if (!out)
    return fail(RKX_EINVAL, "rkx_eval_comp_host: null output");
  double v[2] = {0.0, 0.0};
  // a one-component range written at absolute index i into v - (i & ~1)
  if (int rc = rkx_eval_rng_host(p, i, i, t, y, v - (i & ~1)))
    return rc;
  *out = v[i & 1];
  return RKX_OK;
}

// The full-storage loop order that moves the fewest vectors of n per step
// for a table: D (block-inline.h:253-320) scatters into s+1 accumulators, A
// and E gather each stage from the stage derivatives (A skipping the zero
// entries of the table), F fuses each RHS with the next stage's gather.  All
// give the same results bitwise.  Counts: reads + writes of n doubles.
//
// On BRUSS2D they run up to four stages to a kernel (rkx_kernels_groups.hip)
// and move 15 (D) and 9 vectors a step for 7 stages, 57 and 32 for 13.
static int least_traffic_form(const rkx_ode &p, const rkx_method &m)
{
  // BRUSS2D, stages in groups: one group of up to 4 stages moves y and y_new
  // alone and D's kernel is the simpler (RK4, N = 1000: 17.4 us a step, A
  // 18.9); with more, D's partial sums cost more than E's stage derivatives
  // (DOPRI54 N = 1000 51 and 50 us, N = 2000 246 and 162; 13 stages, N = 1000,
  // 179 and 130)
  if (p.kind == RKX_BRUSS2D)
    return m.s <= 4 ? RKX_IMPL_D : RKX_IMPL_E;
  const int s = m.s;
  int d = (s + 2) + 5;                                   // first and last stage
  for (int i = 1; i < s - 1; ++i)
    d += 5 + 2 * (s - 1 - i);
  int a = 2 + 1, e = 2 + 1;                              // stage 0; output reads y
  for (int l = 1; l < s; ++l) {
    int nz = 0;
    for (int i = 0; i < l; ++i)
      nz += (m.A[l][i] != 0.0);
    a += 4 + nz;
    e += 4 + l;
  }
  for (int i = 0; i < s; ++i) {
    a += (i == 0 || m.b[i] != 0.0 || m.b[i] - m.b_hat[i] != 0.0) ? 1 : 0;
    e += 1;
  }
  a += 1;                                                // y_new
  e += 1;
  int f = 3 + 2 + (s + 2);                               // stage 0, last stage, output
  for (int l = 1; l < s - 1; ++l)
    f += l + 4;
  int best = RKX_IMPL_D, cost = d;
  if (f < cost) { best = RKX_IMPL_F; cost = f; }
  if (a < cost) { best = RKX_IMPL_A; cost = a; }
  if (e < cost) { best = RKX_IMPL_E; cost = e; }
  return best;
}

size_t rkx_solve_footprint(const rkx_ode *p, const rkx_method *m, int impl)
{
  if (check_ode(p) || check_method(m))
    return 0;
  const size_t vec = static_cast<size_t>(p->n) * sizeof(double);
  const size_t fixed = sizeof(state) + sizeof(dev_method) + sizeof(dev_coef);
  const dev_ode dp = make_dev_ode(*p);
  const bool fused =
      sweep_supported(dp, *m) || chain_supported(dp, *m) || pairs_supported(dp, *m);
  const size_t s = static_cast<size_t>(m->s);
  if ((impl == RKX_IMPL_PIPED || impl == RKX_IMPL_PIPEDLS) && !fused)
    impl = least_traffic_form(*p, *m);
  if (impl == RKX_IMPL_A || impl == RKX_IMPL_E)
    return (2 + s + 1) * vec + fixed;            // y x2, v_0..v_{s-1}, w
  if (impl == RKX_IMPL_F)
    return (2 + s + 2) * vec + fixed;            // y x2, v_0..v_{s-1}, w x2
  if (impl == RKX_IMPL_D)
    return (2 + (s - 1) + 2) * vec + fixed;      // y x2, w_1..w_{s-1}, dy, err
  return 2 * vec + fixed;                        // y x2
}

int rkx_solve(const rkx_ode *p, const rkx_method *m, double t0, double te,
              const double *y0_dev, double *y_dev, double tol, const rkx_opts *o_in,
              rkx_stats *st_out)
{
  if (int rc = check_ode(p))
    return rc;
  if (int rc = check_method(m))
    return rc;
  if (!y0_dev || !y_dev)
    return fail(RKX_EINVAL, "rkx_solve: null vector");
  rkx_opts o;
  if (o_in)
    o = *o_in;
  else
    rkx_opts_default(&o);
  if (o.impl < RKX_IMPL_D || o.impl > RKX_IMPL_F)
    return fail(RKX_EINVAL, "rkx_solve: unknown impl");
  if (o.ctrl != RKX_CTRL_DEVICE && o.ctrl != RKX_CTRL_HOST)
    return fail(RKX_EINVAL, "rkx_solve: unknown step-control mode");
  if (o.trace_cap < 0 || (o.trace_cap > 0 && !o.trace))
    return fail(RKX_EINVAL, "rkx_solve: trace_cap without a trace buffer");
  if (o.dump_path)
    o.ctrl = RKX_CTRL_HOST;          // the dump needs every attempted step on the host
  hipStream_t stream = static_cast<hipStream_t>(o.stream);
  if (!stream)
    if (int rc = default_stream(&stream))
      return rc;

  const dev_ode dp = make_dev_ode(*p);
  const int s = m->s;
  int impl = o.impl;
  // fused forms: the row sweep, the tile form or the one-workgroup form for
  // BRUSS2D, the segment kernel for the LV chain, the per-pair kernel for LV
  // pairs; anything else (tables without a compiled pattern or stage count)
  // runs the full-storage loop order with the least traffic.  D, A, E and F
  // run as asked on every problem.
  bool fused = impl == RKX_IMPL_PIPED || impl == RKX_IMPL_PIPEDLS;
  if (fused && !chain_supported(dp, *m) && !pairs_supported(dp, *m) &&
      !sweep_supported(dp, *m)) {
    impl = least_traffic_form(*p, *m);
    fused = false;
  }
  const bool gather = impl == RKX_IMPL_A || impl == RKX_IMPL_E || impl == RKX_IMPL_F;
  // on BRUSS2D the full-storage forms run their stages in groups; these and the
  // fused forms start each step with the control of the one before (step_ring)
  const bool grouped = !fused && dp.kind == RKX_BRUSS2D;
  const bool ringed = fused || grouped;
  const size_t n = static_cast<size_t>(p->n);
  const size_t vec = n * sizeof(double);

  solve_mem mem;
  mem.stream = stream;
  if (int rc = mem.take_pinned())
    return rc;
  double *ybuf[2] = {nullptr, nullptr};
  double *w = nullptr, *dy = nullptr, *err = nullptr, *trace_dev = nullptr;
  double *v = nullptr, *w1 = nullptr;   // gather forms: v_0..v_{s-1}; F's second w
  solve_ctl *ctl_dev = nullptr;
  if (int rc = mem.alloc(reinterpret_cast<void **>(&ctl_dev), sizeof(solve_ctl)))
    return rc;
  state *st_dev = &ctl_dev->st;
  dev_coef *cf_dev = &ctl_dev->coef;
  const step_refs ref{st_dev, &ctl_dev->ring, &ctl_dev->meth, &mem.host->view};
  for (int b = 0; b < 2; ++b)
    if (int rc = mem.alloc(reinterpret_cast<void **>(&ybuf[b]), vec))
      return rc;
  if (impl == RKX_IMPL_D) {
    if (int rc = mem.alloc(reinterpret_cast<void **>(&w), vec * (s - 1)))
      return rc;
    if (int rc = mem.alloc(reinterpret_cast<void **>(&dy), vec))
      return rc;
    if (int rc = mem.alloc(reinterpret_cast<void **>(&err), vec))
      return rc;
  } else if (gather) {
    if (int rc = mem.alloc(reinterpret_cast<void **>(&v), vec * s))
      return rc;
    if (int rc = mem.alloc(reinterpret_cast<void **>(&w), vec))
      return rc;
    if (impl == RKX_IMPL_F)
      if (int rc = mem.alloc(reinterpret_cast<void **>(&w1), vec))
        return rc;
  }
  const gather_masks nz = make_gather_masks(*m);
  if (o.trace_cap > 0)
    if (int rc = mem.alloc(reinterpret_cast<void **>(&trace_dev),
                           sizeof(double) * 3 * static_cast<size_t>(o.trace_cap)))
      return rc;

  solve_ctl hc{};
  fill_dev_method(*m, hc.meth);
  state &hs = hc.st;
  hs.v.t = t0;
  hs.v.te = te;
  hs.v.tol = tol;
  hs.v.h = initial_h(te - t0, tol, o.step_limit, o.h0);
  hs.v.step_limit = o.step_limit;
  hs.v.ord = m->ord;
  hs.v.done = !(t0 < te);
  hs.ctrl = o.ctrl;
  hs.trace = trace_dev;
  hs.trace_cap = o.trace_cap;
  hs.s = s;
  hs.meth = &ctl_dev->meth;
  hs.coef = cf_dev;
  hs.view = &mem.host->view;
  mem.host->view = host_view{t0, hs.v.h, 0, 0, 0, 0};
  if (ringed) {
    hs.ring = ref.ring;
    hc.ring = make_ring(hs.v, trace_dev != nullptr);
  }
  premult(hc.meth, s, hs.v.h, hc.coef);
  RKX_HIP(hipMemcpyAsync(ctl_dev, &hc, sizeof(hc), hipMemcpyHostToDevice, stream));
  RKX_HIP(hipMemcpyAsync(ybuf[0], y0_dev, vec, hipMemcpyDeviceToDevice, stream));

  if (o.tile_waves > 4)
    return fail(RKX_EINVAL, "rkx_solve: tile_waves must be 1..4");
  fused_plan plan;
  if (fused) {
    if (int rc = make_fused_plan(*p, *m, o.tile_rows, o.tile_waves, ref, cf_dev, ybuf[0], ybuf[1],
                                 &plan))
      return fail(rc, std::string("rkx_solve: ") + rkx_last_error());
  } else if (grouped) {
    plan.kind = fused_plan::kGroups;
    plan.form = impl;
    plan.nz = nz;
    plan.groups = stage_group{dp.N,    s,       0, 0, 0, 0, 0, dp.coef, ybuf[0], ybuf[1],
                              gather ? v : w, dy, err, ref};
  }

  // one attempted step; r: the ring slot a fused kernel reads; report: the
  // full-storage forms show the state the step starts from
  auto enqueue_step = [&](int r, bool report) -> hipError_t {
    if (ringed)
      return plan.launch(r, stream);
    if (impl == RKX_IMPL_D)
      return launch_d_step(dp, cf_dev, s, st_dev, ybuf[0], ybuf[1], w, dy, err, report,
                           stream);
    return launch_gather_step(impl, dp, cf_dev, s, nz, st_dev, ybuf[0], ybuf[1], v, w, w1, report,
                              stream);
  };

  RKX_HIP(hipStreamSynchronize(stream));           // the copies above read hc
  const auto t_start = std::chrono::steady_clock::now();
  step_vars fin = hs.v;

  if (hs.v.done) {
    // nothing to integrate
  } else if (o.ctrl == RKX_CTRL_HOST) {
    // One host round trip per step: the device computes the error norm, the
    // host runs the reference's step control with the C library's pow.  All
    // of it goes through pinned memory, with one wait: the stream has done
    // what the host sent by the time the next step's error has come back.
    step_vars &cur = fin;
    solve_mem::pinned &pin = *mem.host;
    pin.coef = hc.coef;
    dump_file dump;
    std::vector<double> ydump;
    for (int r = 0; !cur.done;) {
      RKX_HIP(enqueue_step(r, false));
      r = (r + 1) & (kRing - 1);
      if (ringed)
        RKX_HIP(hipMemcpyAsync(&pin.err, &ref.ring->err[r], sizeof(pin.err), hipMemcpyDeviceToHost,
                               stream));
      else
        RKX_HIP(hipMemcpyAsync(&pin.st, st_dev, sizeof(state), hipMemcpyDeviceToHost, stream));
      RKX_HIP(hipStreamSynchronize(stream));
      const double step_err = ringed ? ring_err(pin.err) : pin.st.err;
      const int attempt = cur.acc + cur.rej;
      if (o.dump_path) {
        // the step's new y is in the other buffer until the decision flips cur
        ydump.resize(n);
        RKX_HIP(hipMemcpy(ydump.data(), ybuf[cur.cur ^ 1], vec, hipMemcpyDeviceToHost));
        if (int rc = dump.append(o.dump_path, cur.t, cur.h, ydump))
          return rc;
      }
      if (o.trace && attempt < o.trace_cap) {
        o.trace[3 * attempt + 0] = cur.t;
        o.trace[3 * attempt + 1] = cur.h;
        o.trace[3 * attempt + 2] = step_err;
      }
      host_finish(cur, step_err);
      if (ringed) {
        pin.slot = step_slot{cur, 0, 0};
        RKX_HIP(hipMemcpyAsync(&ref.ring->slot[r], &pin.slot, sizeof(step_slot),
                               hipMemcpyHostToDevice, stream));
      } else {
        premult(hc.meth, s, cur.h, pin.coef);
        RKX_HIP(hipMemcpyAsync(cf_dev, &pin.coef, sizeof(dev_coef), hipMemcpyHostToDevice, stream));
        pin.st.v = cur;
        RKX_HIP(hipMemcpyAsync(st_dev, &pin.st, sizeof(state), hipMemcpyHostToDevice, stream));
      }
    }
  } else {
    auto enqueue_many = [&](int r, bool) { return plan.launch_many(r, stream); };
    host_view &view = mem.host->view;
    const int kernels = ringed ? 1 : impl == RKX_IMPL_D ? s : impl == RKX_IMPL_F ? s + 1 : 2 * s;
    if (int rc = plan.many > 0 ? run_steps(enqueue_many, 1, plan.many, view, te, o.step_limit,
                                           mem.steps, stream)
                               : run_steps(enqueue_step, kernels, 0, view, te, o.step_limit,
                                           mem.steps, stream))
      return rc;
    fin.t = view.t;
    fin.h = view.h;
    fin.acc = view.acc;
    fin.rej = view.rej;
    fin.cur = view.cur;
  }
  const auto t_end = std::chrono::steady_clock::now();
  RKX_HIP(hipMemcpyAsync(y_dev, ybuf[fin.cur], vec, hipMemcpyDeviceToDevice, stream));
  if (o.trace_cap > 0 && o.ctrl != RKX_CTRL_HOST) {
    const int ntr = std::min(o.trace_cap, fin.acc + fin.rej);
    if (ntr > 0)
      RKX_HIP(hipMemcpyAsync(o.trace, trace_dev, sizeof(double) * 3 * ntr, hipMemcpyDeviceToHost,
                             stream));
  }
  RKX_HIP(hipStreamSynchronize(stream));
  if (st_out) {
    st_out->steps_acc = fin.acc;
    st_out->steps_rej = fin.rej;
    st_out->t = fin.t;
    st_out->h = fin.h;
    st_out->kernel_time = std::chrono::duration<double>(t_end - t_start).count();
    st_out->resident_bytes = rkx_solve_footprint(p, m, impl);
  }
  return RKX_OK;
}

int rkx_solve_host(const rkx_ode *p, const rkx_method *m, double t0, double te, const double *y0,
                   double *y, double tol, const rkx_opts *o, rkx_stats *st)
{
  if (int rc = check_ode(p))
    return rc;
  if (!y0 || !y)
    return fail(RKX_EINVAL, "rkx_solve_host: null vector");
  const size_t vec = static_cast<size_t>(p->n) * sizeof(double);
  solve_mem mem;
  double *d0 = nullptr, *d1 = nullptr;
  if (int rc = mem.alloc(reinterpret_cast<void **>(&d0), vec))
    return rc;
  if (int rc = mem.alloc(reinterpret_cast<void **>(&d1), vec))
    return rc;
  RKX_HIP(hipMemcpy(d0, y0, vec, hipMemcpyHostToDevice));
  if (int rc = rkx_solve(p, m, t0, te, d0, d1, tol, o, st))
    return rc;
  RKX_HIP(hipMemcpy(y, d1, vec, hipMemcpyDeviceToHost));
  return RKX_OK;
}

}  // extern "C"
