// wt_autotune.hip -- measured choice of the temporally blocked kernels'
// tiling for one problem shape, behind the C ABI.
//
// The reference has no tuner: its time loop is a Python loop over torch ops
// (rnn.py:50-67).  This search times the library's own forward (and, with
// gradients, checkpointed adjoint) on the caller's device buffers, starting
// from the library's heuristic plan (wt_plan_resolve) and moving one tuning
// field at a time through its options -- tiles per sample (strips x column
// tiles) around the heuristic's, time-block depth, rows per thread, for the
// forward and the adjoint separately -- then the coupled (depth, rows) pairs,
// keeping any change that is faster by more than 0.5%, for two passes or
// until the time budget runs out.  Every candidate is built through
// wt_plan_create, so a tiling no kernel variant can hold is skipped, and
// every candidate computes the same result (the tiling changes only the
// order of work, not the arithmetic; the forward is bitwise equal across
// tilings, the adjoint's sums likewise).
//
// The search allocates its own device buffers (workspaces, probe outputs,
// seeds, gradients) with hipMalloc and frees them before returning; results
// are cached per shape in the library (behind a mutex) for the life of the
// process.  It uses only the public entry points of include/wavetorch_hip.h.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstring>
#include <map>
#include <mutex>
#include <set>
#include <string>
#include <tuple>
#include <vector>

#include "wt_internal.h"

namespace {

using wt::set_error;

// Options of each field (column-segment family: rows per thread must be a
// compiled variant at 1024 threads).
const int kTblock[] = {4, 6, 8, 12, 16, 20, 24, 32};
const int kCpt[] = {4, 6, 8, 10, 12};
const int kATblock[] = {4, 5, 6, 8, 10, 12, 13, 16, 20, 24};
const int kACpt[] = {4, 6, 8, 10};

struct Cand {
  int s, c, tb, r, as, ac, atb, ar;
  bool operator<(const Cand &o) const {
    return std::tie(s, c, tb, r, as, ac, atb, ar) <
           std::tie(o.s, o.c, o.tb, o.r, o.as, o.ac, o.atb, o.ar);
  }
};

wt_tuning to_tuning(const Cand &k, int ck_every) {
  wt_tuning t;
  std::memset(&t, 0, sizeof(t));
  t.kind = 0;
  t.strips = k.s; t.tcols = k.c; t.tblock = k.tb; t.nt = 1024; t.cpt = k.r;
  t.a_strips = k.as; t.a_tcols = k.ac; t.a_tblock = k.atb; t.a_nt = 1024; t.a_cpt = k.ar;
  t.ck_every = ck_every;
  return t;
}

Cand from_tuning(const wt_tuning &t) {
  Cand k;
  k.s = std::max(1, t.strips); k.c = std::max(1, t.tcols); k.tb = t.tblock; k.r = t.cpt;
  k.as = t.a_strips ? t.a_strips : k.s;
  k.ac = t.a_tcols ? t.a_tcols : k.c;
  k.atb = t.a_tblock ? t.a_tblock : k.tb;
  k.ar = t.a_cpt ? t.a_cpt : k.r;
  return k;
}

// (strips, tcols) options around s0 x c0: s, c in 1..6 or within 0.5x-1.5x of
// s0, c0, tiles at most 2:1, tile count within 4x of s0*c0 either way.
std::vector<std::pair<int, int>> tilings(int Nx, int Ny, int s0, int c0) {
  auto near = [](int v0) {
    std::set<int> v;
    for (int i = 1; i <= 6; ++i) v.insert(i);
    const double r[] = {0.5, 0.625, 0.75, 0.875, 1.125, 1.25, 1.5};
    for (double x : r) v.insert(std::max(1, (int)std::lround(v0 * x)));
    v.insert(v0);
    return v;
  };
  std::vector<std::pair<int, int>> out;
  for (int s : near(s0)) {
    if (s > Nx) continue;
    for (int c : near(c0)) {
      if (c > Ny) continue;
      if (s != s0 || c != c0) {
        const double n0 = (double)s0 * c0, n = (double)s * c;
        if (n < n0 / 4 || n > n0 * 4) continue;
        const double a = ((double)Nx / s) / ((double)Ny / c);
        if (std::max(a, 1.0 / a) > 2.0 + 1e-9 && s * c > 1) continue;
      }
      out.emplace_back(s, c);
    }
  }
  return out;
}

// Device buffers of the search, grown on demand.
struct Buf {
  void *p = nullptr;
  size_t n = 0;
  int grow(size_t want) {
    if (want <= n) return 0;
    if (p) (void)hipFree(p);
    p = nullptr;
    n = 0;
    if (hipMalloc(&p, want) != hipSuccess) return -1;
    n = want;
    return 0;
  }
  ~Buf() {
    if (p) (void)hipFree(p);
  }
};

struct Entry {
  wt_tuning t;
  double ms;
};
std::mutex g_mu;
std::map<std::string, Entry> g_cache;

std::string cache_key(const wt_config *cfg, int B, int T, int ck, int group, int with_grad) {
  char buf[256];
  std::snprintf(buf, sizeof(buf), "%dx%d:B%d:T%d:K%d,%d:g%d:h%g:nl%g,%g,%g,%d:s%d:p%d", cfg->Nx,
                cfg->Ny, B, T, ck, group, with_grad, cfg->h, cfg->sat_b0, cfg->sat_uth, cfg->c_nl,
                cfg->c_clamp, cfg->nsrc_px, cfg->ntap);
  return buf;
}

}  // namespace

extern "C" int wt_autotune(const wt_config *cfg, int32_t B, int32_t T, float cmax,
                           const wt_tuning *start, int32_t with_grad, const float *b,
                           const float *c, const float *rho, const float *x, int32_t reps,
                           double budget_ms, wt_tuning *out, double *best_ms, void *stream) {
  return wt_autotune_group(cfg, B, T, cmax, start, 0, with_grad, b, c, rho, x, reps, budget_ms,
                           out, best_ms, stream);
}

extern "C" int wt_autotune_group(const wt_config *cfg, int32_t B, int32_t T, float cmax,
                                 const wt_tuning *start, int32_t group, int32_t with_grad,
                                 const float *b, const float *c, const float *rho, const float *x,
                                 int32_t reps, double budget_ms, wt_tuning *out, double *best_ms,
                                 void *stream) {
  const char *what = "wt_autotune";
  if (!cfg || !b || !c || !x || !out || group < 0) {
    set_error("%s: invalid argument (null pointer or negative group)", what);
    return WT_EINVAL;
  }
  if (reps < 1 || reps > 100 || !(budget_ms > 0)) {
    set_error("%s: reps %d (1..100), budget_ms %g (> 0)", what, reps, budget_ms);
    return WT_EINVAL;
  }
  hipStream_t st = (hipStream_t)stream;
  wt_tuning base_req;
  std::memset(&base_req, 0, sizeof(base_req));
  if (start) base_req = *start;
  base_req.plain = 0;
  base_req.kind = 0;
  // the heuristic's plan (also validates the configuration, CFL included)
  wt_tuning base;
  int rc = wt_plan_resolve(cfg, B, T, cmax, &base_req, &base, nullptr, nullptr);
  if (rc != WT_OK) return rc;
  const std::string key = cache_key(cfg, B, T, base.ck_every, group, with_grad);
  {
    std::lock_guard<std::mutex> lk(g_mu);
    auto it = g_cache.find(key);
    if (it != g_cache.end()) {
      *out = it->second.t;
      if (best_ms) *best_ms = it->second.ms;
      return WT_OK;
    }
  }
  if (base.kind != 0 || base.plain) {
    // no blocked variant fits this configuration: nothing to search
    *out = base;
    if (best_ms) *best_ms = NAN;
    return WT_OK;
  }

  const int P = std::max(cfg->ntap, 1);
  const size_t nyb = (size_t)B * T * P * sizeof(float);
  const size_t nf = (size_t)cfg->Nx * cfg->Ny * sizeof(float);
  Buf saved, temp, y, ybar, gc, gb, gr, gx;
  if (y.grow(nyb) || ybar.grow(nyb) || gc.grow(nf) || gx.grow((size_t)B * T * sizeof(float)) ||
      ((cfg->sat_b0 > 0 || cfg->c_nl != 0) && (gb.grow(nf) || gr.grow(nf)))) {
    set_error("%s: hipMalloc of the search buffers failed", what);
    return WT_EHIP;
  }
  // seeds: 1e-3 at every probe output (any value drives the same kernels)
  {
    std::vector<float> h(nyb / sizeof(float), 1e-3f);
    if (hipMemcpy(ybar.p, h.data(), nyb, hipMemcpyHostToDevice) != hipSuccess) {
      set_error("%s: hipMemcpy of the seeds failed", what);
      return WT_EHIP;
    }
  }
  struct Events {
    hipEvent_t e[2] = {nullptr, nullptr};
    ~Events() {
      for (hipEvent_t x : e)
        if (x) (void)hipEventDestroy(x);
    }
  } ev;
  if (hipEventCreate(&ev.e[0]) != hipSuccess || hipEventCreate(&ev.e[1]) != hipSuccess) {
    set_error("%s: hipEventCreate failed", what);
    return WT_EHIP;
  }
  hipEvent_t e0 = ev.e[0], e1 = ev.e[1];
  const auto t_start = std::chrono::steady_clock::now();
  auto elapsed_ms = [&] {
    return std::chrono::duration<double, std::milli>(std::chrono::steady_clock::now() - t_start)
        .count();
  };
  const bool nl = cfg->sat_b0 > 0 || cfg->c_nl != 0;

  // time of one candidate (infinity when no variant holds it)
  auto measure = [&](const Cand &k, double &ms_out) -> int {
    ms_out = INFINITY;
    wt_tuning t = to_tuning(k, base.ck_every);
    void *plan = nullptr;
    if (wt_plan_create(cfg, B, T, cmax, &t, &plan) != WT_OK) return WT_OK;  // skipped
    int64_t sb = 0, tb = 0;
    int r = group > 0 ? wt_plan_group(plan, group) : WT_OK;
    if (r == WT_OK) r = wt_workspace_bytes(plan, with_grad, &sb, &tb);
    if (r == WT_OK && (saved.grow((size_t)std::max<int64_t>(sb, 256)) ||
                       temp.grow((size_t)std::max<int64_t>(tb, 256)))) {
      set_error("%s: hipMalloc of a workspace failed (%lld + %lld bytes)", what, (long long)sb,
                (long long)tb);
      r = WT_EHIP;
    }
    auto run = [&]() -> int {
      int q = wt_loop_fwd(plan, b, c, rho, x, (float *)y.p, nullptr, 1, with_grad, saved.p,
                          temp.p, stream);
      if (q != WT_OK || !with_grad) return q;
      return wt_loop_adj(plan, b, c, rho, x, (const float *)ybar.p, nullptr, saved.p, temp.p,
                         (float *)gc.p, nl ? (float *)gb.p : nullptr,
                         nl ? (float *)gr.p : nullptr, (float *)gx.p, stream);
    };
    if (r == WT_OK) r = run();  // warm-up (first launch of each kernel variant)
    for (int i = 0; r == WT_OK && i < reps; ++i) {
      if (hipEventRecord(e0, st) != hipSuccess) { r = WT_EHIP; break; }
      r = run();
      if (r != WT_OK) break;
      if (hipEventRecord(e1, st) != hipSuccess || hipEventSynchronize(e1) != hipSuccess) {
        r = WT_EHIP;
        break;
      }
      float ms = 0.f;
      (void)hipEventElapsedTime(&ms, e0, e1);
      ms_out = std::min(ms_out, (double)ms);
    }
    if (r == WT_EHIP) set_error("%s: a timed run failed (%s)", what,
                                hipGetErrorString(hipGetLastError()));
    wt_plan_destroy(plan);
    return r;
  };

  Cand state = from_tuning(base);
  double best = INFINITY;
  rc = measure(state, best);
  if (rc == WT_OK && !std::isfinite(best)) {
    set_error("%s: the heuristic plan could not be timed", what);
    rc = WT_EUNSUPPORTED;
  }
  std::set<Cand> tried;
  tried.insert(state);
  auto consider = [&](const Cand &k) -> bool {
    if (rc != WT_OK || tried.count(k) || elapsed_ms() > budget_ms) return false;
    tried.insert(k);
    double t = INFINITY;
    rc = measure(k, t);
    if (rc == WT_OK && t < best * 0.995) {
      state = k;
      best = t;
      return true;
    }
    return false;
  };
  const auto ftil = tilings(cfg->Nx, cfg->Ny, state.s, state.c);
  const auto atil = tilings(cfg->Nx, cfg->Ny, state.as, state.ac);
  for (int round = 0; round < 2 && rc == WT_OK; ++round) {
    bool improved = false;
    for (auto &p : ftil) { Cand k = state; k.s = p.first; k.c = p.second; improved |= consider(k); }
    for (int v : kTblock) { Cand k = state; k.tb = v; improved |= consider(k); }
    for (int v : kCpt) { Cand k = state; k.r = v; improved |= consider(k); }
    if (with_grad) {
      for (auto &p : atil) { Cand k = state; k.as = p.first; k.ac = p.second; improved |= consider(k); }
      for (int v : kATblock) { Cand k = state; k.atb = v; improved |= consider(k); }
      for (int v : kACpt) { Cand k = state; k.ar = v; improved |= consider(k); }
    }
    // block depth and rows per thread are coupled: also move them together
    {
      const Cand s0 = state;
      for (int v1 : kTblock)
        for (int v2 : kCpt) { Cand k = s0; k.tb = v1; k.r = v2; improved |= consider(k); }
    }
    if (with_grad) {
      const Cand s0 = state;
      for (int v1 : kATblock)
        for (int v2 : kACpt) { Cand k = s0; k.atb = v1; k.ar = v2; improved |= consider(k); }
    }
    if (!improved) break;
  }
  if (rc != WT_OK) return rc;
  wt_tuning res = to_tuning(state, base.ck_every);
  // report what the library resolves the winner to (fills derived fields)
  wt_tuning resolved;
  rc = wt_plan_resolve(cfg, B, T, cmax, &res, &resolved, nullptr, nullptr);
  if (rc != WT_OK) return rc;
  {
    std::lock_guard<std::mutex> lk(g_mu);
    g_cache[key] = Entry{resolved, best};
  }
  *out = resolved;
  if (best_ms) *best_ms = best;
  return WT_OK;
}
