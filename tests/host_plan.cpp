// host_plan.cpp -- CPU checks of how the engine plans and prepares a pass: how
// it is cut into groups of shots (rtm::plan_groups), over batches of equal,
// growing and random windows, how with one stream only, the control block
// whose allocation fails, and the bound of the captured chunks that are kept.
// Built and run by tests/test_host_plan.py; prints one line per check and
// exits non-zero if one fails.
#include <stdio.h>
#include <string.h>

#include <algorithm>
#include <cmath>
#include <condition_variable>
#include <functional>
#include <map>
#include <mutex>
#include <random>
#include <string>
#include <vector>

#include <hip/hip_runtime.h>

#define private public   // the engine's control block
#include "rtm_engine.h"
#undef private

static int g_fail = 0;
#define CHECK(c, ...)                                                  \
  do {                                                                 \
    if (!(c)) {                                                        \
      printf("FAIL %s:%d: %s -- ", __FILE__, __LINE__, #c);            \
      printf(__VA_ARGS__);                                             \
      printf("\n");                                                    \
      g_fail = 1;                                                      \
    }                                                                  \
  } while (0)

static ShotDev window(int nxl, int nzi, int npml)
{
  ShotDev d;
  memset(&d, 0, sizeof(d));
  d.nxl = nxl; d.nzi = nzi; d.npml = npml;
  d.nxp = nxl + 2 * npml; d.nzp = nzi + 2 * npml;
  return d;
}

struct Plan { std::vector<std::vector<int>> g; bool cached; double total = 0, most = 0, pair = 0; };
static Plan plan(const std::vector<ShotDev>& ds, int phase)
{
  Plan p;
  p.g = rtm::plan_groups(ds, phase, p.cached);
  double prev = 0;
  for (auto& v : p.g) {
    double b = 0;
    for (int j : v) {
      const double x = rtm::live_bytes(ds[j], phase);
      b += x;
      p.most = std::max(p.most, x);
    }
    p.total += b;
    p.pair = std::max(p.pair, prev + b);
    prev = b;
  }
  return p;
}

// every shot once and in order, no empty group
static bool whole(const Plan& p, int n)
{
  int at = 0;
  for (auto& v : p.g) {
    if (v.empty()) return false;
    for (int j : v)
      if (j != at++) return false;
  }
  return at == n;
}

// The reverse pass.  Two neighbouring groups hold 200 MB on average, or 235
// where 200 would leave fewer than 1400 32-row tiles in flight or a shot is
// larger than 100 MB; with one shot more where a cut falls between shots.
static void reverse_bound(const char* name, const std::vector<ShotDev>& ds)
{
  const Plan p = plan(ds, PH_REV);
  const int nb = (int)ds.size(), n = (int)p.g.size();
  CHECK(whole(p, nb), "%s: %d shots, %d groups", name, nb, n);
  CHECK(nb == 1 ? n == 1 : n % 2 == 0 || n == nb, "%s: %d groups of %d shots", name, n, nb);
  double tiles = 0;
  for (const ShotDev& d : ds) tiles += (double)((d.nxp + 63) / 64) * ((d.nzp + 31) / 32);
  auto groups = [&](double bound) { return std::min(nb, 2 * (int)std::ceil(p.total / bound)); };
  if (nb > 1 && p.most <= 117.5e6) {
    const bool few = 2 * tiles / (2 * std::ceil(p.total / 200e6)) < 1400 || p.most > 100e6;
    CHECK(n == groups(few ? 235e6 : 200e6), "%s: %d shots of %.0f MB, %.0f tiles, in %d groups", name, nb, p.total / 1e6,
          tiles, n);
    CHECK(p.pair <= (few ? 235e6 : 200e6) + p.most, "%s: %d shots in %d groups, a pair holds %.0f MB", name, nb, n,
          p.pair / 1e6);
  } else {
    CHECK(n == std::min(2, nb), "%s: %d groups of large shots", name, n);
  }
  CHECK(p.cached == (p.pair <= 270e6), "%s: %d shots, %.0f MB, cached %d", name, nb, p.pair / 1e6, (int)p.cached);
}

// Plans on both sides of each of these lines: equal windows, their number and
// the groups that were the faster ones (rtm_engine.h).
static void known_plans()
{
  struct { int nxl, nzi, npml, shots, groups; } t[] = {
    {301, 512, 50, 16, 2},  {301, 512, 50, 32, 6},   {301, 512, 50, 34, 6},  {301, 512, 50, 64, 10},
    {301, 512, 50, 100, 14}, {301, 512, 50, 160, 22}, {301, 512, 50, 200, 28},
    {1431, 562, 50, 4, 2},  {1764, 970, 50, 4, 4},   {1953, 792, 50, 3, 3},  {2048, 1024, 50, 4, 2},
  };
  for (auto& k : t) {
    const Plan p = plan(std::vector<ShotDev>(k.shots, window(k.nxl, k.nzi, k.npml)), PH_REV);
    CHECK((int)p.g.size() == k.groups, "%d shots of %d x %d (%.0f MB): %zu groups, not %d", k.shots, k.nxl, k.nzi,
          p.total / 1e6, p.g.size(), k.groups);
  }
  // forward halves keep ordinary stores up to 270 MB together
  for (int n : {20, 40, 60}) {
    const Plan f = plan(std::vector<ShotDev>(n, window(301, 512, 50)), PH_FWD);
    CHECK(f.g.size() == 2 && f.cached == (f.total <= 270e6), "%d shots forward, %.0f MB, cached %d", n, f.total / 1e6,
          (int)f.cached);
  }
  printf("ok known plans\n");
}

// the batches of tests/test_gpu_lane_groups.py, which are there for a stream's
// second and third group
static void lane_group_jobs()
{
  std::vector<ShotDev> ragged;
  for (int k = 0; k < 121; k++) ragged.push_back(window(61 + 2 * (37 * k % 120), 300, 32));
  for (const auto& ds : {std::vector<ShotDev>(75, window(301, 300, 32)), ragged}) {
    const Plan p = plan(ds, PH_REV);
    bool equal = true;
    for (auto& g : p.g) equal &= g.size() == p.g[0].size();
    CHECK(p.g.size() >= 6, "%zu shots in %zu groups", ds.size(), p.g.size());
    CHECK(!equal, "%zu shots in groups of the same size", ds.size());
  }
  printf("ok several groups a stream\n");
}

// A control block that cannot be allocated (here: there is no GPU) is not
// counted as there by the next job, which would launch on its addresses; with
// a GPU both calls succeed.
static void control_block()
{
  rtm::Engine e(0);
  const int gpus = [] { int n = 0; return hipGetDeviceCount(&n) == hipSuccess ? n : 0; }();
  for (int call = 0; call < 3; call++) {
    const int rc = e.ensure_cb(10, 100 + 10 * (call == 2));
    CHECK((rc == 0) == (gpus > 0), "call %d returns %d with %d GPUs", call, rc, gpus);
    CHECK((rc == 0) == (e.cb_ != nullptr), "call %d returns %d, block %p", call, rc, e.cb_);
    CHECK(e.cb_ || (!e.d_ds_ && !e.d_tiles_ && !e.d_slots_ && !e.d_stk_ && !e.d_flag_ && !e.lane_[0].tiles &&
                    !e.lane_[1].act), "call %d leaves addresses of no block", call);
    CHECK(hipGetLastError() != hipErrorOutOfMemory, "call %d leaves its error for the next launch", call);
  }
  printf("ok control block\n");
}

// without a second stream (here: there is no GPU) a batch is one group on the
// engine's own: a lane of its own would be the default stream
static void one_lane()
{
  rtm::Engine e(0);
  const std::vector<ShotDev> ds(40, window(301, 512, 50));
  for (int phase : {PH_FWD, PH_REV}) {
    bool cached = true;
    const size_t n = e.groups_of(ds, phase, false, cached).size();
    CHECK((n == 1) == (e.lane_[0].st == nullptr || e.lane_[1].st == nullptr), "%zu groups with streams %p, %p", n,
          (void*)e.lane_[0].st, (void*)e.lane_[1].st);
    CHECK(n > 1 || !cached, "phase %d: all shots at once count as cached", phase);
    const auto t = e.groups_of(ds, phase, true, cached);
    CHECK(t.size() == 1 && t[0].slots.size() == 40 && !cached, "timed launches in %zu groups", t.size());
  }
  printf("ok one lane\n");
}

// the captured chunks that an engine keeps are bounded, the longest unused go
// first (the entries here hold no graph)
static void kept_graphs()
{
  rtm::Engine e(0);
  const int cap = (int)rtm::Engine::kMaxGraphs, n = 3 * cap;
  auto key = [](int i) {
    rtm::GraphKey k;
    memset(&k, 0, sizeof(k));
    k.ntiles = i;
    return k;
  };
  for (int i = 0; i < cap; i++) e.graphs_[key(i)] = {nullptr, ++e.graph_clock_};
  e.trim_graphs();
  CHECK((int)e.graphs_.size() == cap, "%zu of %d kept", e.graphs_.size(), cap);
  for (int i = cap; i < n; i++) e.graphs_[key(i)] = {nullptr, ++e.graph_clock_};
  for (int i = 0; i < 10; i++) e.graphs_[key(7 * i)].used = ++e.graph_clock_;   // old ones used again
  e.trim_graphs();
  CHECK((int)e.graphs_.size() == cap, "%zu of %d kept", e.graphs_.size(), n);
  for (int i = 0; i < n; i++) {
    const bool want = (i % 7 == 0 && i < 70) || i >= n - (cap - 10);
    CHECK((e.graphs_.count(key(i)) == 1) == want, "entry %d of %d", i, n);
  }
  (void)hipGetLastError();
  printf("ok kept graphs\n");
}

int main()
{
  kept_graphs();
  one_lane();
  control_block();
  lane_group_jobs();
  known_plans();
  for (int n : {1, 2, 3, 15, 16, 17, 20, 32, 33, 34, 64, 100, 128, 160, 200, 256})
    reverse_bound("survey", std::vector<ShotDev>(n, window(301, 512, 50)));
  for (int n : {5, 31, 33, 70, 119}) reverse_bound("narrow", std::vector<ShotDev>(n, window(60 + n, 300, 32)));
  for (int n : {2, 3, 4, 9}) reverse_bound("wide", std::vector<ShotDev>(n, window(1200, 768, 50)));
  for (int n : {1, 2, 4, 5}) reverse_bound("large", std::vector<ShotDev>(n, window(2048, 1024, 50)));
  std::mt19937 rng(7);
  for (int k = 0; k < 300; k++) {
    std::vector<ShotDev> ds;
    const int n = 1 + rng() % 120, nz = 60 + rng() % 700;
    for (int j = 0; j < n; j++) ds.push_back(window(40 + rng() % 900, nz, 32));
    const Plan p = plan(ds, PH_REV);
    CHECK(whole(p, n), "random %d: %d shots", k, n);
    const Plan f = plan(ds, PH_FWD);
    CHECK(whole(f, n) && (int)f.g.size() == std::min(2, n), "random %d: forward in %d groups", k, (int)f.g.size());
    reverse_bound("random", ds);
  }
  printf("ok groups of a pass\n");
  if (!g_fail) printf("all plan checks passed\n");
  return g_fail;
}
