// Device allocations that fail inside a solve: the buffers of the direct linear
// solve are optional, so the solve goes on with the PCG; those the solve cannot
// do without give RPGO_ERR_NOMEM.  hipMalloc is interposed: the armed call asks
// the runtime for more than any card has, so its error state is the real one.
#include <dlfcn.h>

#include "harness.h"
#include "rpgo_hip.h"

namespace {
int g_calls = 0, g_fail_at = -1;
}

extern "C" int hipMalloc(void** p, size_t n) {
  using Fn = int (*)(void**, size_t);
  static const Fn real = reinterpret_cast<Fn>(dlsym(RTLD_NEXT, "hipMalloc"));
  return real(p, ++g_calls == g_fail_at ? size_t(1) << 60 : n);
}

namespace {

// a chain of N poses a metre apart with loop closures and a prior
struct Graph {
  std::vector<double> poses, meas, info;
  std::vector<int32_t> kind, i, j;
  rpgo_solve_problem pr{};
};

Graph make_graph(int N) {
  Graph g;
  const auto pose = [](std::vector<double>& v, double x, double y) {
    for (double e : {1., 0., 0., 0., 1., 0., 0., 0., 1., x, y, 0.}) v.push_back(e);
  };
  const auto factor = [&](int kind, int a, int b, double x, double y) {
    g.kind.push_back(kind);
    g.i.push_back(a);
    g.j.push_back(b);
    pose(g.meas, x, y);
    for (int e = 0; e < 36; ++e) g.info.push_back(e % 7 ? 0.0 : 100.0);
  };
  for (int k = 0; k < N; ++k) pose(g.poses, k + 0.1 * std::sin(k), 0.1 * std::cos(3 * k));
  for (int k = 0; k + 1 < N; ++k) factor(RPGO_FACTOR_BETWEEN, k, k + 1, 1 + 0.01 * std::sin(5 * k), 0.0);
  for (int k = 0; k + 20 < N; k += 7) factor(RPGO_FACTOR_BETWEEN, k, k + 20, 20.0, 0.01 * std::cos(k));
  factor(RPGO_FACTOR_PRIOR, 0, 0, 0.0, 0.0);
  g.pr.n_poses = N;
  g.pr.n_factors = (int)g.kind.size();
  g.pr.poses = g.poses.data();
  g.pr.kind = g.kind.data();
  g.pr.key_i = g.i.data();
  g.pr.key_j = g.j.data();
  g.pr.measured = g.meas.data();
  g.pr.information = g.info.data();
  return g;
}

struct Result {
  int rc = 0, calls = 0;
  std::vector<double> poses;
  rpgo_solve_report rep{};
};

// one solve whose fail_at'th allocation fails (0: none)
Result solve(rpgo_ctx* ctx, const Graph& g, const rpgo_solve_params& prm, int fail_at) {
  Result r;
  r.poses.resize(12 * (size_t)g.pr.n_poses);
  g_calls = 0;
  g_fail_at = fail_at > 0 ? fail_at : -1;
  r.rc = rpgo_solve(ctx, &g.pr, &prm, r.poses.data(), nullptr, &r.rep);
  g_fail_at = -1;
  r.calls = g_calls;
  return r;
}

double diff(const Result& a, const Result& b) {
  double d = 0.0;
  for (size_t k = 0; k < a.poses.size(); ++k) d = std::max(d, std::fabs(a.poses[k] - b.poses[k]));
  return d;
}

}  // namespace

TEST(AllocFailure, DirectSolveFallsBackToPcg) {
  const Graph g = make_graph(150);
  rpgo_solve_params prm;
  rpgo_solve_params_default(&prm);
  prm.pcg_rel_tol = 1e-9;
  const auto fresh = [] {
    rpgo_ctx* c = nullptr;
    if (rpgo_ctx_create(0, 0, &c) != RPGO_OK) c = nullptr;
    return c;
  };
  // allocations of the problem alone (no linear step), and of a direct solve
  rpgo_solve_params none = prm;
  none.lm_max_iterations = 0;
  none.pcg_segment = 16;
  rpgo_ctx* c = fresh();
  EXPECT(c != nullptr);
  if (!c) return;
  const int problem = solve(c, g, none, 0).calls;
  rpgo_ctx_destroy(c);
  c = fresh();
  const Result ref = solve(c, g, prm, 0);
  rpgo_ctx_destroy(c);
  EXPECT(ref.rc == RPGO_OK && ref.calls > problem);
  EXPECT(ref.rep.pcg_iterations <= 4 * ref.rep.linearizations);  // the direct path
  std::printf("  %d allocations, %d of them the direct solve's\n", ref.calls, ref.calls - problem);
  for (int k = problem + 1; k <= ref.calls; ++k) {
    std::printf("  allocation %d fails\n", k);
    std::fflush(stdout);
    c = fresh();
    const Result a = solve(c, g, prm, k);
    EXPECT(a.rc == RPGO_OK);
    EXPECT(a.rep.pcg_iterations > 4 * a.rep.linearizations);  // the PCG
    EXPECT(diff(a, ref) < 1e-6);  // steps agree to 1e-9 of their right-hand side
    const Result b = solve(c, g, prm, 0);  // room again: direct, the same bits
    EXPECT(b.rc == RPGO_OK && diff(b, ref) == 0.0);
    rpgo_ctx_destroy(c);
  }
  for (int k : {1, problem}) {
    c = fresh();
    EXPECT(solve(c, g, prm, k).rc == RPGO_ERR_NOMEM);
    rpgo_ctx_destroy(c);
  }
}

RPGO_TEST_MAIN
