// CPU check of the direct solve's elimination plan (csrc/direct_plan.h): the
// factorization the plan describes, carried out on the host with every index
// bounds-checked, solves random block systems of all the shapes the solver
// takes (chains in any order, repeated and reversed factors, loop closures,
// stars, disconnected poses, cliques), against a dense Cholesky solve.
#include <random>

#include "../../kimera-rpgo_amd/csrc/direct_plan.h"
#include "harness.h"

using namespace rpgo;

namespace {

struct Sys {
  int N;
  std::vector<int32_t> kind, fi, fj;
  std::vector<std::vector<double>> D, H;  // 36 per pose, 36 per factor
  std::vector<double> b;
};

Sys random_system(int N, const std::vector<std::pair<int, int>>& edges, unsigned seed) {
  std::mt19937 rng(seed);
  std::normal_distribution<double> g;
  Sys s;
  s.N = N;
  s.D.assign(N, std::vector<double>(36, 0.0));
  s.b.resize(6 * (size_t)N);
  for (auto& v : s.b) v = g(rng);
  for (int k = 0; k < N; ++k)
    for (int i = 0; i < 6; ++i) s.D[k][i * 7] = 0.5;
  for (auto& e : edges) {
    s.kind.push_back(0);
    s.fi.push_back(e.first);
    s.fj.push_back(e.second);
    double J[2][36];
    for (auto& A : J)
      for (double& v : A) v = g(rng);
    auto prod = [&](const double* A, const double* B) {  // A^T B
      std::vector<double> o(36, 0.0);
      for (int i = 0; i < 6; ++i)
        for (int j = 0; j < 6; ++j)
          for (int m = 0; m < 6; ++m) o[i * 6 + j] += A[m * 6 + i] * B[m * 6 + j];
      return o;
    };
    const auto ii = prod(J[0], J[0]), jj = prod(J[1], J[1]);
    for (int q = 0; q < 36; ++q) {
      s.D[e.first][q] += ii[q];
      s.D[e.second][q] += jj[q];
    }
    s.H.push_back(prod(J[0], J[1]));
    if (s.kind.size() % 7 == 3) {  // a prior now and then: no off-diagonal block
      s.kind.push_back(1);
      s.fi.push_back(e.first);
      s.fj.push_back(e.first);
      s.H.push_back(std::vector<double>(36, 1e300));
    }
  }
  return s;
}

std::vector<double> dense_solve(const Sys& s) {
  const int n = 6 * s.N;
  std::vector<double> A((size_t)n * n, 0.0), x(s.b);
  for (int k = 0; k < s.N; ++k)
    for (int q = 0; q < 36; ++q) A[(size_t)(6 * k + q / 6) * n + 6 * k + q % 6] += s.D[k][q];
  for (size_t f = 0; f < s.kind.size(); ++f)
    if (s.kind[f] == 0)
      for (int q = 0; q < 36; ++q) {
        const int r = 6 * s.fi[f] + q / 6, c = 6 * s.fj[f] + q % 6;
        A[(size_t)r * n + c] += s.H[f][q];
        A[(size_t)c * n + r] += s.H[f][q];
      }
  for (int c = 0; c < n; ++c) {
    for (int k = 0; k < c; ++k)
      for (int r = c; r < n; ++r) A[(size_t)r * n + c] -= A[(size_t)r * n + k] * A[(size_t)c * n + k];
    const double p = std::sqrt(A[(size_t)c * n + c]);
    for (int r = c; r < n; ++r) A[(size_t)r * n + c] /= p;
  }
  for (int r = 0; r < n; ++r) {
    for (int k = 0; k < r; ++k) x[r] -= A[(size_t)r * n + k] * x[k];
    x[r] /= A[(size_t)r * n + r];
  }
  for (int r = n - 1; r >= 0; --r) {
    for (int k = r + 1; k < n; ++k) x[r] -= A[(size_t)k * n + r] * x[k];
    x[r] /= A[(size_t)r * n + r];
  }
  return x;
}

// The plan's factorization and both substitutions, front by front
std::vector<double> plan_solve(const Sys& s, const DirectPlan& P, int& bad) {
  std::vector<double> U(P.u_len, 0.0), G(P.g_len, 0.0), x(6 * (size_t)s.N, 0.0);
  for (size_t g = 0; g < P.meta.size(); ++g) {
    const FrontMeta& m = P.meta[g];
    const int n = m.n, np = m.s, d = n - np;
    // dense front: n + 1 block rows (the last, one row, the right-hand side)
    const int w = 6 * n;
    std::vector<double> A((size_t)(w + 1) * w, 0.0);
    for (int q = 0; q < np; ++q) {
      const int pose = P.row_pose.at(m.row_off + q);
      for (int e = 0; e < 36; ++e) A[(size_t)(6 * q + e / 6) * w + 6 * q + e % 6] += s.D.at(pose)[e];
      for (int i = 0; i < 6; ++i) A[(size_t)w * w + 6 * q + i] += s.b[6 * pose + i];
    }
    for (int o = 0; o < m.n_orig; ++o) {
      const FrontOrig& lead = P.origs.at(m.orig_off + o);
      for (int k = 0; k < lead.run; ++k) {
        const FrontOrig& a = P.origs.at(m.orig_off + o + k);
        const int q = a.slot >> 16, R = (a.slot >> 1) & 0x7fff;
        if ((a.slot >> 1) != (lead.slot >> 1) || q >= np || R <= q || R >= n || (k > 0 && a.run != 0)) { ++bad; continue; }
        const int row = P.row_pose.at(m.row_off + R), piv = P.row_pose.at(m.row_off + q);
        if ((a.slot & 1) ? (s.fi.at(a.f) != piv || s.fj.at(a.f) != row) : (s.fi.at(a.f) != row || s.fj.at(a.f) != piv)) ++bad;
        for (int e = 0; e < 36; ++e)
          A[(size_t)(6 * R + e / 6) * w + 6 * q + e % 6] += s.H.at(a.f)[(a.slot & 1) ? (e % 6) * 6 + e / 6 : e];
      }
      if (lead.run > 0 && o + lead.run < m.n_orig && P.origs.at(m.orig_off + o + lead.run).run == 0) ++bad;
    }
    for (int c = 0; c < m.n_child; ++c) {
      const FrontChild& ch = P.childs.at(m.child_off + c);
      const int64_t vec = ch.u_off + (int64_t)ch.d * (ch.d + 1) / 2 * 36;
      for (int k = 0; k < n; ++k) {
        const int pk = P.maps.at(m.map_off + c * n + k);
        if (pk < 0) continue;
        if (pk >= ch.d) { ++bad; continue; }
        for (int i = 0; i < 6; ++i) A[(size_t)w * w + 6 * k + i] += U.at(vec + 6 * pk + i);
        for (int l = 0; l <= k; ++l) {
          const int pl = P.maps.at(m.map_off + c * n + l);
          if (pl < 0) continue;
          if (pl > pk) { ++bad; continue; }
          for (int e = 0; e < 36; ++e)
            A[(size_t)(6 * k + e / 6) * w + 6 * l + e % 6] += U.at(ch.u_off + 36 * ((int64_t)pk * (pk + 1) / 2 + pl) + e);
        }
      }
    }
    // eliminate the pivots' columns from the lower triangle and the last row
    for (int c = 0; c < 6 * np; ++c) {
      const double p = std::sqrt(A[(size_t)c * w + c]);
      for (int r = c; r <= w; ++r) A[(size_t)r * w + c] /= p;
      for (int c2 = c + 1; c2 < w; ++c2)
        for (int r = c2; r <= w; ++r) A[(size_t)r * w + c2] -= A[(size_t)r * w + c] * A[(size_t)c2 * w + c];
    }
    for (int q = 0; q < np; ++q)
      for (int r = 6 * q; r <= w; ++r)
        for (int j = 0; j < 6; ++j) G.at(m.g_off + 6 * (panel_row(n, q) + r - 6 * q) + j) = A[(size_t)r * w + 6 * q + j];
    for (int k = 0; k < d; ++k) {
      for (int l = 0; l <= k; ++l)
        for (int e = 0; e < 36; ++e)
          U.at(m.u_off + 36 * ((int64_t)k * (k + 1) / 2 + l) + e) = A[(size_t)(6 * (np + k) + e / 6) * w + 6 * (np + l) + e % 6];
      for (int i = 0; i < 6; ++i) U.at(m.u_off + 36 * ((int64_t)d * (d + 1) / 2) + 6 * k + i) = A[(size_t)w * w + 6 * (np + k) + i];
    }
  }
  for (size_t g = P.meta.size(); g-- > 0;) {
    const FrontMeta& m = P.meta[g];
    const int n = m.n;
    for (int c = 6 * m.s - 1; c >= 0; --c) {
      const int q = c / 6, j = c % 6;
      const auto at = [&](int r) { return G.at(m.g_off + 6 * (panel_row(n, q) + r - 6 * q) + j); };
      double v = at(6 * n);
      for (int r = c + 1; r < 6 * n; ++r) v -= at(r) * x.at(6 * P.row_pose.at(m.row_off + r / 6) + r % 6);
      x[6 * P.row_pose[m.row_off + q] + j] = v / at(c);
    }
  }
  return x;
}

int check(const char* what, int N, const std::vector<std::pair<int, int>>& edges, unsigned seed, int& rpgo_failures_,
          const DirectLimits& lim = DirectLimits()) {
  const Sys s = random_system(N, edges, seed);
  DirectPlan P;
  EXPECT(build_direct_plan(N, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
  // every pose a pivot once, levels contiguous, no factor between two fronts
  // of a level, every front within the level's bounds and the LDS
  std::vector<int> level(N, -1), front(N, -1);
  int seen = 0;
  for (int l = 0; l < P.levels(); ++l)
    for (int p = P.lvl[l]; p < P.lvl[l + 1]; ++p) {
      const FrontMeta& m = P.meta.at(p);
      EXPECT(m.s >= 1 && m.s <= m.n && m.s <= P.lvl_s[l] && m.n <= P.lvl_n[l] && m.n - m.s <= P.lvl_d[l]);
      EXPECT(panel_bytes(m.n, m.s) <= P.lvl_bytes[l] && P.lvl_bytes[l] <= kPanelBytes);
      // with 2 KB of its own the backward kernel keeps within the LDS too; a
      // thread per pivot component
      EXPECT(back_bytes(m.n, m.s) <= P.lvl_back[l] && P.lvl_back[l] + 2048 <= kPanelBytes && 6 * m.s <= 256);
      for (int q = 0; q < m.s; ++q) {
        const int pose = P.row_pose.at(m.row_off + q);
        EXPECT(level.at(pose) < 0);
        level[pose] = l;
        front[pose] = p;
        ++seen;
      }
    }
  EXPECT(seen == N && P.lvl.back() == (int)P.meta.size());
  for (auto& e : edges) EXPECT(level[e.first] != level[e.second] || front[e.first] == front[e.second]);
  int bad = 0;
  const auto x = plan_solve(s, P, bad), ref = dense_solve(s);
  EXPECT(bad == 0);
  double err = 0.0, nrm = 0.0;
  for (size_t k = 0; k < x.size(); ++k) {
    err = std::max(err, std::fabs(x[k] - ref[k]));
    nrm = std::max(nrm, std::fabs(ref[k]));
  }
  std::printf("  %s N=%d levels=%d max_d=%d err %.1e of %.1e\n", what, N, P.levels(), P.max_d, err, nrm);
  // condition numbers here stay below about 1e5: 1e5 * 6 N * 2^-53 < 1e-7
  EXPECT(err <= 1e-7 * (nrm + 1.0));
  return P.levels();
}

std::vector<std::pair<int, int>> chain(int N) {
  std::vector<std::pair<int, int>> e;
  for (int k = 0; k + 1 < N; ++k) e.push_back({k, k + 1});
  return e;
}

// a chain of N poses and pose N, seen from `seen` of them, evenly spread
std::vector<std::pair<int, int>> chain_hub(int N, int seen) {
  auto e = chain(N);
  for (int k = 0; k < seen; ++k) e.push_back({(int)((int64_t)k * N / seen), N});
  return e;
}

// laps of `lap` poses, joined at every `every`th pose
std::vector<std::pair<int, int>> laps(int N, int lap, int every) {
  auto e = chain(N);
  for (int k = 0; k + lap < N; k += every) e.push_back({k + lap, k});
  return e;
}

bool plan(int N, const std::vector<std::pair<int, int>>& edges, const DirectLimits& lim, DirectPlan& P) {
  std::vector<int32_t> kind(edges.size(), 0), fi, fj;
  for (auto& e : edges) {
    fi.push_back(e.first);
    fj.push_back(e.second);
  }
  return build_direct_plan(N, (int)edges.size(), kind.data(), fi.data(), fj.data(), lim, P);
}

}  // namespace

TEST(DirectPlan, Chains) {
  for (int N : {1, 2, 3, 4, 7, 8, 63, 64, 65, 200}) check("chain", N, chain(N), 10 + N, rpgo_failures_);
  // odd-even reduction: logarithmic in the length
  EXPECT(check("chain", 256, chain(256), 3, rpgo_failures_) <= 12);
}

TEST(DirectPlan, OrdersAndRepeats) {
  std::mt19937 rng(1);
  for (int t = 0; t < 12; ++t) {
    const int N = 2 + (int)(rng() % 70);
    std::vector<int> name(N);
    for (int k = 0; k < N; ++k) name[k] = k;
    std::shuffle(name.begin(), name.end(), rng);
    std::vector<std::pair<int, int>> e;
    for (auto& c : chain(N)) {
      const int a = name[c.first], b = name[c.second];
      if (rng() % 2) e.push_back({a, b});
      else e.push_back({b, a});
      if (rng() % 3 == 0) e.push_back({b, a});  // repeated, other direction
    }
    for (int q = 0; q < N / 4; ++q) {
      const int a = (int)(rng() % N), b = (int)(rng() % N);
      if (a != b) e.push_back({a, b});
    }
    check("shuffled", N, e, 50 + t, rpgo_failures_);
  }
}

TEST(DirectPlan, Shapes) {
  std::vector<std::pair<int, int>> star, clique, two, none;
  for (int k = 1; k < 60; ++k) star.push_back(k % 2 ? std::make_pair(0, k) : std::make_pair(k, 0));
  for (int a = 0; a < 20; ++a)
    for (int b = a + 1; b < 20; ++b) clique.push_back({b, a});
  for (int k = 0; k < 40; ++k)
    if (k != 20) two.push_back({k, k + 1});  // two chains, one of them with a loop
  two.push_back({5, 17});
  check("star", 60, star, 1, rpgo_failures_);
  check("clique", 20, clique, 2, rpgo_failures_);
  for (int a = 20; a < 45; ++a)  // too wide for one panel
    for (int b = 0; b < a; ++b) clique.push_back({b, a});
  EXPECT(check("clique", 45, clique, 6, rpgo_failures_) > 1);
  check("two chains", 41, two, 3, rpgo_failures_);
  check("no factors", 5, none, 4, rpgo_failures_);
  check("laps", 120, laps(120, 12, 3), 5, rpgo_failures_);
}

// Poses around one shared pose: the levels stay logarithmic in the chain (a fan
// halves per level once the first thin levels are past), and the plan solves
TEST(DirectPlan, ChainAndHub) {
  EXPECT(check("hub", 101, chain_hub(100, 100), 7, rpgo_failures_) <= 12 + 10);
  EXPECT(check("hub", 201, chain_hub(200, 60), 8, rpgo_failures_) <= 12 + 12);
  const int sizes[4][2] = {{3000, 300}, {10000, 2000}, {20000, 20000}, {50000, 5000}};
  for (auto& z : sizes) {
    DirectPlan P;
    EXPECT(plan(z[0] + 1, chain_hub(z[0], z[1]), DirectLimits(), P));
    std::printf("  hub %d/%d: %d levels\n", z[1], z[0], P.levels());
    // odd-even reduction to the poses that see the hub, the thin levels, and
    // halving of the fan: at most log2(N) + 12 + log2(N) with a few to spare
    EXPECT(P.levels() <= 12 + 2 * 16 + 4);
  }
}

// The work of planning is linear in the poses around a shared pose (a few
// list entries a factor and level), not quadratic; lists above the length from
// which a level's merges are joined plan the same solve
TEST(DirectPlan, LongLists) {
  std::vector<std::pair<int, int>> star, two;
  for (int k = 0; k < 20000; ++k) star.push_back({k % 2 ? k : 20000, k % 2 ? 20000 : k});
  DirectLimits lim;
  lim.max_steps = 100 * 20000;  // one merge a pose took 2e8
  DirectPlan P;
  EXPECT(plan(20001, star, lim, P) && P.levels() == 2);
  EXPECT(plan(20001, chain_hub(20000, 20000), lim, P));
  // every pose with more than `long_list` neighbours takes the joined merge
  std::vector<std::pair<int, int>> clique;
  two = chain(90);  // two hubs, each seen from all
  for (int k = 0; k < 90; ++k)
    for (int h : {90, 91}) two.push_back({h, k});
  for (int a = 0; a < 30; ++a)
    for (int b = a + 1; b < 30; ++b) clique.push_back({b, a});
  for (int l : {0, 1, 3, 8, 40}) {
    lim = DirectLimits();
    lim.long_list = l;
    const auto hub = chain_hub(120, 90);
    const int direct = check("two hubs", 92, two, 13, rpgo_failures_);
    EXPECT(check("two hubs", 92, two, 13, rpgo_failures_, lim) == direct);
    EXPECT(check("hub", 121, hub, 14, rpgo_failures_, lim) == check("hub", 121, hub, 14, rpgo_failures_));
    check("clique", 30, clique, 15, rpgo_failures_, lim);
    DirectPlan A, B;  // the same plan
    EXPECT(plan(121, hub, lim, A) && plan(121, hub, DirectLimits(), B));
    EXPECT(A.row_pose == B.row_pose && A.maps == B.maps && A.lvl == B.lvl && A.u_len == B.u_len);
  }
}

// The graph that test_direct_gpu.py solves to run every launch of the front
// kernels has levels of each kind
TEST(DirectPlan, LaunchShapes) {
  DirectPlan P;
  EXPECT(plan(20000, laps(20000, 100, 5), DirectLimits(), P));
  int small64 = 0, small256 = 0, front256 = 0, front1024 = 0, split256 = 0, split1024 = 0;
  for (int l = 0; l < P.levels(); ++l) {
    const LevelLaunch h = level_launch(P, l);
    EXPECT(h.split >= 1 && (!h.small || h.split == 1));
    ++(h.small ? (h.threads == 64 ? small64 : small256) : h.threads == 256 ? front256 : front1024);
    if (!h.small && h.split > 1) ++(h.threads == 256 ? split256 : split1024);
    std::printf("  %d fronts of up to %d rows, %d neighbours: %s%d x%d\n", P.lvl[l + 1] - P.lvl[l], P.lvl_n[l],
                P.lvl_d[l], h.small ? "small " : "", h.threads, h.split);
  }
  EXPECT(small64 > 0 && small256 > 0 && front256 > 0 && front1024 > 0 && split256 > 0 && split1024 > 0);
}

// A graph that fills in too much is given up early: random loop closures on a
// fifth of the poses of a chain end in one clique of several hundred
TEST(DirectPlan, RefusedEarly) {
  std::mt19937 rng(3);
  auto e = chain(20000);
  for (int k = 0; k < 4000; ++k) {
    const int a = (int)(rng() % 20000), b = (int)(rng() % 20000);
    if (a != b) e.push_back({a, b});
  }
  DirectPlan P;
  EXPECT(!plan(20000, e, DirectLimits(), P));
  std::printf("  refused after %lld list entries\n", (long long)P.steps);
  EXPECT(P.steps < 100 * 20000);  // 81 a pose; 140 with the smallest degree as the estimate
}

TEST(DirectPlan, PosesHeld) {
  // a chain 0-1-2, a pair 3-4, poses 5 (prior) and 6 alone; factor 7 joins 4 to 2
  const std::vector<int32_t> kind = {0, 0, 0, 1, 1, 1, 1, 0}, fi = {0, 2, 3, 1, 5, 4, 6, 4}, fj = {1, 1, 4, 1, 5, 4, 6, 2};
  const auto held = [&](std::vector<int> off) {
    return poses_held(7, 8, kind.data(), fi.data(), fj.data(),
                      [&](int f) { return std::find(off.begin(), off.end(), f) == off.end(); });
  };
  EXPECT(held({}));
  EXPECT(!held({6}));      // pose 6 without its prior
  EXPECT(!held({4}));
  EXPECT(held({3}));       // the chain by factor 7
  EXPECT(held({5}));       // the pair by factor 7
  EXPECT(held({7}));
  EXPECT(!held({3, 7}));   // the chain by nothing
  EXPECT(!held({5, 7}));
  EXPECT(!held({0}));      // pose 0 cut off
  EXPECT(!held({2, 5}));   // pose 3 cut off
  const int32_t none = 0;
  EXPECT(!poses_held(1, 0, &none, &none, &none, [](int) { return true; }));
  std::vector<int32_t> k(50000, 0), i(50000), j(50000);  // a long chain in order and reversed, prior last
  for (int f = 0; f < 49999; ++f) i[f] = f, j[f] = f + 1;
  k[49999] = 1, i[49999] = j[49999] = 49999;
  EXPECT(poses_held(50000, 50000, k.data(), i.data(), j.data(), [](int) { return true; }));
  EXPECT(!poses_held(50000, 50000, k.data(), i.data(), j.data(), [](int f) { return f != 777; }));
  EXPECT(!poses_held(50000, 50000, k.data(), i.data(), j.data(), [](int f) { return f != 49999; }));
  std::reverse(i.begin(), i.end() - 1);
  std::reverse(j.begin(), j.end() - 1);
  EXPECT(poses_held(50000, 50000, k.data(), j.data(), i.data(), [](int) { return true; }));
  EXPECT(!poses_held(50000, 50000, k.data(), j.data(), i.data(), [](int f) { return f != 49999; }));
}

TEST(DirectPlan, Limits) {
  std::vector<std::pair<int, int>> clique;
  for (int a = 0; a < 20; ++a)
    for (int b = a + 1; b < 20; ++b) clique.push_back({b, a});
  const Sys s = random_system(20, clique, 2);
  DirectPlan P;
  DirectLimits lim;
  lim.max_d = 18;
  EXPECT(!build_direct_plan(20, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
  lim.max_d = 19;
  EXPECT(build_direct_plan(20, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
  lim.max_levels = 19;  // a pose a level
  EXPECT(!build_direct_plan(20, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
  lim.max_levels = 20;
  EXPECT(build_direct_plan(20, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
  lim.max_u = -1;  // the limit counts every pivot's update by itself
  for (int d = 0; d < 20; ++d) lim.max_u += front_update_len(d);
  EXPECT(!build_direct_plan(20, (int)s.kind.size(), s.kind.data(), s.fi.data(), s.fj.data(), lim, P));
}

RPGO_TEST_MAIN
