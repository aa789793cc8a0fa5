// Elimination plan of the direct linear solve (direct.hip): host code only, no
// HIP, so it also builds into the CPU test.
//
// The Gauss-Newton matrix of a pose graph has one 6x6 block per pose and one
// per pair of poses joined by a between factor.  The plan eliminates poses
// level by level: the poses of one level are pairwise not adjacent (in the
// graph with the fill of the earlier levels), so their pivots are independent
// and a level is one launch.  While poses of degree <= 2 exist (the odometry
// chain between loop closures) a level takes an independent set of them, which
// is odd-even reduction of the chain: log2 of the longest run of levels.
// After that, and once kThinLevels of those levels had such poses in less than
// an eighth of the graph, a level takes an independent set of the poses of
// degree at most max(3 dmin, dmin + 4), smallest degree first.  (A chain seen
// from one landmark is a fan: only its two ends have degree 2, every pose
// between them 3.  Two poses a level made 1,003 levels of 10,000 poses seen
// 2,000 times and 10,001 of 20,000 poses all seen; 30 and 28 so.  Chains with
// loop closures end their degree <= 2 phase with at most 12 such levels, so
// their plans do not change.)  The exact minimum degree
// (threshold dmin) gives the least fill but, once the graph is a strip of
// cliques, eats it from its ends in long dependent chains: on a helix of
// 50,000 poses with 5,000 loop closures 1,115 levels and 330,444 update
// blocks, against 99 levels and 461,430 blocks with the relaxed threshold.
// The numeric work is small either way (0.4 M 6x6 products); the number of
// dependent levels is what a GPU pays for.
//
// A run of poses, each the parent of the one before and with one neighbour
// less (the end of the elimination: a clique loses a pose at a time), is one
// front with several pivots: its columns are the same rows, so one workgroup
// eliminates them from one copy in LDS.  The levels of the fronts are the
// heights of the merged tree: 84 -> 23 at 3,000 poses with 601 loop closures,
// 99 -> 25 at 50,000 with 5,000, 20 -> 13 for 500 planar poses with 60.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace rpgo {

// One front: s pivots and their n - s remaining neighbours, n rows of 6x6
// blocks in elimination order.  Column q of its panel holds rows q .. n-1 and
// the right-hand side as one more row of six.
struct FrontMeta {
  int32_t s, n;
  int32_t row_off;     // rows as poses in row_pose, pivots first
  int32_t child_off;   // children: fronts whose first neighbour is a pivot here
  int32_t n_child;
  int32_t map_off;     // child c's map at map_off + c * n
  int32_t orig_off;    // between factors assembled here
  int32_t n_orig;
  int64_t g_off;       // factored panel, in doubles
  int64_t u_off;       // update matrix and vector, in doubles
};

// A child's update matrix; its map gives, per row here, the child's neighbour
// index (-1: not a neighbour of the child)
struct FrontChild {
  int64_t u_off;
  int32_t d;
  int32_t pad;
};

// factor f, its block (column q, row r) and whether its Hij is the transpose
// of the block (row pose first, pivot second).  run: the number of factors of
// the block at its first one, 0 at the others.
struct FrontOrig {
  int32_t f;
  int32_t slot;  // q << 16 | r << 1 | transposed
  int32_t run;
  int32_t pad;
};

inline int64_t front_update_len(int64_t d) { return d * (d + 1) / 2 * 36 + 6 * d; }
// first panel row (of six doubles) of column q of a front of n rows; at q = s
// the rows of the whole panel
#ifdef __HIPCC__
__host__ __device__
#endif
constexpr int panel_row(int n, int q) { return 6 * (q * n - q * (q - 1) / 2) + q; }
// LDS of a front's panel and one more vector of its rows; a front takes
// pivots up to kPanelBytes
constexpr int panel_bytes(int n, int s) { return 48 * (panel_row(n, s) + n); }
constexpr int kPanelBytes = 64 * 1024;
// LDS of the backward substitution: the pivots' triangle and one vector of
// the rows
constexpr int back_bytes(int n, int s) { return 8 * (18 * s * (s + 1) + 6 * n); }

struct DirectPlan {
  int N = 0;
  int max_d = 0;                    // neighbours of the widest pivot
  int64_t u_len = 0, g_len = 0;     // doubles of all update matrices and panels
  int64_t steps = 0;                // list entries touched while eliminating, also when refused
  std::vector<int> lvl;             // level offsets into meta
  std::vector<int> lvl_bytes;       // largest panel_bytes of each level
  std::vector<int> lvl_back;        // largest back_bytes
  std::vector<int> lvl_s, lvl_n, lvl_d;  // most pivots, rows, neighbours of a front
  std::vector<FrontMeta> meta;      // by level
  std::vector<FrontChild> childs;
  std::vector<FrontOrig> origs;
  std::vector<int32_t> row_pose;
  std::vector<int32_t> maps;
  int levels() const { return (int)lvl.size() - 1; }
};

// How a level is launched: workgroups of `threads` threads, `split` of them for
// each front.
//
// Where every front of the level is small its update rows go to single lanes: a
// tile of 16x16 is larger than the whole update below three neighbours, and at
// n = 8 both take 8 us.  A wavefront a front where the level fills the chip by
// itself: 22,520 fronts 50 us; four wavefronts run a front's three chains of
// loads side by side: levels of 100 to 600 fronts 11 -> 7.8 us.
//
// Wide fronts of a narrow level share their update tiles among workgroups, each
// repeating the panel.  Sixteen wavefronts for the pivots' latency, four where
// fronts outnumber half the CUs: levels of 207 to 1,166 fronts 28-45 -> 20-26 us.
struct LevelLaunch {
  bool small;
  int threads, split;
};

inline LevelLaunch level_launch(const DirectPlan& P, int l) {
  const int n = P.lvl[l + 1] - P.lvl[l];
  if (P.lvl_n[l] <= 8) return {true, n > 4096 ? 64 : 256, 1};
  const int T = (6 * P.lvl_d[l] + 16) / 16, tiles = T * (T + 1) / 2, waves = n > 128 ? 4 : 16;
  return {false, 64 * waves, std::max(1, std::min((tiles + waves - 1) / waves, 1024 / n))};
}

// Limits of a plan: past any of them build_direct_plan returns false and the
// caller keeps its iterative solve.  Where the line lies: loop closures
// between random poses (outliers left in the graph) end in one wide clique,
// eliminated a pose a level.  LM on helices with loop closures 1/5 of the
// poses, outliers kept, direct / PCG: 2,000 poses, 50 % (widest front 122, 118
// MB of updates) 197 / 417 ms; 5,000, 10 % (162, 370 MB) 387 / 629 ms; with one
// pivot a front (wide fronts have one either way) 5,000, 20 % (223, 754 MB) 622
// / 474 ms; 10,000, 10 % (256, 1.7 GB) 803 / 611 ms.
// Graphs after PCM stay far below in width (50,000 poses with 5,000 loop
// closures: 32, 140 MB; with 10,000 58, 514 MB).
struct DirectLimits {
  int max_d = 192;                   // a front's column in LDS: 56 KB
  int64_t max_u = 256ll << 20;       // doubles of update matrices (2 GB), and
  int64_t max_u_pose = 2000;         // per pose, from u_free on
  int64_t u_free = 64ll << 20;
  int64_t max_steps = 400ll << 20;   // list entries touched while eliminating
  int64_t max_maps = 64ll << 20;
  // elimination levels: about 8 us each, forward and backward, so that these
  // cost what 300 PCG iterations of 57 us do at 50,000 poses
  int max_levels = 2048;
  // A pose with more neighbours than this is merged with all its neighbours of
  // a level at once.  A merge for each walked its whole list every time: 350 ms
  // for a star of 20,000 poses and for as many in a chain that all see one
  // pose, 2 and 7 ms so.  Shorter lists keep the merge, which is a quarter
  // faster for them; from 256 on graphs with outliers plan up to 20 % slower.
  int long_list = 512;
};

// Whether the factors hold every pose: each is joined to a prior by factors for
// which counts(f) is true.  Where they do not, a part of the graph can move as a
// whole and the undamped matrix is singular; its last pivots are rounding noise
// (up to 1e-9 of the diagonal at 50,000 poses) as large as the smallest pivots
// of regular systems, so this is decided from the graph and not from them.
template <class Counts>
bool poses_held(int N, int F, const int32_t* kind, const int32_t* fi, const int32_t* fj, Counts&& counts) {
  std::vector<int32_t> up(N);
  std::vector<char> held(N, 0);
  for (int v = 0; v < N; ++v) up[v] = v;
  const auto root = [&](int v) {
    while (up[v] != v) v = up[v] = up[up[v]];
    return v;
  };
  for (int f = 0; f < F; ++f) {
    if (!counts(f)) continue;
    const int a = root(fi[f]);
    if (kind[f] != 0) {
      held[a] = 1;
      continue;
    }
    const int b = root(fj[f]), lo = std::min(a, b);
    held[lo] = held[a] | held[b];
    up[std::max(a, b)] = lo;
  }
  for (int v = 0; v < N; ++v)
    if (up[v] == v && !held[v]) return false;
  return true;
}

namespace plan_detail {

// Sorted neighbour lists in one growing pool.
struct Lists {
  std::vector<int32_t> pool;
  std::vector<int64_t> off;
  std::vector<int32_t> len, cap;
  const int32_t* at(int v) const { return pool.data() + off[v]; }
  void assign(int v, const int32_t* src, int n) {
    if (n > cap[v]) {
      off[v] = (int64_t)pool.size();
      cap[v] = n + n / 2 + 2;
      pool.resize(pool.size() + cap[v]);
    }
    std::copy(src, src + n, pool.data() + off[v]);
    len[v] = n;
  }
};

constexpr int kThinLevels = 12;

}  // namespace plan_detail

inline bool build_direct_plan(int N, int F, const int32_t* kind, const int32_t* fi, const int32_t* fj,
                              const DirectLimits& lim, DirectPlan& P) {
  using plan_detail::kThinLevels;
  using plan_detail::Lists;
  P = DirectPlan();
  P.N = N;
  Lists A;
  A.off.resize(N);
  A.len.assign(N, 0);
  A.cap.resize(N);
  // neighbour lists, sorted and unique
  {
    std::vector<int64_t> pos(N + 1, 0);
    for (int f = 0; f < F; ++f)
      if (kind[f] == 0) {
        ++pos[fi[f] + 1];
        ++pos[fj[f] + 1];
      }
    for (int v = 0; v < N; ++v) pos[v + 1] += pos[v];
    A.pool.resize(pos[N] + 1);
    for (int v = 0; v < N; ++v) {
      A.off[v] = pos[v];
      A.cap[v] = (int32_t)(pos[v + 1] - pos[v]);
    }
    for (int f = 0; f < F; ++f)
      if (kind[f] == 0) {
        A.pool[pos[fi[f]]++] = fj[f];
        A.pool[pos[fj[f]]++] = fi[f];
      }
    for (int v = 0; v < N; ++v) {
      int32_t* a = A.pool.data() + A.off[v];
      std::sort(a, a + A.cap[v]);
      A.len[v] = (int32_t)(std::unique(a, a + A.cap[v]) - a);
    }
  }
  std::vector<int32_t> alive(N), order;
  for (int v = 0; v < N; ++v) alive[v] = v;
  order.reserve(N);
  std::vector<int32_t> mark(N, -1), elim(N, -1), seen(N, -1), stamp(N, -1), tmp, longs;
  std::vector<int32_t> bucket_off, cand;
  int64_t& steps = P.steps;
  int64_t u_len = 0;
  int thin_levels = 0;
  int32_t gen = -1;
  const int64_t max_u = std::min(lim.max_u, std::max(lim.u_free, lim.max_u_pose * N));
  for (int level = 0; !alive.empty(); ++level) {
    if (level >= lim.max_levels) return false;
    int dmin = A.len[alive[0]];
    size_t chain_poses = 0;
    int64_t degrees = 0;
    for (int v : alive) {
      dmin = std::min(dmin, (int)A.len[v]);
      degrees += A.len[v];
      chain_poses += A.len[v] <= 2;
    }
    const bool thin = dmin <= 2 && 8 * chain_poses < alive.size();
    thin_levels += thin;
    // The update matrices still to come are more than a fifth of one of the mean
    // degree for every remaining pose (a clique of them makes a third, accepted
    // graphs 0.29 and more): give up early when that is too much.  With the
    // smallest degree in its place 50,000 poses with outliers were refused after
    // twice the list entries.
    if (u_len + (int64_t)(alive.size() / 5) * front_update_len(degrees / (int64_t)alive.size()) > max_u) return false;
    const int thr = dmin <= 2 && !(thin && thin_levels > kThinLevels) ? 2 : std::max(3 * dmin, dmin + 4);
    // candidates by degree, then index (counting sort)
    bucket_off.assign(thr + 2, 0);
    for (int v : alive)
      if (A.len[v] <= thr) ++bucket_off[A.len[v] + 1];
    for (int d = 0; d <= thr; ++d) bucket_off[d + 1] += bucket_off[d];
    cand.resize(bucket_off[thr + 1]);
    for (int v : alive)
      if (A.len[v] <= thr) cand[bucket_off[A.len[v]]++] = v;
    const size_t first = order.size();
    for (int v : cand) {
      if (mark[v] == level) continue;
      mark[v] = level;
      const int32_t* a = A.at(v);
      for (int k = 0; k < A.len[v]; ++k) mark[a[k]] = level;
      order.push_back(v);
      elim[v] = level;
    }
    steps += (int64_t)alive.size();
    int level_max = 0;
    for (size_t q = first; q < order.size(); ++q) {
      const int v = order[q], d = A.len[v];
      level_max = std::max(level_max, d);
      u_len += front_update_len(d);
      if (d > lim.max_d || u_len > max_u || steps > lim.max_steps) return false;
      for (int k = 0; k < d; ++k) {
        // neighbour a: drop v, add v's other neighbours (merge of two sorted lists)
        const int a = A.at(v)[k];
        if (A.len[a] > lim.long_list) {  // once for all of the level, below
          if (seen[a] != level) longs.push_back(a);
          seen[a] = level;
          continue;
        }
        const int32_t *x = A.at(a), *y = A.at(v);
        const int nx = A.len[a], ny = d;
        tmp.clear();
        int i = 0, j = 0;
        while (i < nx || j < ny) {
          int w;
          if (j == ny || (i < nx && x[i] <= y[j])) {
            w = x[i];
            if (j < ny && y[j] == w) ++j;
            ++i;
          } else {
            w = y[j++];
          }
          if (w != v && w != a) tmp.push_back(w);
        }
        steps += nx + ny;
        A.assign(a, tmp.data(), (int)tmp.size());
      }
    }
    for (const int a : longs) {
      const int32_t* x = A.at(a);
      const int nx = A.len[a];
      tmp.clear();
      stamp[a] = ++gen;
      const auto add = [&](int w) {
        if (stamp[w] != gen) tmp.push_back(w);
        stamp[w] = gen;
      };
      steps += nx;
      for (int k = 0; k < nx; ++k) {
        if (elim[x[k]] != level) {
          add(x[k]);
          continue;
        }
        std::for_each(A.at(x[k]), A.at(x[k]) + A.len[x[k]], add);
        steps += A.len[x[k]];
      }
      if (steps > lim.max_steps) return false;
      std::sort(tmp.begin(), tmp.end());
      A.assign(a, tmp.data(), (int)tmp.size());
    }
    longs.clear();
    P.max_d = std::max(P.max_d, level_max);
    size_t keep = 0;
    for (int v : alive)
      if (elim[v] < 0) alive[keep++] = v;
    alive.resize(keep);
  }
  // neighbours as elimination positions, ascending; parents
  std::vector<int32_t>& pos = mark;
  for (int p = 0; p < N; ++p) pos[order[p]] = p;
  std::vector<int64_t> nb_off(N + 1, 0);
  for (int p = 0; p < N; ++p) nb_off[p + 1] = nb_off[p] + A.len[order[p]];
  if (nb_off[N] + N > INT32_MAX / 36) return false;
  std::vector<int32_t> nb(nb_off[N]), par(N, -1);
  for (int p = 0; p < N; ++p) {
    const int32_t* a = A.at(order[p]);
    int32_t* o = nb.data() + nb_off[p];
    const int d = A.len[order[p]];
    for (int k = 0; k < d; ++k) o[k] = pos[a[k]];
    if (d > 2) std::sort(o, o + d);
    else if (d == 2 && o[0] > o[1]) std::swap(o[0], o[1]);
    if (d > 0) par[p] = o[0];
  }
  const auto deg = [&](int p) { return (int)(nb_off[p + 1] - nb_off[p]); };
  // fronts: a pose joins its child with one neighbour more (the rows are then
  // the same), the one that ends the longest run
  std::vector<int32_t> best(N, -1), run(N, 1), next(N, -1), sn(N, -1), idx(N, 0), first_of;
  for (int p = 0; p < N; ++p) {
    if (best[p] >= 0) {
      run[p] += run[best[p]];
      next[best[p]] = p;
    }
    const int q = par[p];
    if (q >= 0 && deg(p) == deg(q) + 1 && (best[q] < 0 || run[p] > run[best[q]])) best[q] = p;
  }
  for (int p = 0; p < N; ++p) {
    if (best[p] >= 0) continue;  // not the start of a run
    for (int q = p; q >= 0;) {
      const int n = deg(q) + 1, id = (int)first_of.size();
      first_of.push_back(q);
      int s = 0;
      do {
        sn[q] = id;
        idx[q] = s++;
        q = next[q];
      } while (q >= 0 && panel_bytes(n, s + 1) <= kPanelBytes);
    }
  }
  const int M = (int)first_of.size();
  std::vector<int32_t> size(M, 0), last(M, 0), height(M, 0), at(M), n_orig(M, 0), n_child(M, 0);
  for (int p = 0; p < N; ++p) {
    ++size[sn[p]];
    last[sn[p]] = p;
  }
  int levels = 0;
  for (int p = 0; p < N; ++p) {  // a front's children end before its own last pivot
    const int g = sn[p];
    if (p != last[g]) continue;
    levels = std::max(levels, height[g] + 1);
    if (par[p] >= 0) {
      const int q = sn[par[p]];
      height[q] = std::max(height[q], height[g] + 1);
      ++n_child[q];
    }
  }
  for (int f = 0; f < F; ++f)
    if (kind[f] == 0) ++n_orig[sn[std::min(pos[fi[f]], pos[fj[f]])]];
  P.lvl.assign(levels + 1, 0);
  P.lvl_bytes.assign(levels, 0);
  P.lvl_back.assign(levels, 0);
  P.lvl_s.assign(levels, 0);
  P.lvl_n.assign(levels, 0);
  P.lvl_d.assign(levels, 0);
  for (int g = 0; g < M; ++g) ++P.lvl[height[g] + 1];
  for (int l = 0; l < levels; ++l) P.lvl[l + 1] += P.lvl[l];
  {
    std::vector<int> o(P.lvl.begin(), P.lvl.end() - 1);
    for (int g = 0; g < M; ++g) at[g] = o[height[g]]++;
  }
  P.meta.resize(M);
  for (int g = 0; g < M; ++g) {
    FrontMeta& m = P.meta[at[g]];
    m = FrontMeta{};
    m.s = size[g];
    m.n = deg(first_of[g]) + 1;
    m.n_child = n_child[g];
    m.n_orig = n_orig[g];
    m.row_off = first_of[g];  // replaced below
  }
  int64_t rows = 0, maps = 0, childs = 0, origs = 0;
  for (int g = 0, l = 0; g < M; ++g) {
    FrontMeta& m = P.meta[g];
    while (g >= P.lvl[l + 1]) ++l;
    const int p = m.row_off, d = m.n - m.s;
    m.row_off = (int32_t)rows;
    m.child_off = (int32_t)childs;
    m.map_off = (int32_t)maps;
    m.orig_off = (int32_t)origs;
    m.g_off = P.g_len;
    m.u_off = P.u_len;
    rows += m.n;
    maps += (int64_t)m.n_child * m.n;
    childs += m.n_child;
    origs += m.n_orig;
    P.g_len += 6ll * panel_row(m.n, m.s);
    P.u_len += front_update_len(d);
    if (maps > lim.max_maps) return false;
    P.lvl_bytes[l] = std::max(P.lvl_bytes[l], panel_bytes(m.n, m.s));
    P.lvl_back[l] = std::max(P.lvl_back[l], back_bytes(m.n, m.s));
    P.lvl_d[l] = std::max(P.lvl_d[l], d);
    P.lvl_s[l] = std::max(P.lvl_s[l], m.s);
    P.lvl_n[l] = std::max(P.lvl_n[l], m.n);
    P.row_pose.push_back(order[p]);
    for (int64_t k = nb_off[p]; k < nb_off[p + 1]; ++k) P.row_pose.push_back(order[nb[k]]);
  }
  // children and row maps (in the order of the children's first pivots)
  P.childs.resize(childs);
  P.maps.resize(maps);
  std::vector<int32_t>& fill = n_child;
  std::fill(fill.begin(), fill.end(), 0);
  for (int g = 0; g < M; ++g) {
    const int c = last[g], dc = deg(c);
    if (dc == 0) continue;
    const int q = sn[par[c]];
    const FrontMeta& m = P.meta[at[q]];
    const int k = fill[q]++;
    P.childs[m.child_off + k] = FrontChild{P.meta[at[g]].u_off, dc, 0};
    int32_t* map = P.maps.data() + m.map_off + (int64_t)k * m.n;
    const int32_t *x = nb.data() + nb_off[c], *y = nb.data() + nb_off[first_of[q]];
    int j = 0;  // the child's neighbours are a subset of the rows
    for (int r = 0; r < m.n; ++r) {
      const int row = r == 0 ? first_of[q] : y[r - 1];
      map[r] = j < dc && x[j] == row ? j++ : -1;
    }
    if (j != dc) return false;  // not reached: fill makes them one
  }
  // between factors, assembled at the endpoint eliminated first
  P.origs.resize(origs);
  std::fill(n_orig.begin(), n_orig.end(), 0);
  for (int f = 0; f < F; ++f) {
    if (kind[f] != 0) continue;
    const int a = pos[fi[f]], b = pos[fj[f]], lo = std::min(a, b), hi = std::max(a, b), g = sn[lo];
    const int32_t *y = nb.data() + nb_off[first_of[g]], *e = nb.data() + nb_off[first_of[g] + 1];
    const int r = sn[hi] == g ? idx[hi] : (int)(std::lower_bound(y, e, hi) - y) + 1;
    // the block has row-pose rows and pivot columns: Hij (rows i, columns j)
    // is its transpose when the pivot is key i
    P.origs[P.meta[at[g]].orig_off + n_orig[g]++] = FrontOrig{f, idx[lo] << 16 | r << 1 | (a < b ? 1 : 0), 1, 0};
  }
  for (int g = 0; g < M; ++g) {
    const FrontMeta& m = P.meta[g];
    if (m.n_orig < 2) continue;
    FrontOrig* o = P.origs.data() + m.orig_off;
    std::sort(o, o + m.n_orig, [](const FrontOrig& a, const FrontOrig& b) {
      return (a.slot >> 1) != (b.slot >> 1) ? (a.slot >> 1) < (b.slot >> 1) : a.f < b.f;
    });
    for (int i = 0, j; i < m.n_orig; i = j) {
      for (j = i + 1; j < m.n_orig && (o[j].slot >> 1) == (o[i].slot >> 1); ++j) o[j].run = 0;
      o[i].run = j - i;
    }
  }
  return true;
}

}  // namespace rpgo
