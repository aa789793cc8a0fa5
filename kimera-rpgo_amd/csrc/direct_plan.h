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
// After that a level takes an independent set of the poses of degree at most
// max(3 dmin, dmin + 4), smallest degree first.  The exact minimum degree
// (threshold dmin) gives the least fill but, once the graph is a strip of
// cliques, eats it from its ends in long dependent chains: on a helix of
// 50,000 poses with 5,000 loop closures 1,148 levels and 320,187 update
// blocks, against 83 levels and 445,827 blocks with the relaxed threshold.
// The numeric work is small either way (0.4 M 6x6 products); the number of
// dependent levels is what a GPU pays for.
#pragma once

#include <algorithm>
#include <cstdint>
#include <vector>

namespace rpgo {

// One eliminated pose.  Its front is the pose itself (position 0) and its d
// remaining neighbours (positions 1 .. d, in elimination order).
struct FrontMeta {
  int32_t pose;
  int32_t d;
  int32_t nb_off;      // neighbours in nb_pose; its G blocks start at 36 * nb_off
  int32_t child_off;   // children: fronts whose first neighbour is this pose
  int32_t n_child;
  int32_t orig_off;    // between factors assembled here
  int32_t n_orig;
  int32_t pad;
  int64_t u_off;       // update matrix and vector, in doubles
};

// A child's update matrix and the map from this front's positions to the
// child's neighbour indices (-1: not a neighbour of the child)
struct FrontChild {
  int64_t u_off;
  int32_t map_off;
  int32_t d;
};

// factor f, its block's position in the front and whether its Hij is the
// transpose of the block (neighbour rows, pivot columns)
struct FrontOrig {
  int32_t f;
  int32_t slot_t;  // 2 * position + transposed
};

inline int64_t front_update_len(int64_t d) { return d * (d + 1) / 2 * 36 + 6 * d; }

struct DirectPlan {
  int N = 0;
  int max_d = 0;
  int64_t u_len = 0;                // doubles of all update matrices
  std::vector<int> lvl;             // level offsets into meta
  std::vector<int> lvl_max_d;       // largest front of each level
  std::vector<FrontMeta> meta;      // in elimination order
  std::vector<FrontChild> childs;
  std::vector<FrontOrig> origs;
  std::vector<int32_t> nb_pose;     // neighbours as poses
  std::vector<int32_t> maps;
  int levels() const { return (int)lvl.size() - 1; }
};

// Limits of a plan: past any of them build_direct_plan returns false and the
// caller keeps its iterative solve.  Where the line lies: loop closures
// between random poses (outliers left in the graph) end in one wide clique,
// eliminated a pose a level.  LM on helices with loop closures 1/5 of the
// poses, outliers kept, direct / PCG: 2,000 poses, 50 % (widest front 122, 118
// MB of updates) 233 / 419 ms; 5,000, 10 % (162, 370 MB) 465 / 626 ms; 5,000,
// 20 % (223, 754 MB) 622 / 474 ms; 10,000, 10 % (256, 1.7 GB) 803 / 611 ms.
// Graphs after PCM stay far below in width (50,000 poses: 26, 135 MB; with
// 10,000 loop closures 58, 514 MB).
struct DirectLimits {
  int max_d = 192;                   // a front's column in LDS: 56 KB
  int64_t max_u = 256ll << 20;       // doubles of update matrices (2 GB), and
  int64_t max_u_pose = 2000;         // per pose, from u_free on
  int64_t u_free = 64ll << 20;
  int64_t max_steps = 400ll << 20;   // list entries touched while eliminating
  int64_t max_maps = 64ll << 20;
};

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

}  // namespace plan_detail

inline bool build_direct_plan(int N, int F, const int32_t* kind, const int32_t* fi, const int32_t* fj,
                              const DirectLimits& lim, DirectPlan& P) {
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
  std::vector<int32_t> mark(N, -1), elim(N, -1), tmp;
  std::vector<int32_t> bucket_off, cand;
  int64_t steps = 0, u_len = 0;
  const int64_t max_u = std::min(lim.max_u, std::max(lim.u_free, lim.max_u_pose * N));
  P.lvl.push_back(0);
  for (int level = 0; !alive.empty(); ++level) {
    int dmin = A.len[alive[0]];
    for (int v : alive) dmin = std::min(dmin, (int)A.len[v]);
    // the fill still to come is more than a quarter of what the remaining
    // poses' present degree would make: give up early when that is too much
    if (u_len + (int64_t)(alive.size() / 4) * front_update_len(dmin) > max_u) return false;
    const int thr = dmin <= 2 ? 2 : std::max(3 * dmin, dmin + 4);
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
    P.max_d = std::max(P.max_d, level_max);
    P.lvl_max_d.push_back(level_max);
    P.lvl.push_back((int)order.size());
    size_t keep = 0;
    for (int v : alive)
      if (elim[v] < 0) alive[keep++] = v;
    alive.resize(keep);
  }
  P.u_len = u_len;
  // elimination positions; fronts
  std::vector<int32_t>& pos = mark;
  for (int p = 0; p < N; ++p) pos[order[p]] = p;
  P.meta.resize(N);
  int64_t nb_total = 0, uo = 0;
  for (int v = 0; v < N; ++v) nb_total += A.len[v];
  if (nb_total > INT32_MAX / 36) return false;
  P.nb_pose.resize(nb_total);
  std::vector<int32_t> nb(nb_total);  // neighbours as positions, ascending
  int32_t no = 0;
  for (int p = 0; p < N; ++p) {
    const int v = order[p], d = A.len[v];
    FrontMeta& m = P.meta[p];
    m = FrontMeta{};
    m.pose = v;
    m.d = d;
    m.nb_off = no;
    m.u_off = uo;
    for (int k = 0; k < d; ++k) nb[no + k] = pos[A.at(v)[k]];
    std::sort(nb.begin() + no, nb.begin() + no + d);
    for (int k = 0; k < d; ++k) P.nb_pose[no + k] = order[nb[no + k]];
    no += d;
    uo += front_update_len(d);
  }
  // children (a front's parent is its first neighbour) and position maps
  for (int p = 0; p < N; ++p)
    if (P.meta[p].d > 0) ++P.meta[nb[P.meta[p].nb_off]].n_child;
  int32_t co = 0;
  int64_t mo = 0;
  for (int p = 0; p < N; ++p) {
    P.meta[p].child_off = co;
    co += P.meta[p].n_child;
    mo += (int64_t)P.meta[p].n_child * (P.meta[p].d + 1);
    P.meta[p].n_child = 0;
  }
  if (mo > lim.max_maps) return false;
  P.childs.resize(co);
  P.maps.resize(mo);
  int32_t map_off = 0;
  std::vector<int32_t> map_base(N);
  {
    int64_t m = 0;
    std::vector<int32_t> cnt(N, 0);
    for (int p = 0; p < N; ++p)
      if (P.meta[p].d > 0) ++cnt[nb[P.meta[p].nb_off]];
    for (int p = 0; p < N; ++p) {
      map_base[p] = (int32_t)m;
      m += (int64_t)cnt[p] * (P.meta[p].d + 1);
    }
  }
  (void)map_off;
  for (int c = 0; c < N; ++c) {  // ascending: a front's children in elimination order
    const FrontMeta& cm = P.meta[c];
    if (cm.d == 0) continue;
    const int p = nb[cm.nb_off];
    FrontMeta& m = P.meta[p];
    FrontChild& ch = P.childs[m.child_off + m.n_child];
    ch.u_off = cm.u_off;
    ch.d = cm.d;
    ch.map_off = map_base[p] + m.n_child * (m.d + 1);
    ++m.n_child;
    int32_t* map = P.maps.data() + ch.map_off;
    map[0] = 0;
    int j = 1;  // child neighbours past the parent itself, a subset of the parent's
    for (int k = 1; k <= m.d; ++k) {
      const bool hit = j < cm.d && nb[cm.nb_off + j] == nb[m.nb_off + k - 1];
      map[k] = hit ? j++ : -1;
    }
    if (j != cm.d) return false;  // not reached: fill makes the child's rest a subset
  }
  // between factors, assembled at the endpoint eliminated first
  for (int f = 0; f < F; ++f)
    if (kind[f] == 0) ++P.meta[std::min(pos[fi[f]], pos[fj[f]])].n_orig;
  int32_t oo = 0;
  for (int p = 0; p < N; ++p) {
    P.meta[p].orig_off = oo;
    oo += P.meta[p].n_orig;
    P.meta[p].n_orig = 0;
  }
  P.origs.resize(oo);
  for (int f = 0; f < F; ++f) {
    if (kind[f] != 0) continue;
    const int a = pos[fi[f]], b = pos[fj[f]];
    FrontMeta& m = P.meta[std::min(a, b)];
    const int32_t* s = nb.data() + m.nb_off;
    const int slot = (int)(std::lower_bound(s, s + m.d, std::max(a, b)) - s) + 1;
    // the block has neighbour rows and pivot columns: Hij (rows i, columns j)
    // is its transpose when the pivot is key i
    P.origs[m.orig_off + m.n_orig++] = FrontOrig{f, 2 * slot + (a < b ? 1 : 0)};
  }
  return true;
}

}  // namespace rpgo
