// Direct solve of the damped Gauss-Newton system (H + lambda damp) dx = b: a
// multifrontal block Cholesky in FP64 on the elimination plan of
// direct_plan.h, one launch per level, the pivots of a level independent.
//
// A front is a run of s pivots and the rows they share.  Its workgroup gathers
// the pivots' columns (diagonal blocks, damping, the between factors assembled
// here, the children's update matrices) into LDS, factors the panel column by
// column, and writes the update matrix
//   U_kl = sum over children U_kl - sum over pivots G_kq G_lq^T      (k >= l)
// for its parent; the right-hand side is one more row of the same elimination,
// so the forward substitution costs no pass of its own.  The backward
// substitution runs the levels in reverse.  Every sum has a fixed order: no
// atomics, the same result on every run.
//
// Why not more PCG: the two-level PCG takes 300 to 900 iterations per linear
// step on dead-reckoned helices (condition number 4e10 at 50,000 poses), each
// four dependent launches.  The whole factorization is about 0.2 GFLOP and
// 270 MB there; what bounds it is the chain of dependent levels, 23 to 25 at
// 50,000 poses with 5,000 loop closures, each 22 to 38 us forward and 9 back.
// PCG -> this, wall time of the call, on one box: LM at 50,000 poses 698 -> 54
// ms, GNC at 3,000 poses 1,272 -> 225 ms, planar GNC at 500 poses 674 -> 68 ms,
// eight GNC solves of 200-2,000 poses on four lanes 1,747 -> 228 ms.
#include <cmath>
#include <new>

#include "rpgo_internal.h"
#include "rpgo_solver.h"
#include "solver_device.h"

namespace rpgo {

// A pivot this far below the pose's own Hessian diagonal is rounding: the
// matrix is singular or indefinite to FP64 and the solve is left to the PCG.
// The smallest pivots of regular systems are about 1e-10 (the end of a
// 50,000-pose chain).  It does not tell a free graph: there the noise itself
// reaches 1e-9, so an undamped step needs poses_held.
constexpr double kPivotMin = 1e-13;

__device__ __forceinline__ void load6(const double* __restrict__ s, double (&v)[6]) {
  const double2* q = reinterpret_cast<const double2*>(s);  // every block row is 16-byte aligned
#pragma unroll
  for (int e = 0; e < 3; ++e) {
    const double2 a = q[e];
    v[2 * e] = a.x;
    v[2 * e + 1] = a.y;
  }
}

__device__ __forceinline__ void add6(const double* __restrict__ s, double (&v)[6]) {
  double a[6];
  load6(s, a);
#pragma unroll
  for (int e = 0; e < 6; ++e) v[e] += a[e];
}

__device__ __forceinline__ void store6(double* s, const double (&v)[6]) {
  double2* q = reinterpret_cast<double2*>(s);
#pragma unroll
  for (int e = 0; e < 3; ++e) q[e] = make_double2(v[2 * e], v[2 * e + 1]);
}

// v <- v L^-T for one row of six; L lower, row-major, its diagonal inverted
__device__ __forceinline__ void row_solve(const double (&L)[36], double (&v)[6]) {
#pragma unroll
  for (int j = 0; j < 6; ++j) {
#pragma unroll
    for (int k = 0; k < j; ++k) v[j] -= v[k] * L[j * 6 + k];
    v[j] *= L[j * 7];
  }
}

// 6x6 Cholesky of the block at s, in every thread (broadcast reads); L lower
// with its diagonal inverted.  False when a pivot is noise of its pose's own
// diagonal hd, or NaN.
__device__ __forceinline__ bool block_factor(const double* s, const double (&hd)[6], double (&L)[36]) {
  bool ok = true;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
#pragma unroll
    for (int r = c; r < 6; ++r) {
      double v = s[r * 6 + c];
#pragma unroll
      for (int k = 0; k < c; ++k) v -= L[r * 6 + k] * L[c * 6 + k];
      if (r == c) {
        ok = ok && v > kPivotMin * hd[c] && v > 0.0;
        L[c * 7] = rsqrt(fmax(v, 1e-300));
      } else {
        L[r * 6 + c] = v * L[c * 7];
      }
    }
  }
  return ok;
}

__device__ __forceinline__ void load_lower(const double* s, double (&L)[36]) {
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = 0; c <= r; ++c) L[r * 6 + c] = s[r * 6 + c];
}

// v += the children's update rows at block (R, C), row i; R = -1: their
// vectors at C.  Two children at a time, so their loads overlap.
__device__ __forceinline__ void gather_children(const FrontMeta& m, const FrontChild* __restrict__ childs,
                                                const int* __restrict__ maps, const double* U, int R, int C, int i,
                                                double (&v)[6]) {
  for (int c = 0; c < m.n_child; c += 2) {
    double a[2][6];
#pragma unroll
    for (int u = 0; u < 2; ++u) {
#pragma unroll
      for (int e = 0; e < 6; ++e) a[u][e] = 0.0;
      if (c + u < m.n_child) {
        const FrontChild ch = childs[m.child_off + c + u];
        const int* map = maps + m.map_off + (size_t)(c + u) * m.n;
        const int pl = map[C], pk = R < 0 ? pl : map[R];
        if (pl >= 0 && pk >= 0)
          load6(U + ch.u_off + (R < 0 ? 36 * ((size_t)ch.d * (ch.d + 1) / 2) + 6 * pl
                                      : 36 * ((size_t)pk * (pk + 1) / 2 + pl) + 6 * i),
                a[u]);
      }
    }
#pragma unroll
    for (int e = 0; e < 6; ++e) v[e] = (v[e] + a[0][e]) + a[1][e];
  }
}

// the sum of a run of between factors of one block, row i
__device__ __forceinline__ void gather_factors(const FrontOrig* __restrict__ o, int i, const double* __restrict__ Hij,
                                               double (&v)[6]) {
  const int run = o->run;
  for (int k = 0; k < run; ++k) {
    const double* B = Hij + (size_t)o[k].f * 36;
    if (o[k].slot & 1) {
#pragma unroll
      for (int j = 0; j < 6; ++j) v[j] += B[j * 6 + i];
    } else {
      add6(B + 6 * i, v);
    }
  }
}

// block index of the lower triangle -> row and column
__device__ __forceinline__ void tri_index(int blk, int* k, int* l) {
  int r = (int)((sqrtf(8.0f * (float)blk + 1.0f) - 1.0f) * 0.5f);
  while ((r + 1) * (r + 2) / 2 <= blk) ++r;
  while (r * (r + 1) / 2 > blk) --r;
  *k = r;
  *l = blk - r * (r + 1) / 2;
}

// Element (ri, ci) of a front's update matrix (scalar rows and columns of the
// front from 6 s on; row 6 n: the update vector): its place from u_off, or -1
// above the block diagonal
__device__ __forceinline__ long long update_at(int n, int s, int ri, int ci) {
  const int k = ri / 6 - s, i = ri % 6, l = ci / 6 - s, j = ci % 6;
  if (ci >= 6 * n || ri > 6 * n || k < l) return -1;
  const long long blk = (long long)k * (k + 1) / 2;
  if (ri == 6 * n) return 36 * ((long long)(n - s) * (n - s + 1) / 2) + 6 * l + j;
  return 36 * (blk + l) + 6 * i + j;
}

typedef double d4 __attribute__((ext_vector_type(4)));

// Where element (row ri, scalar column ci) of the panel stands, less 6 ri
__device__ __forceinline__ int panel_col(int n, int ci) {
  const int q = (ci * 43691) >> 18;  // ci / 6, exact below 49,152
  return 6 * (__mul24(6 * q, n) - 3 * __mul24(q, q - 1) - 5 * q) + ci - 6 * q;
}

// c - P(r0 .., k0 .. k1) P(c0 .., k0 .. k1)^T of the panel in LDS, a 16x16
// tile: lane holds column lane % 16, rows 4 r + lane / 16.  Rows past the
// panel repeat its last one (their results are not stored).
__device__ __forceinline__ d4 tile_product(const double* row, int n, int r0, int c0, int k0, int k1, int lane, d4 c) {
  const int ra = 6 * min(r0 + (lane & 15), 6 * n), rb = 6 * min(c0 + (lane & 15), 6 * n);
  for (int k = k0; k < k1; k += 4) {
    const int g = k + (lane >> 4);
    const double* col = row + panel_col(n, min(g, k1 - 1));
    const double a = col[ra], b = col[rb];
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(g < k1 ? -a : 0.0, g < k1 ? b : 0.0, c, 0, 0, 0);
  }
  return c;
}

// A front's panel from the Hessian, the between factors and the children's
// updates; `mid` runs while those loads are in flight.
template <int TB, class F>
__device__ __forceinline__ void front_gather(const FrontMeta& m, const FrontChild* __restrict__ childs,
                                             const FrontOrig* __restrict__ origs, const int* __restrict__ maps,
                                             const int* __restrict__ rows, const double* __restrict__ D,
                                             const double* __restrict__ hdiag, const double* __restrict__ b,
                                             const double* __restrict__ Hij, double lambda, int diag_damping,
                                             const double* U, double* row, F&& mid) {
  const int tid = threadIdx.x, n = m.n, s = m.s, w = 6 * n + 1;
  // the pivots' own diagonals behind the panel (a load per pivot in the
  // factorization would be two memory latencies each)
  for (int q = tid; q < s; q += TB) {
    double v[6];
    load6(hdiag + (size_t)rows[m.row_off + q] * 6, v);
    store6(row + 6 * (panel_row(n, s) + q), v);
  }
  // panel rows: column q, row i of block R (R = n: the right-hand side)
  for (int t = tid; t < s * w; t += TB) {
    const int q = t / w, rr = t - q * w, R = rr / 6, i = rr - 6 * R;
    if (R < q) continue;
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (R == n) {
      load6(b + (size_t)rows[m.row_off + q] * 6, v);
      gather_children(m, childs, maps, U, -1, q, 0, v);
    } else {
      if (R == q) {
        const size_t pose = (size_t)rows[m.row_off + q];
        load6(D + pose * 36 + 6 * i, v);
        const double dd = diag_damping ? fmin(fmax(hdiag[pose * 6 + i], 1e-6), 1e32) : 1.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) v[j] += j == i ? lambda * dd : 0.0;
      }
      gather_children(m, childs, maps, U, R, q, i, v);
    }
    store6(row + 6 * (panel_row(n, q) + rr - 6 * q), v);
  }
  // the between factors' blocks, each by the first of its run; by other
  // wavefronts than the panel's first rows and `mid`, so that the three chains
  // of dependent loads run side by side
  const FrontOrig* og = origs + m.orig_off;
  const int to = (tid + TB / 2) % TB;
  double ov[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  if (to < 6 * m.n_orig) gather_factors(og + to / 6, to % 6, Hij, ov);
  mid();
  __syncthreads();
  if (m.n_orig == 0) return;
  for (int t = to; t < 6 * m.n_orig; t += TB) {
    const FrontOrig* o = og + t / 6;
    if (o->run == 0) continue;
    const int q = o->slot >> 16, R = (o->slot >> 1) & 0x7fff;
    if (t != to) {
#pragma unroll
      for (int e = 0; e < 6; ++e) ov[e] = 0.0;
      gather_factors(o, t % 6, Hij, ov);
    }
    double* r = row + 6 * (panel_row(n, q) + 6 * (R - q) + t % 6);
    add6(r, ov);
    store6(r, ov);
  }
  __syncthreads();
}

// The 6x6 pivot of column q and the rows below it; afterwards the factor's
// block stands in place of the pivot.  Only wavefronts with rows to solve
// factor the pivot: all sixteen of a workgroup doing so cost 1.5 us a pivot in
// LDS reads and FP64 issue.
template <int TB>
__device__ __forceinline__ void front_pivot(const FrontMeta& m, int q, double* row, int* bad) {
  const int tid = threadIdx.x, nr = 6 * (m.n - q), w0 = __builtin_amdgcn_readfirstlane(tid & ~63);
  double* col = row + 6 * panel_row(m.n, q);
  double L[36];
  bool ok = true;
  if (w0 == 0 || 6 + w0 <= nr) {
    double hd[6];
    load6(row + 6 * (panel_row(m.n, m.s) + q), hd);
    ok = block_factor(col, hd, L);
    for (int t = 6 + tid; t <= nr; t += TB) {
      double v[6];
      load6(col + 6 * t, v);
      row_solve(L, v);
      store6(col + 6 * t, v);
    }
  }
  __syncthreads();
  if (tid == 0) {
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int c = 0; c <= r; ++c) col[r * 6 + c] = L[r * 6 + c];
    if (!ok && blockIdx.y == 0) *bad = 1;
  }
}

#define RPGO_FRONT_PARAMS                                                                                      \
  int first, const FrontMeta *__restrict__ meta, const FrontChild *__restrict__ childs,                        \
      const FrontOrig *__restrict__ origs, const int *__restrict__ maps, const int *__restrict__ rows,         \
      const double *__restrict__ D, const double *__restrict__ hdiag, const double *__restrict__ b,            \
      const double *__restrict__ Hij, double lambda, int diag_damping, double *U, double *__restrict__ G,      \
      int *__restrict__ bad

// Small fronts (the thousands of the first levels), every update row of six
// by one lane
template <int TB>
__global__ void __launch_bounds__(TB) k_front_small(RPGO_FRONT_PARAMS) {
  extern __shared__ __align__(16) double row[];
  const int tid = threadIdx.x, t0 = TB - 1 - tid;
  const FrontMeta m = meta[first + blockIdx.x];
  const int n = m.n, s = m.s, d = n - s, nblk = d * (d + 1) / 2, ntask = 6 * nblk + d;
  // the first update row's children are loaded before the panel is factored
  const auto children = [&](int t, double (&v)[6]) {
    if (t < 6 * nblk) {
      int k, l;
      tri_index(t / 6, &k, &l);
      gather_children(m, childs, maps, U, s + k, s + l, t % 6, v);
    } else {
      gather_children(m, childs, maps, U, -1, s + t - 6 * nblk, 0, v);
    }
  };
  double pre[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
  front_gather<TB>(m, childs, origs, maps, rows, D, hdiag, b, Hij, lambda, diag_damping, U, row, [&] {
    if (t0 < ntask) children(t0, pre);
  });
  for (int q = 0; q < s; ++q) {
    const double* col = row + 6 * panel_row(n, q);
    front_pivot<TB>(m, q, row, bad);
    // the panel's other columns
    const int wq = 6 * (n - q) - 5, nc = s - 1 - q;
    for (int t = tid; t < nc * wq; t += TB) {
      const int C = t / wq, rr = t - C * wq;  // both from q + 1
      if (rr < 6 * C) continue;
      double* r = row + 6 * (panel_row(n, q + 1 + C) + rr - 6 * C);
      const double* hc = col + 36 * (C + 1);
      double v[6], g[6];
      load6(r, v);
      load6(col + 6 * (6 + rr), g);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        double h[6];
        load6(hc + 6 * j, h);
#pragma unroll
        for (int k = 0; k < 6; ++k) v[j] -= g[k] * h[k];
      }
      store6(r, v);
    }
    __syncthreads();
  }
  {
    const double2* src = reinterpret_cast<const double2*>(row);
    double2* dst = reinterpret_cast<double2*>(G + m.g_off);
    for (int t = tid; t < 3 * panel_row(n, s); t += TB) dst[t] = src[t];
  }
  for (int t = t0; t < ntask; t += TB) {
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (t == t0) {
#pragma unroll
      for (int e = 0; e < 6; ++e) v[e] = pre[e];
    } else {
      children(t, v);
    }
    int k = d, l = t - 6 * nblk, i = 0;  // the right-hand side's row is row 0 of block n
    if (t < 6 * nblk) {
      tri_index(t / 6, &k, &l);
      i = t % 6;
    }
    for (int q = 0; q < s; ++q) {
      const double* col = row + 6 * panel_row(n, q);
      double g[6];
      load6(col + 36 * (s + k - q) + 6 * i, g);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        double h[6];
        load6(col + 36 * (s + l - q) + 6 * j, h);
#pragma unroll
        for (int e = 0; e < 6; ++e) v[j] -= g[e] * h[e];
      }
    }
    store6(U + m.u_off + 6 * (size_t)t, v);
  }
}

// Wider fronts, a workgroup each (gridDim.y of them share a front's update
// tiles, each repeating the panel).  What bounds it is latency: meta, maps and
// update matrix are dependent loads, then each pivot is a 6x6 Cholesky and two
// barriers (1.6 us; the 3,000-pose graph's levels of five to ten pivots take
// 23 to 37 us, where a launch per pivot took 6.7 us and a gap each).  Updates
// go 16x16 tiles at a time through the matrix cores; by rows of six in vector
// FMA they were bound by the LDS (21 16-byte reads for 36 FMAs) and a level of
// 50,000 poses took 45 us against 34.
template <int TB>
__global__ void __launch_bounds__(TB) k_front(RPGO_FRONT_PARAMS) {
  extern __shared__ __align__(16) double row[];
  constexpr int NW = TB / 64;
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const FrontMeta m = meta[first + blockIdx.x];
  const int n = m.n, s = m.s, T = (6 * (n - s) + 16) / 16, ntile = T * (T + 1) / 2;
  // children's sum of update tile (ti, tj)
  const auto children = [&](int t) {
    d4 c = {0.0, 0.0, 0.0, 0.0};
    int ti, tj;
    tri_index(t, &ti, &tj);
    const int ci = 6 * s + 16 * tj + (lane & 15), r0 = 6 * s + 16 * ti + (lane >> 4);
    if (ci >= 6 * n) return c;
    const int l = ci / 6, j = ci - 6 * l;
    for (int k = 0; k < m.n_child; k += 2) {  // two children's loads overlap
      double v[2][4];
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        const bool has = k + u < m.n_child;
        const FrontChild ch = childs[m.child_off + (has ? k + u : k)];
        const int* map = maps + m.map_off + (size_t)(has ? k + u : k) * n;
        const int pl = map[l];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int ri = r0 + 4 * r, R = ri / 6;
          const int pk = ri >= 6 * n ? ch.d : map[R];
          const size_t o = 36 * ((size_t)pk * (pk + 1) / 2 + (ri == 6 * n ? 0 : pl)) +
                           (ri == 6 * n ? 6 * pl : 6 * (ri - 6 * R)) + j;
          v[u][r] = has && pl >= 0 && pk >= pl && R >= l && ri <= 6 * n ? U[ch.u_off + o] : 0.0;
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r) c[r] = (c[r] + v[0][r]) + v[1][r];
    }
    return c;
  };
  const int t0 = blockIdx.y * NW + NW - 1 - wv;
  d4 pre = {0.0, 0.0, 0.0, 0.0};
  // the first tile's children are loaded before the panel is factored
  front_gather<TB>(m, childs, origs, maps, rows, D, hdiag, b, Hij, lambda, diag_damping, U, row, [&] {
    if (n > s && t0 < ntile) pre = children(t0);
  });
  for (int q = 0; q < s; ++q) {
    front_pivot<TB>(m, q, row, bad);
    // the panel's other columns: a strip of 16 rows to two wavefronts, each
    // every other tile, its own fragments held over them
    const int c0 = 6 * (q + 1), nct = (6 * s - c0 + 15) / 16, nrt = (6 * n + 16 - c0) / 16;
    const int g0 = 6 * q + (lane >> 4), g1 = min(g0 + 4, 6 * q + 5);
    const double *f0 = row + panel_col(n, g0), *f1 = row + panel_col(n, g1);
    for (int ti = nct > 0 ? wv >> 1 : nrt; ti < nrt; ti += NW / 2) {
      const int ra = 6 * min(c0 + 16 * ti + (lane & 15), 6 * n), r0 = c0 + 16 * ti + (lane >> 4);
      const double a0 = -f0[ra], a1 = lane < 32 ? -f1[ra] : 0.0;
      for (int tj = wv & 1; tj < nct && tj <= ti; tj += 2) {
        const int ci = min(c0 + 16 * tj + (lane & 15), 6 * s - 1), rb = 6 * (c0 + 16 * tj + (lane & 15));
        const int rc = min(rb, 36 * n);
        double* p = row + panel_col(n, ci);
        const double b0 = f0[rc], b1 = f1[rc];
        d4 c;
#pragma unroll
        for (int r = 0; r < 4; ++r) c[r] = p[6 * min(r0 + 4 * r, 6 * n)];
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(a0, b0, c, 0, 0, 0);
        c = __builtin_amdgcn_mfma_f64_16x16x4f64(a1, lane < 32 ? b1 : 0.0, c, 0, 0, 0);
        const bool in = rb < 36 * s;
        const int top = ci - ci % 6;
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (in && r0 + 4 * r <= 6 * n && r0 + 4 * r >= top) p[6 * (r0 + 4 * r)] = c[r];
      }
    }
    __syncthreads();
  }
  // the factored panel, then the update tiles
  {
    const double2* src = reinterpret_cast<const double2*>(row);
    double2* dst = reinterpret_cast<double2*>(G + m.g_off);
    const int np = 3 * panel_row(n, s);
    for (int t = blockIdx.y * TB + tid; t < np; t += TB * gridDim.y) dst[t] = src[t];
  }
  if (n == s) return;
  for (int t = t0; t < ntile; t += NW * gridDim.y) {
    int ti, tj;
    tri_index(t, &ti, &tj);
    const int c0 = 6 * s + 16 * tj, r0 = 6 * s + 16 * ti;
    if (c0 >= 6 * n) continue;
    const d4 c = tile_product(row, n, r0, c0, 0, 6 * s, lane, t == t0 ? pre : children(t));
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const long long o = update_at(n, s, r0 + 4 * r + (lane >> 4), c0 + (lane & 15));
      if (o >= 0) U[m.u_off + o] = c[r];
    }
  }
}

// Forward substitution of another right-hand side with the stored factor
// (iterative refinement): the panel copied to LDS, a front's vector behind it,
// the update vectors in the fronts' own vector slots.
template <int TB>
__global__ void __launch_bounds__(TB) k_front_forward(int first, const FrontMeta* __restrict__ meta,
                                                      const FrontChild* __restrict__ childs,
                                                      const int* __restrict__ maps, const int* __restrict__ rows,
                                                      const double* __restrict__ b, double* G, double* U) {
  extern __shared__ __align__(16) double row[];
  const int tid = threadIdx.x;
  const FrontMeta m = meta[first + blockIdx.x];
  const int n = m.n, s = m.s, np = panel_row(n, s), d = n - s, w0 = __builtin_amdgcn_readfirstlane(tid & ~63);
  double* vec = row + 6 * np;
  {
    const double2* src = reinterpret_cast<const double2*>(G + m.g_off);
    double2* dst = reinterpret_cast<double2*>(row);
    for (int t = tid; t < 3 * np; t += TB) dst[t] = src[t];
  }
  for (int R = tid; R < n; R += TB) {
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (R < s) load6(b + (size_t)rows[m.row_off + R] * 6, v);
    gather_children(m, childs, maps, U, -1, R, 0, v);
    store6(vec + 6 * R, v);
  }
  __syncthreads();
  for (int q = 0; q < s; ++q) {
    const double* col = row + 6 * panel_row(n, q);
    if (w0 > 0 && 6 + w0 >= 6 * (n - q)) {  // no rows for this wavefront
      __syncthreads();
      continue;
    }
    double L[36], y[6];
    load_lower(col, L);
    load6(vec + 6 * q, y);
    row_solve(L, y);
    if (tid == 0) store6(G + m.g_off + 6 * (panel_row(n, q) + 6 * (n - q)), y);
    for (int t = 6 + tid; t < 6 * (n - q); t += TB) {
      double h[6], v = vec[6 * q + t];
      load6(col + 6 * t, h);
#pragma unroll
      for (int k = 0; k < 6; ++k) v -= h[k] * y[k];
      vec[6 * q + t] = v;
    }
    __syncthreads();
  }
  double* u = U + m.u_off + 36 * ((size_t)d * (d + 1) / 2);
  for (int t = tid; t < 6 * d; t += TB) u[t] = vec[6 * s + t];
}

// Backward substitution of one level, a workgroup a front: the neighbours'
// part of every pivot at once (thread e = (pivot, component), the rows split
// among TB / (6 s) parts, partials added in a fixed order), then the pivots
// from the last to the first on the triangle in LDS.
template <int TB>
__global__ void __launch_bounds__(TB) k_back(int first, const FrontMeta* __restrict__ meta,
                                             const int* __restrict__ rows, const double* __restrict__ G, double* x) {
  extern __shared__ __align__(16) double tri[];
  __shared__ double red[TB];
  const int tid = threadIdx.x;
  const FrontMeta m = meta[first + blockIdx.x];
  const int n = m.n, s = m.s, ns = 6 * s, w0 = __builtin_amdgcn_readfirstlane(tid & ~63);
  const double* P = G + m.g_off;
  double* xs = tri + 18 * s * (s + 1);  // the neighbours' x, later the pivots'
  for (int R = s + tid; R < n; R += TB) {
    double v[6];
    load6(x + 6 * (size_t)rows[m.row_off + R], v);
    store6(xs + 6 * (R - s), v);
  }
  for (int q = 0; q < s; ++q) {  // rows of the pivots, blocks (q, q .. s-1)
    const double2* src = reinterpret_cast<const double2*>(P + 6 * panel_row(n, q));
    double2* dst = reinterpret_cast<double2*>(tri + 36 * (q * s - q * (q - 1) / 2));
    for (int t = tid; t < 18 * (s - q); t += TB) dst[t] = src[t];
  }
  const int parts = TB / ns, part = tid / ns, e = tid - part * ns, eq = e / 6, j = e - 6 * eq;
  double y = tid < ns ? P[6 * (panel_row(n, eq) + 6 * (n - eq)) + j] : 0.0;
  __syncthreads();
  double acc = 0.0;
  if (part < parts) {
    const double* B = P + 6 * panel_row(n, eq) + 36 * (s - eq) + j;
    for (int r = part; r < n - s; r += parts)
#pragma unroll
      for (int i = 0; i < 6; ++i) acc += B[36 * r + 6 * i] * xs[6 * r + i];
  }
  red[tid] = acc;
  __syncthreads();
  if (tid < ns) {
    double t = 0.0;
    for (int k = 0; k < parts; ++k) t += red[k * ns + tid];
    y -= t;
    xs[tid] = y;
  }
  __syncthreads();
  for (int q = s - 1; q >= 0; --q) {
    if (w0 > 0 && w0 >= 6 * q) {  // no components for this wavefront
      __syncthreads();
      continue;
    }
    double L[36], r[6];
    load_lower(tri + 36 * (q * s - q * (q - 1) / 2), L);
    load6(xs + 6 * q, r);
#pragma unroll
    for (int i = 5; i >= 0; --i) {
#pragma unroll
      for (int k = i + 1; k < 6; ++k) r[i] -= L[k * 6 + i] * r[k];
      r[i] *= L[i * 7];
    }
    if (tid == 0) store6(x + 6 * (size_t)rows[m.row_off + q], r);
    if (tid < 6 * q) {
      const double* B = tri + 36 * (eq * s - eq * (eq - 1) / 2 + q - eq) + j;
#pragma unroll
      for (int i = 0; i < 6; ++i) y -= B[6 * i] * r[i];
      xs[tid] = y;
    }
    __syncthreads();
  }
}

// Row i of H x at pose p on the chain layout, in the order of
// k_pcg_spmv_chain: diagonal, link to p+1, link from p-1, extras
__device__ __forceinline__ double chain_row(int N, int p, int i, const double* __restrict__ Ds,
                                            const double* __restrict__ Cs, const int* __restrict__ eoff,
                                            const int* __restrict__ ext, const int* __restrict__ extq,
                                            const double* __restrict__ Hij, const double* __restrict__ x) {
  double v[6];
  load6(x + (size_t)p * 6, v);
  double acc = 0.0;
#pragma unroll
  for (int c = 0; c < 6; ++c) acc += Ds[(size_t)(i * 6 + c) * N + p] * v[c];
  load6(x + (size_t)(p + 1 < N ? p + 1 : p) * 6, v);  // Cs is zero at p = N - 1
  double s = 0.0;
#pragma unroll
  for (int c = 0; c < 6; ++c) s += Cs[(size_t)(i * 6 + c) * N + p] * v[c];
  acc += s;
  if (p > 0) {
    load6(x + (size_t)(p - 1) * 6, v);
    s = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) s += Cs[(size_t)(c * 6 + i) * N + p - 1] * v[c];
    acc += s;
  }
  for (int k = eoff[p]; k < eoff[p + 1]; ++k) {
    const int t = ext[k];
    const double* B = Hij + (size_t)(t >> 1) * 36;
    load6(x + (size_t)extq[k] * 6, v);
    s = 0.0;
#pragma unroll
    for (int c = 0; c < 6; ++c) s += ((t & 1) ? B[c * 6 + i] : B[i * 6 + c]) * v[c];
    acc += s;
  }
  return acc;
}

// hx = H dx on the chain layout (the rows of k_pcg_spmv_chain without the
// damping), the residual r = b - hx - lambda damp dx, and this workgroup's
// parts of b.dx, dx.hx, |r|^2 and |b|^2.
__global__ void __launch_bounds__(384) k_direct_check(int N, const double* __restrict__ Ds,
                                                      const double* __restrict__ Cs, const int* __restrict__ eoff,
                                                      const int* __restrict__ ext, const int* __restrict__ extq,
                                                      const double* __restrict__ Hij,
                                                      const double* __restrict__ hdiag, double lambda,
                                                      int diag_damping, const double* __restrict__ b,
                                                      const double* __restrict__ x, double* __restrict__ r,
                                                      double* __restrict__ part) {
  __shared__ double red[16];
  const int i = threadIdx.x >> 6, p = blockIdx.x * 64 + (threadIdx.x & 63);
  double s0 = 0.0, s1 = 0.0, s2 = 0.0, s3 = 0.0;
  if (p < N) {
    const double hx = chain_row(N, p, i, Ds, Cs, eoff, ext, extq, Hij, x);
    const double dd = diag_damping ? fmin(fmax(hdiag[(size_t)p * 6 + i], 1e-6), 1e32) : 1.0;
    const double xi = x[(size_t)p * 6 + i], bi = b[(size_t)p * 6 + i];
    const double ri = bi - (hx + lambda * dd * xi);
    r[(size_t)p * 6 + i] = ri;
    s0 = bi * xi;
    s1 = xi * hx;
    s2 = ri * ri;
    s3 = bi * bi;
  }
  s0 = block_sum(s0, red);
  s1 = block_sum(s1, red);
  s2 = block_sum(s2, red);
  s3 = block_sum(s3, red);
  if (threadIdx.x == 0) {
    double* o = part + 4 * (size_t)blockIdx.x;
    o[0] = s0;
    o[1] = s1;
    o[2] = s2;
    o[3] = s3;
  }
}

// out[0..3] = sums of part's n rows of four, out[4] = sum of cpart's nc
// entries, out[5] = *bad; one workgroup, fixed order; out is pinned host memory
__global__ void __launch_bounds__(256) k_direct_reduce(int n, const double* __restrict__ part, int nc,
                                                       const double* __restrict__ cpart, const int* __restrict__ bad,
                                                       double* __restrict__ out) {
  __shared__ double red[16];
  double s[5] = {0.0, 0.0, 0.0, 0.0, 0.0};
  for (int k = threadIdx.x; k < n; k += 256) {
    const double2 a = reinterpret_cast<const double2*>(part)[2 * k], c = reinterpret_cast<const double2*>(part)[2 * k + 1];
    s[0] += a.x;
    s[1] += a.y;
    s[2] += c.x;
    s[3] += c.y;
  }
  for (int k = threadIdx.x; k < nc; k += 256) s[4] += cpart[k];
#pragma unroll
  for (int q = 0; q < 5; ++q) {
    const double v = block_sum(s[q], red);
    if (threadIdx.x == 0) out[q] = v;
  }
  if (threadIdx.x == 0) out[5] = bad ? (double)*bad : 0.0;
}

// y += a, the former y kept in old
__global__ void k_direct_axpy(long long n, const double* __restrict__ a, double* __restrict__ y,
                              double* __restrict__ old) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t >= n) return;
  const double v = y[t];
  old[t] = v;
  y[t] = v + a[t];
}

// ------------------------------------------------------------------ host
static_assert(panel_bytes(DirectLimits().max_d + 1, 1) <= kPanelBytes, "one pivot's panel in LDS");
static_assert(6 * (DirectLimits().max_d + 1) + 16 < 49152, "panel_col's division by six");

// Whether the weights of this nonlinear solve hold every pose (*held: -1 until
// it is known).  Factors whose weights do not change in a run are looked at once.
int SolverRun::poses_held_now(hipStream_t st, const rpgo_solve_problem* pr, int* held) {
  if (*held >= 0) return RPGO_OK;
  if (held_always == 1) {
    *held = 1;
    return RPGO_OK;
  }
  std::vector<double> wt(F);
  RPGO_HIP_CHECK(hipMemcpyAsync(wt.data(), w.ptr, sizeof(double) * F, hipMemcpyDeviceToHost, st));
  RPGO_HIP_CHECK(hipStreamSynchronize(st));
  const auto holds = [&](int f) {
    if (!(wt[f] > kHoldWeight)) return false;
    for (int e = 0; e < 36; e += 7)  // a factor of some directions only holds none
      if (!(pr->information[36 * (size_t)f + e] > 0.0)) return false;
    return true;
  };
  if (held_always < 0)
    held_always = poses_held(N, F, pr->kind, pr->key_i, pr->key_j,
                             [&](int f) { return (!prm.use_gnc || f < n_known) && holds(f); });
  *held = held_always == 1 || poses_held(N, F, pr->kind, pr->key_i, pr->key_j, holds);
  return RPGO_OK;
}

int SolverRun::direct_setup(hipStream_t st, const rpgo_solve_problem* pr) {
  direct_ready = false;
  // an explicit preconditioner choice asks for the PCG
  if (prm.pcg_segment > 0 || prm.pcg_coarse != 0 || F <= 0) return RPGO_OK;
  DirectPlan& P = plan;
  try {
    if (!build_direct_plan(N, F, pr->kind, pr->key_i, pr->key_j, DirectLimits(), P)) return RPGO_OK;
  } catch (const std::bad_alloc&) {
    return RPGO_OK;
  }
  const size_t bytes[5] = {P.meta.size() * sizeof(FrontMeta), P.childs.size() * sizeof(FrontChild),
                           P.origs.size() * sizeof(FrontOrig), P.row_pose.size() * sizeof(int32_t),
                           P.maps.size() * sizeof(int32_t)};
  const void* src[5] = {P.meta.data(), P.childs.data(), P.origs.data(), P.row_pose.data(), P.maps.data()};
  DevBuf* dst[5] = {&d_meta, &d_childs, &d_origs, &d_rows, &d_maps};
  const size_t nblk = (size_t)(N + 63) / 64, ncost = (size_t)(F + 255) / 256;
  int failed = 0;
  for (int k = 0; k < 5 && !failed; ++k) failed = dst[k]->reserve(bytes[k]);
  if (failed || d_U.reserve(sizeof(double) * (size_t)P.u_len) || d_G.reserve(sizeof(double) * (size_t)P.g_len) ||
      d_part.reserve(sizeof(double) * (4 * nblk + ncost)) || d_bad.reserve(sizeof(int)) || !pinned_scalars()) {
    // no room: keep the iterative solve, with the memory these buffers hold
    // and without the failed allocation's error, which the next launch's check
    // would report
    (void)hipGetLastError();
    direct_release();
    return RPGO_OK;
  }
  for (int k = 0; k < 5; ++k)
    if (bytes[k]) RPGO_HIP_CHECK(hipMemcpyAsync(dst[k]->ptr, src[k], bytes[k], hipMemcpyHostToDevice, st));
  RPGO_HIP_CHECK(hipMemsetAsync(d_bad.ptr, 0, sizeof(int), st));
  held_always = -1;
  direct_ready = true;
  return RPGO_OK;
}

// Factor H + lambda damp and substitute forward with b: one launch per level.
int SolverRun::direct_factor(hipStream_t st, double lambda) {
  const DirectPlan& P = plan;
  for (int l = 0; l < P.levels(); ++l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first;
    const size_t lds = (size_t)P.lvl_bytes[l];
#define RPGO_FRONT_ARGS                                                                                          \
  first, d_meta.as<FrontMeta>(), d_childs.as<FrontChild>(), d_origs.as<FrontOrig>(), d_maps.as<int>(),           \
      d_rows.as<int>(), D.as<double>(), hdiag.as<double>(), b64.as<double>(), Hij.as<double>(), lambda,          \
      prm.lm_diagonal_damping, d_U.as<double>(), d_G.as<double>(), d_bad.as<int>()
    const LevelLaunch how = level_launch(P, l);
    const dim3 grid(n, how.split);
    if (how.small && how.threads == 64) k_front_small<64><<<grid, 64, lds, st>>>(RPGO_FRONT_ARGS);
    else if (how.small) k_front_small<256><<<grid, 256, lds, st>>>(RPGO_FRONT_ARGS);
    else if (how.threads == 256) k_front<256><<<grid, 256, lds, st>>>(RPGO_FRONT_ARGS);
    else k_front<1024><<<grid, 1024, lds, st>>>(RPGO_FRONT_ARGS);
#undef RPGO_FRONT_ARGS
  }
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

int SolverRun::direct_backward(hipStream_t st, double* out) {
  const DirectPlan& P = plan;
  for (int l = P.levels() - 1; l >= 0; --l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first;
    const size_t lds = (size_t)P.lvl_back[l];
    if (level_launch(P, l).small)
      k_back<64><<<n, 64, lds, st>>>(first, d_meta.as<FrontMeta>(), d_rows.as<int>(), d_G.as<double>(), out);
    else
      k_back<256><<<n, 256, lds, st>>>(first, d_meta.as<FrontMeta>(), d_rows.as<int>(), d_G.as<double>(), out);
  }
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

// residual of dx and the sums of k_direct_check into d_part
int SolverRun::direct_check(hipStream_t st, double lambda) {
  k_direct_check<<<(unsigned)((N + 63) / 64), 384, 0, st>>>(
      N, Ds.as<double>(), Cs.as<double>(), ext_off.as<int>(), ext.as<int>(), ext_q.as<int>(), Hij.as<double>(),
      hdiag.as<double>(), lambda, prm.lm_diagonal_damping, b64.as<double>(), dx.as<double>(), r.as<double>(),
      d_part.as<double>());
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

// One refinement step: dx += (H + lambda damp)^-1 r with the stored factor; the
// step before it stays in q
int SolverRun::direct_refine(hipStream_t st) {
  const DirectPlan& P = plan;
  for (int l = 0; l < P.levels(); ++l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first;
    const size_t lds = (size_t)P.lvl_bytes[l];
#define RPGO_FORWARD_ARGS                                                                                     \
  first, d_meta.as<FrontMeta>(), d_childs.as<FrontChild>(), d_maps.as<int>(), d_rows.as<int>(), r.as<double>(), \
      d_G.as<double>(), d_U.as<double>()
    if (level_launch(P, l).small) k_front_forward<64><<<n, 64, lds, st>>>(RPGO_FORWARD_ARGS);
    else k_front_forward<256><<<n, 256, lds, st>>>(RPGO_FORWARD_ARGS);
#undef RPGO_FORWARD_ARGS
  }
  int rc;
  if ((rc = direct_backward(st, zv.as<double>()))) return rc;
  const long long n6 = 6ll * N;
  k_direct_axpy<<<(unsigned)((n6 + 255) / 256), 256, 0, st>>>(n6, zv.as<double>(), dx.as<double>(), q.as<double>());
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

// One linear step by the factorization, the step's candidate poses xn and
// their weighted cost: *lin the model decrease b.dx - dx.H dx / 2 (undamped
// H), *cost_new the cost.  *ok = false when a pivot was not positive or the
// residual stayed above what the caller asked for: the caller then takes the
// iterative solve.
int SolverRun::direct_step(hipStream_t st, double lambda, double* lin, double* cost_new, bool* ok) {
  int rc;
  double* h = pinned_scalars();
  const int nblk = (N + 63) / 64, ncost = (F + 255) / 256;
  double* cpart = d_part.as<double>() + 4 * (size_t)nblk;
  const double tol = std::min(prm.pcg_rel_tol, kDirectTol);
  *ok = false;
  double best = INFINITY;
  if ((rc = direct_factor(st, lambda))) return rc;
  if ((rc = direct_backward(st, dx.as<double>()))) return rc;
  stats.pcg_iterations += 1;
  for (int refine = 0;; ++refine) {
    if ((rc = direct_check(st, lambda))) return rc;
    retract(st);
    cost_partials(st, xn.as<double>(), cpart);
    k_direct_reduce<<<1, 256, 0, st>>>(nblk, d_part.as<double>(), ncost, cpart, d_bad.as<int>(), h + 32);
    RPGO_HIP_CHECK(hipGetLastError());
    RPGO_HIP_CHECK(hipStreamSynchronize(st));
    const double bdx = h[32], xhx = h[33], rr = h[34], bb = h[35], bad = h[37];
    if (bad != 0.0) {
      RPGO_HIP_CHECK(hipMemsetAsync(d_bad.ptr, 0, sizeof(int), st));
      return RPGO_OK;
    }
    const double residual = std::sqrt(bb > 0.0 ? rr / bb : rr);  // b = 0: dx and r are 0, or NaN
    const double before = best;
    if (refine == 0 && !(residual < 1e-2)) return RPGO_OK;
    if (residual < best) {
      best = residual;
      *lin = bdx - 0.5 * xhx;
      *cost_new = h[36];
    } else if (refine > 0) {  // the refinement lost: the step before it
      RPGO_HIP_CHECK(hipMemcpyAsync(dx.ptr, q.ptr, sizeof(double) * 6 * N, hipMemcpyDeviceToDevice, st));
      retract(st);
    }
    // done at the tolerance, after the last refinement, or when a refinement
    // no longer gains (the residual's own rounding)
    if (best <= tol || refine == kDirectRefine || !(residual <= 0.25 * before)) {
      *ok = best <= std::max(prm.pcg_rel_tol, kDirectAccept);
      return RPGO_OK;
    }
    if ((rc = direct_refine(st))) return rc;
    stats.pcg_iterations += 1;
  }
}

// One refinement of the accepted step that ends a nonlinear solve of a large
// graph, its poses in xn and their cost; kept unless the cost is not finite or
// rises by 1e-6 of itself.  (It moves the step by about 1e-4 of its length, and
// the last step by default gains less than 1e-5 of the cost.)
int SolverRun::direct_finish(hipStream_t st, double lambda, double* cost_new) {
  if (N < kDirectFinishMin) return RPGO_OK;
  int rc;
  double cost = 0.0;
  if ((rc = direct_check(st, lambda))) return rc;  // the residual of the step in dx
  if ((rc = direct_refine(st))) return rc;
  stats.pcg_iterations += 1;
  retract(st);
  if ((rc = direct_cost(st, xn.as<double>(), &cost))) return rc;
  if (cost <= *cost_new * (1.0 + 1e-6)) {
    *cost_new = cost;
    return RPGO_OK;
  }
  RPGO_HIP_CHECK(hipMemcpyAsync(dx.ptr, q.ptr, sizeof(double) * 6 * N, hipMemcpyDeviceToDevice, st));
  retract(st);
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

// weighted cost at poses xp in one read-back (the reduction's other sums unused)
int SolverRun::direct_cost(hipStream_t st, const double* xp, double* out) {
  double* h = pinned_scalars();
  double* cpart = d_part.as<double>() + 4 * (size_t)((N + 63) / 64);
  cost_partials(st, xp, cpart);
  k_direct_reduce<<<1, 256, 0, st>>>(0, d_part.as<double>(), (F + 255) / 256, cpart, nullptr, h + 32);
  RPGO_HIP_CHECK(hipGetLastError());
  RPGO_HIP_CHECK(hipStreamSynchronize(st));
  *out = h[36];
  return RPGO_OK;
}

}  // namespace rpgo
