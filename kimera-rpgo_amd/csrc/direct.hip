// Direct solve of the damped Gauss-Newton system (H + lambda damp) dx = b: a
// multifrontal block Cholesky in FP64 on the elimination plan of
// direct_plan.h, one launch per level, the pivots of a level independent.
//
// A front is one pose and its d remaining neighbours.  Its workgroup gathers
// the pivot's column (diagonal block, damping, the between factors assembled
// here, the children's update matrices) into LDS, factors the 6x6 pivot,
// forms G_k = F_k L^-T for the neighbours, and writes the update matrix
//   U_kl = sum over children U_kl - G_k G_l^T      (k >= l)
// for its parent; the right-hand side is one more row of the same elimination,
// so the forward substitution costs no pass of its own.  The backward
// substitution runs the levels in reverse.  Every sum has a fixed order: no
// atomics, the same result on every run.
//
// Why not more PCG: the two-level PCG takes 300 to 900 iterations per linear
// step on dead-reckoned helices (condition number 4e10 at 50,000 poses), each
// four dependent launches.  The whole factorization is about 0.2 GFLOP and
// 270 MB there; what bounds it is the chain of dependent levels (83 at 50,000
// poses with 5,000 loop closures), each about as long as one PCG launch.
// LM at 50,000 poses 429 -> 36 ms, GNC at 3,000 poses 1,404 -> 378 ms, planar
// GNC at 500 poses 855 -> 110 ms, eight GNC solves of 200-2,000 poses on four
// lanes 1,689 -> 285 ms (PCG -> this, wall time of the call).
#include <cmath>
#include <new>

#include "replay64.h"
#include "rpgo_internal.h"
#include "rpgo_solver.h"
#include "solver_device.h"

namespace rpgo {

// A pivot this far below the pose's own Hessian diagonal is rounding noise of
// a singular system (a graph without a prior under Gauss-Newton): the solve
// is left to the PCG, which takes semidefinite systems.  The smallest pivots
// of regular ones stay well above (about 1e-10 at the end of a 50,000-pose
// chain).
constexpr double kPivotMin = 1e-13;

// rows of a front column in LDS: 6 (d + 1) rows of the blocks, then the
// right-hand side
__host__ __device__ constexpr size_t front_lds_doubles(int d) { return 36 * (size_t)(d + 1) + 6; }

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

template <int TB>
__global__ void __launch_bounds__(TB) k_front(int first, const FrontMeta* __restrict__ meta,
                                              const FrontChild* __restrict__ childs,
                                              const FrontOrig* __restrict__ origs, const int* __restrict__ maps,
                                              const double* __restrict__ D, const double* __restrict__ hdiag,
                                              const double* __restrict__ b, const double* __restrict__ Hij,
                                              double lambda, int diag_damping, double* U, double* __restrict__ G,
                                              double* __restrict__ Lo, double* __restrict__ Y,
                                              int* __restrict__ bad) {
  extern __shared__ __align__(16) double row[];
  const int p = first + blockIdx.x, tid = threadIdx.x;
  const FrontMeta m = meta[p];
  const int d = m.d, nrow = 6 * (d + 1);
  for (int t = tid; t <= nrow; t += TB) {
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (t < nrow) {
      const int k = t / 6, i = t - 6 * k;
      if (k == 0) {
        load6(D + (size_t)m.pose * 36 + 6 * i, v);
        const double dd = diag_damping ? fmin(fmax(hdiag[(size_t)m.pose * 6 + i], 1e-6), 1e32) : 1.0;
#pragma unroll
        for (int j = 0; j < 6; ++j) v[j] += j == i ? lambda * dd : 0.0;
      } else {
        for (int o = 0; o < m.n_orig; ++o) {
          const FrontOrig a = origs[m.orig_off + o];
          if ((a.slot_t >> 1) != k) continue;
          const double* B = Hij + (size_t)a.f * 36;
          if (a.slot_t & 1) {
#pragma unroll
            for (int j = 0; j < 6; ++j) v[j] += B[j * 6 + i];
          } else {
            add6(B + 6 * i, v);
          }
        }
      }
      for (int c = 0; c < m.n_child; ++c) {
        const FrontChild ch = childs[m.child_off + c];
        const int pk = maps[ch.map_off + k];
        if (pk >= 0) add6(U + ch.u_off + 36 * (pk * (pk + 1) / 2) + 6 * i, v);
      }
    } else {
      load6(b + (size_t)m.pose * 6, v);
      for (int c = 0; c < m.n_child; ++c) {
        const FrontChild ch = childs[m.child_off + c];
        add6(U + ch.u_off + 36 * ((size_t)ch.d * (ch.d + 1) / 2), v);
      }
    }
    store6(row + 6 * t, v);
  }
  __syncthreads();
  // 6x6 Cholesky of the pivot, in every thread (broadcast reads of rows 0-5,
  // which nothing writes until the next barrier)
  double L[36], hd[6];
  load6(hdiag + (size_t)m.pose * 6, hd);
  bool ok = true;
#pragma unroll
  for (int c = 0; c < 6; ++c) {
#pragma unroll
    for (int r = c; r < 6; ++r) {
      double v = row[r * 6 + c];
#pragma unroll
      for (int k = 0; k < c; ++k) v -= L[r * 6 + k] * L[c * 6 + k];
      if (r == c) {
        ok = ok && v > kPivotMin * hd[c] && v > 0.0;  // false for NaN too
        L[c * 7] = 1.0 / sqrt(fmax(v, 1e-300));
      } else {
        L[r * 6 + c] = v * L[c * 7];
      }
    }
  }
  for (int t = 6 + tid; t <= nrow; t += TB) {
    double v[6];
    load6(row + 6 * t, v);
    row_solve(L, v);
    store6(row + 6 * t, v);
    if (blockIdx.y == 0) {
      if (t < nrow) store6(G + 36 * (size_t)m.nb_off + 6 * (t - 6), v);
      else store6(Y + 6 * (size_t)p, v);
    }
  }
  if (tid == 0 && blockIdx.y == 0) {
#pragma unroll
    for (int r = 0; r < 6; ++r)
#pragma unroll
      for (int c = 0; c <= r; ++c) Lo[(size_t)p * 36 + r * 6 + c] = L[r * 6 + c];
    if (!ok) *bad = 1;
  }
  __syncthreads();
  // update rows: row i of block (k, l), then the update vector's blocks
  const int nblk = d * (d + 1) / 2, ntask = 6 * nblk + d;
  for (int t = blockIdx.y * TB + tid; t < ntask; t += TB * gridDim.y) {
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (t < 6 * nblk) {
      const int blk = t / 6, i = t - 6 * blk;
      int k = (int)((sqrtf(8.0f * (float)blk + 1.0f) - 1.0f) * 0.5f);
      while ((k + 1) * (k + 2) / 2 <= blk) ++k;
      while (k * (k + 1) / 2 > blk) --k;
      const int l = blk - k * (k + 1) / 2;
      for (int c = 0; c < m.n_child; ++c) {
        const FrontChild ch = childs[m.child_off + c];
        const int pk = maps[ch.map_off + k + 1], pl = maps[ch.map_off + l + 1];
        if (pk >= 0 && pl >= 0) add6(U + ch.u_off + 36 * (pk * (pk + 1) / 2 + pl) + 6 * i, v);
      }
      double g[6];
      load6(row + 36 * (k + 1) + 6 * i, g);
#pragma unroll
      for (int j = 0; j < 6; ++j) {
        double h[6];
        load6(row + 36 * (l + 1) + 6 * j, h);
#pragma unroll
        for (int q = 0; q < 6; ++q) v[j] -= g[q] * h[q];
      }
      store6(U + m.u_off + 36 * (size_t)blk + 6 * i, v);
    } else {
      const int k = t - 6 * nblk;
      for (int c = 0; c < m.n_child; ++c) {
        const FrontChild ch = childs[m.child_off + c];
        const int pk = maps[ch.map_off + k + 1];
        if (pk >= 0) add6(U + ch.u_off + 36 * ((size_t)ch.d * (ch.d + 1) / 2) + 6 * pk, v);
      }
      double y[6];
      load6(row + 6 * nrow, y);
#pragma unroll
      for (int i = 0; i < 6; ++i) {
        double h[6];
        load6(row + 36 * (k + 1) + 6 * i, h);
#pragma unroll
        for (int q = 0; q < 6; ++q) v[i] -= h[q] * y[q];
      }
      store6(U + m.u_off + 36 * (size_t)nblk + 6 * k, v);
    }
  }
}

// Forward substitution of another right-hand side with the stored factor
// (iterative refinement): one wavefront per front, the update vectors in the
// fronts' own vector slots.
__global__ void __launch_bounds__(64) k_front_forward(int first, const FrontMeta* __restrict__ meta,
                                                      const FrontChild* __restrict__ childs,
                                                      const int* __restrict__ maps, const double* __restrict__ b,
                                                      const double* __restrict__ G, const double* __restrict__ Lo,
                                                      double* U, double* __restrict__ Y) {
  const int p = first + blockIdx.x, lane = threadIdx.x;
  const FrontMeta m = meta[p];
  const int d = m.d;
  double y[6], L[36];
  load6(b + (size_t)m.pose * 6, y);
  for (int c = 0; c < m.n_child; ++c) {
    const FrontChild ch = childs[m.child_off + c];
    add6(U + ch.u_off + 36 * ((size_t)ch.d * (ch.d + 1) / 2), y);
  }
#pragma unroll
  for (int r = 0; r < 6; ++r)
#pragma unroll
    for (int c = 0; c <= r; ++c) L[r * 6 + c] = Lo[(size_t)p * 36 + r * 6 + c];
  row_solve(L, y);
  if (lane == 0) store6(Y + 6 * (size_t)p, y);
  double* u = U + m.u_off + 36 * ((size_t)d * (d + 1) / 2);
  for (int k = lane; k < d; k += 64) {
    double v[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    for (int c = 0; c < m.n_child; ++c) {
      const FrontChild ch = childs[m.child_off + c];
      const int pk = maps[ch.map_off + k + 1];
      if (pk >= 0) add6(U + ch.u_off + 36 * ((size_t)ch.d * (ch.d + 1) / 2) + 6 * pk, v);
    }
#pragma unroll
    for (int i = 0; i < 6; ++i) {
      double h[6];
      load6(G + 36 * (size_t)(m.nb_off + k) + 6 * i, h);
#pragma unroll
      for (int q = 0; q < 6; ++q) v[i] -= h[q] * y[q];
    }
    store6(u + 6 * k, v);
  }
}

// Backward substitution of one front by one wavefront: x = L^-T (y - sum_k
// G_k^T x_k), ten neighbours at a time (lane 6 g + j: neighbours g, g + 10,
// ..., component j), partials added in a fixed order.  s: 64 doubles of LDS.
__device__ __forceinline__ void front_backward(int p, int lane, const FrontMeta* __restrict__ meta,
                                               const int* __restrict__ nb, const double* __restrict__ G,
                                               const double* __restrict__ Lo, const double* __restrict__ Y,
                                               double* x, double* s) {
  const FrontMeta m = meta[p];
  const int g = lane / 6, j = lane - 6 * g;
  double acc = 0.0;
  if (g < 10)
    for (int k = g; k < m.d; k += 10) {
      const double* B = G + 36 * (size_t)(m.nb_off + k) + j;
      double xk[6];
      load6(x + 6 * (size_t)nb[m.nb_off + k], xk);
#pragma unroll
      for (int i = 0; i < 6; ++i) acc += B[6 * i] * xk[i];
    }
  s[lane] = acc;
  fold_wave_sync();
  double L[36], r[6];
#pragma unroll
  for (int i = 0; i < 6; ++i)
#pragma unroll
    for (int c = 0; c <= i; ++c) L[i * 6 + c] = Lo[(size_t)p * 36 + i * 6 + c];
  load6(Y + 6 * (size_t)p, r);
#pragma unroll
  for (int i = 0; i < 6; ++i) {
    double t = 0.0;
#pragma unroll
    for (int q = 0; q < 10; ++q) t += s[6 * q + i];
    r[i] -= t;
  }
#pragma unroll
  for (int i = 5; i >= 0; --i) {
#pragma unroll
    for (int k = i + 1; k < 6; ++k) r[i] -= L[k * 6 + i] * r[k];
    r[i] *= L[i * 7];
  }
  if (lane == 0) store6(x + 6 * (size_t)m.pose, r);
  fold_wave_sync();
}

// One level, four fronts per workgroup
__global__ void __launch_bounds__(256) k_back_level(int first, int count, const FrontMeta* __restrict__ meta,
                                                    const int* __restrict__ nb, const double* __restrict__ G,
                                                    const double* __restrict__ Lo, const double* __restrict__ Y,
                                                    double* x) {
  __shared__ double s[4][64];
  const int wv = threadIdx.x >> 6, q = blockIdx.x * 4 + wv;
  if (q < count) front_backward(first + q, threadIdx.x & 63, meta, nb, G, Lo, Y, x, s[wv]);
}

// Levels n_lvl-1 down to l0 (few fronts each) in one workgroup, a barrier
// between levels instead of a launch
__global__ void __launch_bounds__(1024) k_back_top(int l0, int n_lvl, const int* __restrict__ lvl,
                                                   const FrontMeta* __restrict__ meta, const int* __restrict__ nb,
                                                   const double* __restrict__ G, const double* __restrict__ Lo,
                                                   const double* __restrict__ Y, double* x) {
  __shared__ double s[16][64];
  const int wv = threadIdx.x >> 6;
  for (int l = n_lvl - 1; l >= l0; --l) {
    for (int p = lvl[l] + wv; p < lvl[l + 1]; p += 16)
      front_backward(p, threadIdx.x & 63, meta, nb, G, Lo, Y, x, s[wv]);
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

__global__ void k_direct_axpy(long long n, const double* __restrict__ a, double* __restrict__ y) {
  const long long t = (long long)blockIdx.x * blockDim.x + threadIdx.x;
  if (t < n) y[t] += a[t];
}

// ------------------------------------------------------------------ host
static_assert(front_lds_doubles(DirectLimits().max_d) * sizeof(double) <= 64 * 1024, "front column in LDS");

int SolverRun::direct_setup(hipStream_t st, const int32_t* h_kind, const int32_t* h_fi, const int32_t* h_fj) {
  direct_ready = false;
  // an explicit preconditioner choice asks for the PCG
  if (prm.pcg_segment > 0 || prm.pcg_coarse != 0 || !h_kind || F <= 0) return RPGO_OK;
  DirectPlan& P = plan;
  try {
    if (!build_direct_plan(N, F, h_kind, h_fi, h_fj, DirectLimits(), P)) return RPGO_OK;
  } catch (const std::bad_alloc&) {
    return RPGO_OK;
  }
  const size_t bytes[6] = {P.meta.size() * sizeof(FrontMeta), P.childs.size() * sizeof(FrontChild),
                           P.origs.size() * sizeof(FrontOrig), P.nb_pose.size() * sizeof(int32_t),
                           P.maps.size() * sizeof(int32_t), P.lvl.size() * sizeof(int)};
  const void* src[6] = {P.meta.data(), P.childs.data(), P.origs.data(), P.nb_pose.data(), P.maps.data(), P.lvl.data()};
  DevBuf* dst[6] = {&d_meta, &d_childs, &d_origs, &d_nb, &d_maps, &d_lvl};
  for (int k = 0; k < 6; ++k)
    if (dst[k]->reserve(bytes[k])) return RPGO_OK;  // no room: keep the iterative solve
  const size_t nblk = (size_t)(N + 63) / 64, ncost = (size_t)(F + 255) / 256;
  if (d_U.reserve(sizeof(double) * (size_t)P.u_len) || d_G.reserve(sizeof(double) * 36 * P.nb_pose.size()) ||
      d_L.reserve(sizeof(double) * 36 * (size_t)N) || d_Y.reserve(sizeof(double) * 6 * (size_t)N) ||
      d_part.reserve(sizeof(double) * (4 * nblk + ncost)) || d_bad.reserve(sizeof(int)))
    return RPGO_OK;
  if (!pinned_scalars()) return RPGO_OK;
  for (int k = 0; k < 6; ++k)
    if (bytes[k]) RPGO_HIP_CHECK(hipMemcpyAsync(dst[k]->ptr, src[k], bytes[k], hipMemcpyHostToDevice, st));
  RPGO_HIP_CHECK(hipMemsetAsync(d_bad.ptr, 0, sizeof(int), st));
  direct_ready = true;
  return RPGO_OK;
}

// Factor H + lambda damp and substitute forward with b: one launch per level.
int SolverRun::direct_factor(hipStream_t st, double lambda) {
  const DirectPlan& P = plan;
  for (int l = 0; l < P.levels(); ++l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first, d = P.lvl_max_d[l];
    const size_t lds = front_lds_doubles(d) * sizeof(double);
#define RPGO_FRONT_ARGS                                                                                       \
  first, d_meta.as<FrontMeta>(), d_childs.as<FrontChild>(), d_origs.as<FrontOrig>(), d_maps.as<int>(),        \
      D.as<double>(), hdiag.as<double>(), b64.as<double>(), Hij.as<double>(), lambda, prm.lm_diagonal_damping, \
      d_U.as<double>(), d_G.as<double>(), d_L.as<double>(), d_Y.as<double>(), d_bad.as<int>()
    if (d <= 4) {
      k_front<64><<<n, 64, lds, st>>>(RPGO_FRONT_ARGS);
    } else {
      // wide fronts of a narrow level share their update rows among
      // workgroups, each repeating the pivot column
      const int rounds = (3 * d * (d + 1) + d + 255) / 256;
      const int split = std::max(1, std::min(rounds, 1024 / n));
      k_front<256><<<dim3(n, split), 256, lds, st>>>(RPGO_FRONT_ARGS);
    }
#undef RPGO_FRONT_ARGS
  }
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

int SolverRun::direct_backward(hipStream_t st, double* out) {
  const DirectPlan& P = plan;
  // levels of at most kTop fronts from the top down in one workgroup
  constexpr int kTop = 48;
  int l0 = P.levels();
  while (l0 > 0 && P.lvl[l0] - P.lvl[l0 - 1] <= kTop) --l0;
  if (l0 < P.levels())
    k_back_top<<<1, 1024, 0, st>>>(l0, P.levels(), d_lvl.as<int>(), d_meta.as<FrontMeta>(), d_nb.as<int>(),
                                   d_G.as<double>(), d_L.as<double>(), d_Y.as<double>(), out);
  for (int l = l0 - 1; l >= 0; --l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first;
    k_back_level<<<(n + 3) / 4, 256, 0, st>>>(first, n, d_meta.as<FrontMeta>(), d_nb.as<int>(), d_G.as<double>(),
                                              d_L.as<double>(), d_Y.as<double>(), out);
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

// One refinement step: dx += (H + lambda damp)^-1 r with the stored factor
int SolverRun::direct_refine(hipStream_t st) {
  const DirectPlan& P = plan;
  for (int l = 0; l < P.levels(); ++l) {
    const int first = P.lvl[l], n = P.lvl[l + 1] - first;
    k_front_forward<<<n, 64, 0, st>>>(first, d_meta.as<FrontMeta>(), d_childs.as<FrontChild>(), d_maps.as<int>(),
                                      r.as<double>(), d_G.as<double>(), d_L.as<double>(), d_U.as<double>(),
                                      d_Y.as<double>());
  }
  int rc;
  if ((rc = direct_backward(st, zv.as<double>()))) return rc;
  const long long n6 = 6ll * N;
  k_direct_axpy<<<(unsigned)((n6 + 255) / 256), 256, 0, st>>>(n6, zv.as<double>(), dx.as<double>());
  RPGO_HIP_CHECK(hipGetLastError());
  return RPGO_OK;
}

// One linear step by the factorization, the step's candidate poses xn and
// their weighted cost: *lin the model decrease b.dx - dx.H dx / 2 (undamped
// H), *cost_new the cost.  *ok = false when a pivot was not positive or the
// residual stayed large: the caller then takes the iterative solve.
int SolverRun::direct_step(hipStream_t st, double lambda, double* lin, double* cost_new, bool* ok) {
  int rc;
  double* h = pinned_scalars();
  const int nblk = (N + 63) / 64, ncost = (F + 255) / 256;
  double* cpart = d_part.as<double>() + 4 * (size_t)nblk;
  *ok = false;
  double prev = INFINITY;
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
    *lin = bdx - 0.5 * xhx;
    *cost_new = h[36];
    last_residual = bb > 0.0 ? std::sqrt(rr / bb) : 0.0;
    if (!(rr == rr) || !(last_residual < 1e-2)) return RPGO_OK;
    // done at the tolerance, after the last refinement, or when a refinement
    // no longer gains (the residual's own rounding)
    const double tol = std::min(prm.pcg_rel_tol, kDirectTol);
    if (last_residual <= tol || refine == kDirectRefine || last_residual > 0.25 * prev) {
      *ok = true;
      return RPGO_OK;
    }
    prev = last_residual;
    if ((rc = direct_refine(st))) return rc;
    stats.pcg_iterations += 1;
  }
}

// One refinement of the accepted step that ends a nonlinear solve of a large
// graph, its poses in xn and their cost
int SolverRun::direct_finish(hipStream_t st, double lambda, double* cost_new) {
  if (N < kDirectFinishMin) return RPGO_OK;
  int rc;
  if ((rc = direct_check(st, lambda))) return rc;  // the residual of the step in dx
  if ((rc = direct_refine(st))) return rc;
  stats.pcg_iterations += 1;
  retract(st);
  return direct_cost(st, xn.as<double>(), cost_new);
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
