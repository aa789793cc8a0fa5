// Internal state of the robust pose-graph solve (solver.hip).
#pragma once

#include <cstring>

#include "direct_plan.h"
#include "rpgo_internal.h"

namespace rpgo {

constexpr int kPcgChunk = 8;       // PCG iterations per captured graph launch
constexpr int kCoarseSegMax = 256;  // rigid segments of the coarse preconditioner level (maximum)
constexpr int kCoarseSegSmall = 128;  // default below kCoarseLargeN poses
constexpr int kCoarseLargeN = 10000;  // poses from which the default is kCoarseSegMax
constexpr int kCoarseMax = 6 * kCoarseSegMax;
// A direct solve is refined to this relative residual (or pcg_rel_tol where
// that is smaller), in at most kDirectRefine steps.  A factorization's
// residual is rounding spread over every mode, so the soft modes of a long
// chain need it smaller than a PCG's: 50,000 poses with 1,600 loop closures
// stopped 1.4e-7 (relative) from the converged steps at 1e-6, 5e-9 at 1e-10.
constexpr double kDirectTol = 1e-10;
constexpr int kDirectRefine = 3;
// and accepted at pcg_rel_tol or this, whichever is larger: the residual's own
// rounding, which a refinement cannot lower, ends at 7e-10 on 18 drawn graphs
// and at 4e-9 on chains held by a weak prior.  Above, the step is the PCG's.
constexpr double kDirectAccept = 1e-8;
// From this many poses the last step of a nonlinear solve gets one more
// refinement.  The factor takes damping and diagonal rounded to one FP64
// number, an error of about 1e-16 of the diagonal with the same sign at every
// pose; along the softest mode of 50,000 poses that shortens a step by 8e-5,
// 3e-8 of the poses when it is the last (earlier steps' errors are corrected
// by the later ones).  Below, the bias is far under the solve's 1e-10.
constexpr int kDirectFinishMin = 8192;
// A factor below this weight does not hold a pose (poses_held): the noise of
// singular systems reaches 1e-9 of the diagonal, a factor of 1e3 below.
constexpr double kHoldWeight = 1e-6;
// A step is undamped up to this lambda: lambda damp is lost in the FP64
// diagonal (LM reaches 1e-20 to 1e-66 in GNC's later solves).  Down to 1e-14 a
// free graph's direct and PCG steps move it alike to a tenth, at 1e-15 to a
// sixth, at 1e-16 to a third.
constexpr double kUndamped = 1e-16;

struct GraphKey {
  int N = 0, S = 0, Sc = 0, nseg_c = 0;
  const void *hist = nullptr, *p = nullptr, *Minv = nullptr, *Hij = nullptr, *inc = nullptr,
             *inc_q = nullptr, *Ainv = nullptr, *Pb = nullptr, *Ds = nullptr, *ext = nullptr;
  bool operator==(const GraphKey& o) const {
    return N == o.N && S == o.S && Sc == o.Sc && nseg_c == o.nseg_c && hist == o.hist && p == o.p &&
           Minv == o.Minv && Hij == o.Hij && inc == o.inc && inc_q == o.inc_q && Ainv == o.Ainv &&
           Pb == o.Pb && Ds == o.Ds && ext == o.ext;
  }
};

struct SolverRun {
  struct Stats {
    int lm_iterations = 0;
    int lm_rejections = 0;
    int pcg_iterations = 0;
    int linearizations = 0;
    double mu_init = -1.0;
  };
  int N = 0, F = 0, n_known = 0;
  rpgo_solve_params prm{};
  Stats stats;
  // problem (device)
  DevBuf x0, x, xn;             // FP64 poses
  DevBuf kind, fi, fj, z, info;  // factors
  DevBuf w, barc, known, err, cost;
  // Gauss-Newton system
  DevBuf Hii, Hjj, Hij, gi, gj;  // per-factor contributions
  DevBuf inc_off, inc_cnt, inc;  // pose -> incident factors
  DevBuf inc_q;                  // per incidence: the factor's other pose (-1: not a between factor)
  DevBuf D, Minv, hdiag, b64;
  DevBuf chain, Useg;             // odometry chain links, preconditioner off-diagonals
  DevBuf Ds, Cs;                  // entry-major diagonal and chain-link blocks (chain SpMV)
  DevBuf ext_off, ext, ext_q;     // per pose: between incidences that are not chain links
  DevBuf dx, r, zv, p, q, hx;     // PCG vectors (FP64)
  DevBuf sc;                      // FP64 scalars
  DevBuf hist;                    // PCG residual history (per iteration)
  DevBuf Pb, Ac, Lci, Ainv, cres, ccor;  // coarse level: prolongation blocks, coarse matrix,
                                     // its inverse factor, FP32 inverse, coarse vectors
  DevBuf LcT;                        // the coarse Cholesky factor transposed (column access)
  bool polish = false;               // refinement pass: a step that raises the cost is rejected
  hipGraphExec_t graph_exec = nullptr;  // captured PCG chunk
  GraphKey graph_key;
  bool use_graphs = true;
  // direct solve (direct.hip): the plan of the current problem, its device
  // copy, and the factor's storage
  bool direct_ready = false;
  int held_always = -1;            // every pose held whatever GNC's weights become (-1: not known)
  DirectPlan plan;
  DevBuf d_meta, d_childs, d_origs, d_rows, d_maps;
  DevBuf d_U, d_G, d_part, d_bad;
  // pinned host buffers of this run's readbacks (scalars; one PCG chunk's
  // residual history), allocated on first use
  double* h_scalars = nullptr;
  double* h_history = nullptr;

  int alloc(int N_, int F_);
  void spmv_dev(hipStream_t st, const double* lam, const double* x, double* y);
  int build_incidence(hipStream_t st);
  int linearize(hipStream_t st);
  void spmv(hipStream_t st, double lambda, const double* x, double* y);
  int pcg(hipStream_t st, double lambda, int* iters);
  int coarse_setup(hipStream_t st, double lambda, int* Sc, int* nseg);
  void pcg_step(hipStream_t st, int S, int Sc, int nseg_c, int first, int a);
  int model_decrease(hipStream_t st, double* out);
  int total_cost(hipStream_t st, const double* xp, double* out);
  int compute_errors(hipStream_t st, const double* xp);
  int nonlinear_solve(hipStream_t st, const rpgo_solve_problem* pr, bool from_x0, double* cost, int* iters);
  int read_scalars(hipStream_t st, int count, double* out);
  double* pinned_scalars();
  double* pinned_history();
  void retract(hipStream_t st);
  void cost_partials(hipStream_t st, const double* xp, double* part);
  int direct_setup(hipStream_t st, const rpgo_solve_problem* pr);
  int poses_held_now(hipStream_t st, const rpgo_solve_problem* pr, int* held);
  int direct_factor(hipStream_t st, double lambda);
  int direct_backward(hipStream_t st, double* out);
  int direct_check(hipStream_t st, double lambda);
  int direct_refine(hipStream_t st);
  int direct_step(hipStream_t st, double lambda, double* lin, double* cost_new, bool* ok);
  int direct_finish(hipStream_t st, double lambda, double* cost_new);
  bool last_step(double cur, double nw, int it) const;
  int direct_cost(hipStream_t st, const double* xp, double* out);
  int run(hipStream_t st, const rpgo_solve_problem* pr, rpgo_solve_report* rep);
  double* cost_buf() { return cost.as<double>(); }
  void direct_release() {
    direct_ready = false;
    for (DevBuf* v : {&d_meta, &d_childs, &d_origs, &d_rows, &d_maps, &d_U, &d_G, &d_part, &d_bad}) v->release();
  }
  void release() {
    direct_release();
    if (graph_exec) (void)hipGraphExecDestroy(graph_exec);
    graph_exec = nullptr;
    if (h_scalars) (void)hipHostFree(h_scalars);
    if (h_history) (void)hipHostFree(h_history);
    h_scalars = h_history = nullptr;
    for (DevBuf* v : {&hist,&x0, &x, &xn, &kind, &fi, &fj, &z, &info, &w, &barc, &known, &err, &cost, &Hii,
                      &Hjj, &Hij, &gi, &gj, &inc_off, &inc_cnt, &inc, &inc_q, &D, &Minv, &hdiag, &b64,
                      &chain, &Useg, &Ds, &Cs, &ext_off, &ext, &ext_q, &Pb, &Ac, &Lci, &LcT, &Ainv, &cres,
                      &ccor,
                      &dx, &r, &zv, &p, &q, &hx, &sc})
      v->release();
  }
};

// chi^2 quantile (inverse regularized lower incomplete gamma), host side
double chi2_quantile(double p, double dof);

}  // namespace rpgo
