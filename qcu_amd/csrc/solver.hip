// solver.hip -- even-odd BiCGSTAB on the odd-site Schur system for a batch of
// systems, FP64 or mixed precision with FP64 reliable updates.
//
// Schur form (symmetric, reducing to include/lattice_bistabcg.h:99-132 and
// src/bistabcg.cu:73-96 for Wilson, A = 1):
//   Mhat x_o = x_o - kappa^2 Ao^-1 D_oe Ae^-1 D_eo x_o
//   bhat     = Ao^-1 (b_o + kappa D_oe Ae^-1 b_e)
//   x_e      = Ae^-1 (b_e + kappa D_eo x_o)
// The recurrence is the reference's (include/lattice_bistabcg.h:227-307).  Its
// scalars stay on the device, one state per system; the host looks at them
// once per chunk of iterations, and a chunk is captured once as a hipGraph and
// replayed.  Systems that stop are skipped by every kernel until the batch
// is done.
#include <chrono>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#include "../../include/qcu.h"
#include "qcu_lattice.h"
#include "qcu_solver.h"

namespace qcu {

// QCU_TRACE=1 prints the wall time of every solver phase to stderr
struct PhaseTrace {
  bool on;
  hipStream_t s;
  std::chrono::steady_clock::time_point t;
  explicit PhaseTrace(hipStream_t st)
      : on(getenv("QCU_TRACE") != nullptr), s(st), t(std::chrono::steady_clock::now()) {}
  void mark(const char *what) {
    if (!on) return;
    (void)hipStreamSynchronize(s);
    auto n = std::chrono::steady_clock::now();
    fprintf(stderr, "[qcu] %-28s %9.3f ms\n", what, std::chrono::duration<double, std::milli>(n - t).count());
    t = n;
  }
};

// ---------------------------------------------------------------- work space
int VecSet::create(int prec_, int px_, int n, bool precond) {
  prec = prec_;
  px = px_;
  QCU_TRY(r.create(prec, n));
  QCU_TRY(rt.create(prec, n));
  QCU_TRY(p.create(prec, n));
  QCU_TRY(v.create(prec, n));
  QCU_TRY(s.create(prec, n));
  QCU_TRY(t.create(prec, n));
  QCU_TRY(tmp.create(prec, n));
  QCU_TRY(x.create(px, n));
  if (precond) {
    QCU_TRY(ph.create(prec, n));
    QCU_TRY(sh.create(prec, n));
  }
  return 0;
}

VecSet::~VecSet() {
  for (auto &kv : graphs) (void)hipGraphExecDestroy(kv.second);
}

int Solver::init(const BatchOp *op_, hipStream_t s) {
  op = op_;
  stream = s;
  QCU_CHECK(op->nvsites < (1LL << 31), QCU_ERR_DIMS, "batch too large");
  n = (int)op->nvsites;
  nsys = op->nsys;
  QCU_TRY(be.create(P64, n));
  QCU_TRY(bo.create(P64, n));
  QCU_TRY(bh.create(P64, n));
  QCU_TRY(xe.create(P64, n));
  QCU_TRY(xo.create(P64, n));
  QCU_TRY(r64.create(P64, n));
  QCU_TRY(t64.create(P64, n));
  // partials of the smallest block size (64) used by any reducing kernel
  const size_t npart = (size_t)(op->max_blocks(64) + 1) * kMaxRhs * 4;
  const size_t bytes = npart * sizeof(double) + nsys * sizeof(SysState) + 4 * nsys * sizeof(double) + 256;
  QCU_TRY(scratch.alloc(bytes));
  char *base = (char *)scratch.p;
  partials = (double *)base;
  base += npart * sizeof(double);
  st = (SysState *)base;
  base += nsys * sizeof(SysState);
  dscal = (double *)base;
  QCU_HIP(hipMemsetAsync(scratch.p, 0, bytes, stream));
  QCU_HIP(hipHostMalloc((void **)&host_st, nsys * sizeof(SysState), hipHostMallocDefault));
  QCU_HIP(hipHostMalloc((void **)&host_scal, 4 * nsys * sizeof(double), hipHostMallocDefault));
  QCU_HIP(hipStreamSynchronize(stream));
  return 0;
}

Solver::~Solver() {
  sets.clear();
  if (host_st) (void)hipHostFree(host_st);
  if (host_scal) (void)hipHostFree(host_scal);
}

VecSet *Solver::get_set(int prec, bool precond, int *rc) {
  const int key = prec * 2 + (precond ? 1 : 0);
  auto it = sets.find(key);
  if (it != sets.end()) return it->second.get();
  std::unique_ptr<VecSet> vs(new VecSet());
  const int px = (prec == P64) ? P64 : P32;
  *rc = vs->create(prec, px, n, precond);
  if (*rc) return nullptr;
  VecSet *raw = vs.get();
  sets[key] = std::move(vs);
  return raw;
}

// ---------------------------------------------------------------- operators
// Mhat x (FP64) into out; tmp is scratch
static int apply_mhat64(Solver &S, SpinorPtr out, SpinorPtr x, SpinorPtr tmp) {
  const BatchOp &op = *S.op;
  const LaunchCfg cfg = tuned_cfg(op, P64);
  SpinorPtr none{};
  QCU_TRY(hop(op, P64, tmp, x, 0, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg, S.stream));
  QCU_TRY(hop(op, P64, out, tmp, 1, EPI_XPAY, x, RED_NONE, none, nullptr, nullptr, cfg, S.stream));
  return 0;
}

// one BiCGSTAB iteration of every running system, no host interaction
static int enqueue_iteration(Solver &S, VecSet &V, Precond *K) {
  const BatchOp &op = *S.op;
  const int prec = V.prec;
  const LaunchCfg cfg = tuned_cfg(op, prec);
  SysState *st = S.st;
  SpinorPtr none{};
  QCU_TRY(bicg_p_update(op, V.p.ptr(), V.r.ptr(), V.v.ptr(), prec, st, S.stream));
  SpinorPtr pin = V.p.ptr();
  if (K) {
    QCU_TRY(K->apply(S, V.ph.ptr(), V.p.ptr(), prec, st));
    pin = V.ph.ptr();
  }
  QCU_TRY(hop(op, prec, V.tmp.ptr(), pin, 0, EPI_PLAIN, none, RED_NONE, none, st, nullptr, cfg, S.stream));
  QCU_TRY(hop(op, prec, V.v.ptr(), V.tmp.ptr(), 1, EPI_XPAY, pin, RED_DOT_Y_OUT, V.rt.ptr(), st, S.partials, cfg,
              S.stream));
  QCU_TRY(bicg_s_update(op, V.s.ptr(), V.r.ptr(), V.v.ptr(), prec, st, S.stream));
  SpinorPtr sin = V.s.ptr();
  if (K) {
    QCU_TRY(K->apply(S, V.sh.ptr(), V.s.ptr(), prec, st));
    sin = V.sh.ptr();
  }
  QCU_TRY(hop(op, prec, V.tmp.ptr(), sin, 0, EPI_PLAIN, none, RED_NONE, none, st, nullptr, cfg, S.stream));
  if (K) {
    // t = Mhat s_hat; omega = <t, s> / <t, t> needs s, not s_hat
    QCU_TRY(hop(op, prec, V.t.ptr(), V.tmp.ptr(), 1, EPI_XPAY, sin, RED_NONE, none, st, nullptr, cfg, S.stream));
    QCU_TRY(omega_dot(op, V.t.ptr(), V.s.ptr(), prec, st, S.partials, S.stream));
    QCU_TRY(bicg_xr_update_pc(op, V.x.ptr(), V.px, V.r.ptr(), V.rt.ptr(), V.ph.ptr(), V.sh.ptr(), V.s.ptr(),
                              V.t.ptr(), prec, st, S.partials, S.stream));
  } else {
    QCU_TRY(hop(op, prec, V.t.ptr(), V.tmp.ptr(), 1, EPI_XPAY, sin, RED_OUT_X, none, st, S.partials, cfg,
                S.stream));
    QCU_TRY(bicg_xr_update(op, V.x.ptr(), V.px, V.r.ptr(), V.rt.ptr(), V.p.ptr(), V.s.ptr(), V.t.ptr(), prec, st,
                           S.partials, S.stream));
  }
  return 0;
}

// `n` iterations: small batches without a preconditioner in five launches each
// (FP64, FP32; an even number, since p changes places with every iteration)
static bool split_chunk(const Solver &S, const VecSet &V, const Precond *K, int n) {
  return !K && V.prec != P16 && V.px == V.prec && n % 2 == 0 && hop_is_split(*S.op, tuned_cfg(*S.op, V.prec));
}

static int prepare_split(Solver &S, VecSet &V) {
  QCU_TRY(V.p2.create(V.prec, S.n));
  const size_t part = (size_t)(S.op->max_blocks(64) + 1) * kMaxRhs * 3 * sizeof(double);
  return V.split_buf.alloc(2 * part + S.nsys * sizeof(SysState));
}

// split: as split_chunk() said when prepare_split() made room for it.  Asked again, it
// may say something else: another thread's tuning changes the shapes at any time.
static int enqueue_chunk(Solver &S, VecSet &V, Precond *K, int n, bool split) {
  if (!split) {
    for (int k = 0; k < n; ++k) QCU_TRY(enqueue_iteration(S, V, K));
    return 0;
  }
  const size_t part = (size_t)(S.op->max_blocks(64) + 1) * kMaxRhs * 3;
  double *buf = (double *)V.split_buf.p;
  SplitIter it;
  it.p[0] = V.p.ptr();
  it.p[1] = V.p2.ptr();
  it.r = V.r.ptr();
  it.rt = V.rt.ptr();
  it.v = V.v.ptr();
  it.s = V.s.ptr();
  it.t = V.t.ptr();
  it.tmp = V.tmp.ptr();
  it.x = V.x.ptr();
  it.st[0] = S.st;
  it.st[1] = (SysState *)(buf + 2 * part);
  it.part[0] = buf;
  it.part[1] = buf + part;
  return split_iterations(*S.op, V.prec, it, n, S.stream);
}

static int run_chunk(Solver &S, VecSet &V, Precond *K, int chunk, bool use_graph) {
  const bool split = split_chunk(S, V, K, chunk);
  if (split) QCU_TRY(prepare_split(S, V));
  if (!use_graph) return enqueue_chunk(S, V, K, chunk, split);
  if (V.graph_tune != tune_generation()) {
    // the graphs hold the launch shapes of their capture: a newly tuned (or
    // set) shape needs new graphs
    for (auto &g : V.graphs) (void)hipGraphExecDestroy(g.second);
    V.graphs.clear();
    V.graph_tune = tune_generation();
  }
  if (K && V.graph_net != K->uid()) {
    // graphs captured with another preconditioner hold its device buffers: drop them all
    for (auto g = V.graphs.begin(); g != V.graphs.end();) {
      if (g->first & 1) {
        (void)hipGraphExecDestroy(g->second);
        g = V.graphs.erase(g);
      } else {
        ++g;
      }
    }
    V.graph_net = K->uid();
  }
  const long key = ((long)chunk << 8) | (K ? 1 : 0);
  auto it = V.graphs.find(key);
  if (it == V.graphs.end()) {
    hipGraph_t graph;
    QCU_HIP(hipStreamBeginCapture(S.stream, hipStreamCaptureModeThreadLocal));
    const int rc = enqueue_chunk(S, V, K, chunk, split);
    hipError_t e = hipStreamEndCapture(S.stream, &graph);
    if (rc) return rc;
    QCU_HIP(e);
    hipGraphExec_t exec;
    QCU_HIP(hipGraphInstantiate(&exec, graph, nullptr, nullptr, 0));
    (void)hipGraphDestroy(graph);
    V.graphs[key] = exec;
    it = V.graphs.find(key);
  }
  QCU_HIP(hipGraphLaunch(it->second, S.stream));
  return 0;
}

static int read_states(Solver &S) {
  QCU_HIP(hipMemcpyAsync(S.host_st, S.st, S.nsys * sizeof(SysState), hipMemcpyDeviceToHost, S.stream));
  QCU_HIP(hipStreamSynchronize(S.stream));
  return 0;
}

static int write_states(Solver &S) {
  QCU_HIP(hipMemcpyAsync(S.st, S.host_st, S.nsys * sizeof(SysState), hipMemcpyHostToDevice, S.stream));
  return 0;
}

// How many iterations until a running system needs the host: from the mean
// decrease of its residual per iteration so far.  Iterations launched beyond that
// only run kernels that return at once, but each costs its launches (60 us at
// 32^3x64, where a reliable update every 3 or 4 iterations would waste as many).
struct Pace {
  std::vector<double> lrr, rate;  // log |r|^2 when last seen, its decrease per iteration (0: unknown)
  std::vector<int> iter;
  Pace(const SysState *hs, int nsys) : lrr(nsys), rate(nsys, 0.0), iter(nsys) { restarted(hs, nsys); }
  void restarted(const SysState *hs, int nsys) {
    for (int k = 0; k < nsys; ++k) {
      lrr[k] = std::log(hs[k].rr);
      iter[k] = hs[k].iter;
    }
  }
  void seen(const SysState *hs, int nsys) {
    for (int k = 0; k < nsys; ++k) {
      const int n = hs[k].iter - iter[k];
      if (n <= 0) continue;
      const double l = std::log(hs[k].rr);
      rate[k] = (lrr[k] - l) / n;
      lrr[k] = l;
      iter[k] = hs[k].iter;
    }
  }
  int next(const SysState *hs, int nsys, int chunk, bool pairs) const {
    int n = 1;
    for (int k = 0; k < nsys; ++k) {
      if (hs[k].done != 0) continue;
      const double target = std::max(hs[k].rr_stop, hs[k].delta2 * hs[k].rr_ref);
      const double need = (std::log(hs[k].rr) - std::log(target)) / rate[k];
      // unknown, or no decrease: half a chunk where updates are expected, else all of it
      int m = hs[k].delta2 > 0 ? (chunk + 1) / 2 : chunk;
      if (rate[k] > 0 && std::isfinite(need)) m = need >= chunk ? chunk : (need > 1 ? (int)std::ceil(need) : 1);
      n = std::max(n, m);
    }
    return pairs ? (n + 1) & ~1 : n;
  }
};

// Solve Mhat x_o = bhat (bhat in S.bh) for the systems with active[k]; the
// solution accumulates in S.xo (FP64): the iterated correction V.x is folded
// into it at every reliable update.  warm: start from the current S.xo.
// A system stops when |bhat - Mhat x_o|^2 < target2[k] (recomputed in FP64).
static int schur_solve(Solver &S, int prec, const std::vector<double> &target2, double delta, int max_iter,
                       int chunk, bool adaptive, bool use_graph, Precond *K, bool warm, const std::vector<int> &active,
                       std::vector<SolveStats> &stats) {
  const BatchOp &op = *S.op;
  const int nsys = S.nsys;
  int rc = 0;
  VecSet *V = S.get_set(prec, K != nullptr, &rc);
  if (!V) return rc;
  SysState *hs = S.host_st;
  std::memset(hs, 0, nsys * sizeof(SysState));
  for (int k = 0; k < nsys; ++k) {
    hs[k].rr_stop = target2[k];
    hs[k].delta2 = (prec == P64) ? 0.0 : delta * delta;
    hs[k].done = active[k] ? 0 : 4;
  }
  QCU_TRY(write_states(S));
  SpinorPtr src = S.bh.ptr();
  if (warm) {
    QCU_TRY(apply_mhat64(S, S.r64.ptr(), S.xo.ptr(), S.t64.ptr()));
    QCU_TRY(xmy_norm(op, S.bh.ptr(), S.r64.ptr(), S.st, S.partials, 0, S.stream));
    src = S.r64.ptr();
  } else {
    QCU_TRY(zero_spinor(op, S.xo.ptr(), P64, S.stream));
  }
  // V.x = 0, r = src, r~ = r, p = v = 0
  QCU_TRY(bicg_init(op, V->r.ptr(), V->rt.ptr(), V->p.ptr(), V->v.ptr(), V->x.ptr(), prec, src, S.st, S.partials,
                    S.stream));
  QCU_TRY(read_states(S));
  PhaseTrace trace(S.stream);
  trace.mark("  init");
  std::vector<int> stuck(nsys, 0);
  for (int k = 0; k < nsys; ++k) stats[k] = SolveStats{0, 0, 0, 0};
  Pace pace(hs, nsys);
  const bool pairs = split_chunk(S, *V, K, 2);  // iterations come in pairs
  int iters = 0;
  bool folded = false;  // V.x is zero
  for (;;) {
    bool running = false, pending = false;
    for (int k = 0; k < nsys; ++k) {
      running = running || hs[k].done == 0;
      pending = pending || (hs[k].done >= 1 && hs[k].done <= 3);
    }
    if (!running && !pending) break;
    if (!pending) {
      const int n = std::min(adaptive ? pace.next(hs, nsys, chunk, pairs) : chunk, max_iter - iters);
      if (n <= 0) break;
      folded = false;
      QCU_TRY(run_chunk(S, *V, K, n, use_graph && n == chunk));
      QCU_TRY(read_states(S));
      pace.seen(hs, nsys);
      for (int k = 0; k < nsys; ++k) iters = std::max(iters, hs[k].iter);
      trace.mark("  chunk");
      continue;
    }
    // reliable update of every system still in the batch: fold the correction into
    // the FP64 solution and recompute the residual in FP64 (this is also the
    // convergence check), with the scalars of a continued recurrence
    std::vector<int> why(nsys);
    for (int k = 0; k < nsys; ++k) why[k] = hs[k].done;
    QCU_TRY(fold(op, V->x.ptr(), V->px, S.xo.ptr(), S.stream));
    folded = true;
    {
      const LaunchCfg cfg = tuned_cfg(op, P64);
      SpinorPtr none{};
      QCU_TRY(hop(op, P64, S.t64.ptr(), S.xo.ptr(), 0, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg,
                  S.stream));
      QCU_TRY(hop(op, P64, S.r64.ptr(), S.t64.ptr(), 1, EPI_XPAY, S.xo.ptr(), RED_RES, S.bh.ptr(), S.st, S.partials,
                  cfg, S.stream));
    }
    QCU_TRY(reliable_residual(op, V->r.ptr(), V->rt.ptr(), S.r64.ptr(), prec, S.st, S.partials, S.stream));
    QCU_TRY(read_states(S));
    bool restart = false, left = false;
    for (int k = 0; k < nsys; ++k) {
      if (why[k] == 4) continue;
      stats[k].reliable += 1;
      stats[k].iters = hs[k].iter;
      const double rr_true = hs[k].tmp[0];
      int d = 0;
      if (rr_true < target2[k]) {
        d = 4;
        stats[k].converged = 1;
      } else if (hs[k].iter >= max_iter || !std::isfinite(rr_true)) {
        d = 4;
      } else if (why[k] == 1 && ++stuck[k] > 8) {
        d = 4;  // the iterated residual keeps claiming convergence: a precision floor
      } else if (why[k] == 2 && ++stats[k].restarts > 20) {
        d = 4;
      }
      if (d == 0 && why[k] == 1) hs[k].rr_stop = std::min(hs[k].rr_stop, target2[k]) * 0.01;
      if (d == 0 && why[k] == 2) restart = true;
      left = left || d == 0;
      hs[k].done = d;
    }
    if (!left) {
      trace.mark("  reliable update");
      break;
    }
    if (restart) {
      // a breakdown restarts the Krylov spaces of the batch from the current residuals
      QCU_TRY(spinor_convert(op, V->rt.ptr(), prec, S.r64.ptr(), S.stream));
      QCU_TRY(zero_spinor(op, V->p.ptr(), prec, S.stream));
      QCU_TRY(zero_spinor(op, V->v.ptr(), prec, S.stream));
      for (int k = 0; k < nsys; ++k) {
        hs[k].rho_prev[0] = 1;
        hs[k].rho_prev[1] = 0;
        hs[k].alpha[0] = hs[k].omega[0] = 1;
        hs[k].alpha[1] = hs[k].omega[1] = 0;
      }
      QCU_TRY(write_states(S));
      QCU_TRY(reliable_residual(op, V->r.ptr(), V->rt.ptr(), S.r64.ptr(), prec, S.st, S.partials, S.stream));
      QCU_TRY(read_states(S));
    }
    for (int k = 0; k < nsys; ++k)
      if (hs[k].done == 0) hs[k].done = !std::isfinite(hs[k].rr) ? 2 : (hs[k].rr < hs[k].rr_stop ? 1 : 0);
    QCU_TRY(write_states(S));
    pace.restarted(hs, nsys);
    trace.mark("  reliable update");
  }
  if (!folded) QCU_TRY(fold(op, V->x.ptr(), V->px, S.xo.ptr(), S.stream));
  for (int k = 0; k < nsys; ++k) stats[k].iters = std::max(stats[k].iters, hs[k].iter);
  return 0;
}

// ---------------------------------------------------------------- CG on the normal equations
// CGNR on the odd Schur system: CG on Mhat^+ Mhat x_o = Mhat^+ bhat in FP64, with
//   Mhat^+ = 1 - kappa^2 gamma5 D_oe Ae^-1 D_eo gamma5 Ao^-1
// (gamma5-hermiticity of the hop, A Hermitian and commuting with gamma5).  The
// stop test uses the Schur residual |bhat - Mhat x_o|^2 carried by the
// recursion res -= alpha Mhat p.  Scalars stay on the device (per system).
static int cgnr_iteration(Solver &S) {
  const BatchOp &op = *S.op;
  const LaunchCfg cfg = tuned_cfg(op, P64);
  SysState *st = S.st;
  SpinorPtr none{};
  const SpinorPtr z = S.cg_z.ptr(), p = S.cg_p.ptr(), q = S.cg_q.ptr(), t1 = S.t64.ptr(), t2 = S.xe.ptr();
  // q = Mhat p ; alpha = rho / |q|^2
  QCU_TRY(hop(op, P64, t1, p, 0, EPI_PLAIN, none, RED_NONE, none, st, nullptr, cfg, S.stream));
  QCU_TRY(hop(op, P64, q, t1, 1, EPI_XPAY, p, RED_NONE, none, st, nullptr, cfg, S.stream));
  QCU_TRY(cg_qnorm(op, q, st, S.partials, S.stream));
  // x += alpha p ; res -= alpha q ; |res|^2
  QCU_TRY(cg_xr(op, S.xo.ptr(), S.r64.ptr(), p, q, st, S.partials, S.stream));
  // z = Mhat^+ res ; beta = |z|^2 / rho ; p = z + beta p
  QCU_TRY(g5_clinv(op, t1, S.r64.ptr(), st, S.stream));
  QCU_TRY(hop(op, P64, t2, t1, 0, EPI_PLAIN, none, RED_NONE, none, st, nullptr, cfg, S.stream, true));
  QCU_TRY(hop(op, P64, t1, t2, 1, EPI_PLAIN, none, RED_NONE, none, st, nullptr, cfg, S.stream, false));
  QCU_TRY(cg_z(op, z, S.r64.ptr(), t1, FK_CG_RHO, st, S.partials, S.stream));
  QCU_TRY(cg_p(op, p, z, st, S.stream));
  return 0;
}

static int cgnr_solve(Solver &S, const std::vector<double> &target2, int max_iter, int chunk, bool warm,
                      const std::vector<int> &active, std::vector<SolveStats> &stats) {
  const BatchOp &op = *S.op;
  const int nsys = S.nsys;
  if (!S.cg_z.data.p) {
    QCU_TRY(S.cg_z.create(P64, S.n));
    QCU_TRY(S.cg_p.create(P64, S.n));
    QCU_TRY(S.cg_q.create(P64, S.n));
  }
  SysState *hs = S.host_st;
  std::memset(hs, 0, nsys * sizeof(SysState));
  for (int k = 0; k < nsys; ++k) {
    hs[k].rr_stop = target2[k];
    hs[k].done = active[k] ? 0 : 4;
  }
  QCU_TRY(write_states(S));
  const LaunchCfg cfg = tuned_cfg(op, P64);
  SpinorPtr none{};
  if (!warm) QCU_TRY(zero_spinor(op, S.xo.ptr(), P64, S.stream));
  // res = bhat - Mhat x_o, |res|^2 into tmp[0]
  QCU_TRY(apply_mhat64(S, S.r64.ptr(), S.xo.ptr(), S.t64.ptr()));
  QCU_TRY(xmy_norm(op, S.bh.ptr(), S.r64.ptr(), S.st, S.partials, 1, S.stream));
  // z = Mhat^+ res, rho = |z|^2, p = z
  QCU_TRY(g5_clinv(op, S.t64.ptr(), S.r64.ptr(), S.st, S.stream));
  QCU_TRY(hop(op, P64, S.xe.ptr(), S.t64.ptr(), 0, EPI_PLAIN, none, RED_NONE, none, S.st, nullptr, cfg, S.stream,
              true));
  QCU_TRY(hop(op, P64, S.t64.ptr(), S.xe.ptr(), 1, EPI_PLAIN, none, RED_NONE, none, S.st, nullptr, cfg, S.stream,
              false));
  QCU_TRY(cg_z(op, S.cg_z.ptr(), S.r64.ptr(), S.t64.ptr(), FK_CG_INIT, S.st, S.partials, S.stream));
  QCU_TRY(cg_p(op, S.cg_p.ptr(), S.cg_z.ptr(), S.st, S.stream));
  QCU_TRY(read_states(S));
  for (int k = 0; k < nsys; ++k) stats[k] = SolveStats{0, 0, 0, 0};
  int iters = 0;
  for (;;) {
    bool running = false;
    for (int k = 0; k < nsys; ++k) running = running || hs[k].done == 0;
    if (!running || iters >= max_iter) break;
    const int n = std::min(chunk, max_iter - iters);
    for (int j = 0; j < n; ++j) QCU_TRY(cgnr_iteration(S));
    QCU_TRY(read_states(S));
    for (int k = 0; k < nsys; ++k) iters = std::max(iters, hs[k].iter);
  }
  for (int k = 0; k < nsys; ++k) {
    stats[k].iters = hs[k].iter;
    stats[k].converged = hs[k].done == 1 ? 1 : 0;
  }
  return 0;
}

// per-system |b - M x|^2 and |b|^2 of the internal FP64 fields into S.host_scal[2k],
// [2k+1]; te: D_eo x_o where the caller has it, else formed in t
static int residuals_internal(Solver &S, SpinorPtr xe, SpinorPtr xo, SpinorPtr be, SpinorPtr bo, SpinorPtr t,
                              const SpinorPtr *te) {
  const BatchOp &op = *S.op;
  const LaunchCfg cfg = tuned_cfg(op, P64);
  SpinorPtr none{};
  if (!te) QCU_TRY(hop(op, P64, t, xo, 0, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg, S.stream, false));
  QCU_TRY(residual_parity(op, be, xe, te ? *te : t, 0, S.partials, S.dscal, false, S.stream));
  QCU_TRY(hop(op, P64, t, xe, 1, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg, S.stream, false));
  QCU_TRY(residual_parity(op, bo, xo, t, 1, S.partials, S.dscal, true, S.stream));
  QCU_HIP(hipMemcpyAsync(S.host_scal, S.dscal, 2 * S.nsys * sizeof(double), hipMemcpyDeviceToHost, S.stream));
  QCU_HIP(hipStreamSynchronize(S.stream));
  return 0;
}

int true_residuals(Solver &S, const void *const *x_ext, const void *const *b_ext, double *res) {
  QCU_TRY(systems_to_batch(x_ext, *S.op, S.xe.ptr(), S.xo.ptr(), S.stream));
  QCU_TRY(systems_to_batch(b_ext, *S.op, S.be.ptr(), S.bo.ptr(), S.stream));
  QCU_TRY(residuals_internal(S, S.xe.ptr(), S.xo.ptr(), S.be.ptr(), S.bo.ptr(), S.r64.ptr(), nullptr));
  for (int k = 0; k < S.nsys; ++k) {
    const double num = S.host_scal[2 * k], den = S.host_scal[2 * k + 1];
    res[k] = den > 0 ? sqrt(num / den) : sqrt(num);
  }
  return 0;
}

int full_solve(Solver &S, void *const *x_ext, const void *const *b_ext, const QcuSolveParam &prm, QcuSolveInfo *info) {
  const BatchOp &op = *S.op;
  const int nsys = S.nsys;
  auto t0 = std::chrono::steady_clock::now();
  PhaseTrace trace(S.stream);
  QCU_TRY(systems_to_batch(b_ext, op, S.be.ptr(), S.bo.ptr(), S.stream));
  // bhat = Ao^-1 (b_o + kappa D_oe Ae^-1 b_e)
  const LaunchCfg cfg = tuned_cfg(op, P64);
  SpinorPtr none{};
  // (with |b|^2 per system for the stopping rule)
  QCU_TRY(cl_axpy(op, S.t64.ptr(), S.be.ptr(), 0.0, false, none, 1, 0, S.stream, S.dscal, S.partials));
  QCU_TRY(hop(op, P64, S.r64.ptr(), S.t64.ptr(), 1, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg, S.stream,
              false));
  QCU_TRY(cl_axpy(op, S.bh.ptr(), S.bo.ptr(), 0.0, true, S.r64.ptr(), 1, 1, S.stream, S.dscal + nsys, S.partials));
  QCU_HIP(hipMemcpyAsync(S.host_scal, S.dscal, 2 * nsys * sizeof(double), hipMemcpyDeviceToHost, S.stream));
  QCU_HIP(hipStreamSynchronize(S.stream));
  std::vector<double> target2(nsys), res(nsys, INFINITY);
  for (int k = 0; k < nsys; ++k) {
    const double b2 = S.host_scal[k] + S.host_scal[nsys + k];
    // legacy: Re<r,r> < tol on the Schur residual, as the reference
    target2[k] = prm.legacy_stop ? prm.tol : 0.25 * prm.tol * prm.tol * b2;
  }
  trace.mark("b_hat + norms");
  // iterations per graph: a preconditioned solve reaches a reliable update every
  // 2-4; unless the caller set a length, fewer are launched where fewer are expected
  const int chunk = prm.chunk > 0 ? prm.chunk : (prm.precond ? 4 : 8);
  const int max_iter = prm.max_iter > 0 ? prm.max_iter : 10000;
  const double delta = prm.reliable_delta > 0 ? prm.reliable_delta : 0.1;
  Precond *K = (Precond *)prm.precond;
  std::vector<int> active(nsys, 1), fallback(nsys, 0), total_iters(nsys, 0), total_rel(nsys, 0),
      restarts(nsys, 0), converged(nsys, 0);
  std::vector<SolveStats> st(nsys);
  bool warm = false;
  for (int attempt = 0; attempt < 8; ++attempt) {
    int budget = max_iter;
    for (int k = 0; k < nsys; ++k)
      if (active[k]) budget = std::min(budget, max_iter - total_iters[k]);
    if (prm.method == QCU_METHOD_CGNR)
      QCU_TRY(cgnr_solve(S, target2, std::max(budget, 0), chunk, warm, active, st));
    else
      QCU_TRY(schur_solve(S, prm.precision, target2, delta, std::max(budget, 0), chunk, prm.chunk <= 0,
                          prm.use_graph != 0, K, warm, active, st));
    trace.mark("schur solve");
    bool stalled = false;
    for (int k = 0; k < nsys; ++k) {
      if (!active[k]) continue;
      total_iters[k] += st[k].iters;
      total_rel[k] += st[k].reliable;
      restarts[k] += st[k].restarts;
      stalled = stalled || !st[k].converged;
    }
    warm = true;
    if (stalled && K && budget > 0) {
      // a stalled preconditioned solve falls back to the plain method from the current x_o
      K = nullptr;
      for (int k = 0; k < nsys; ++k)
        if (active[k] && !st[k].converged) fallback[k] = 1;
      for (int k = 0; k < nsys; ++k) active[k] = active[k] && !st[k].converged ? 1 : 0;
      continue;
    }
    // x_e = Ae^-1 (b_e + kappa D_eo x_o), then the FP64 true residual of each system
    QCU_TRY(hop(op, P64, S.t64.ptr(), S.xo.ptr(), 0, EPI_PLAIN, none, RED_NONE, none, nullptr, nullptr, cfg, S.stream,
                false));
    QCU_TRY(cl_axpy(op, S.xe.ptr(), S.be.ptr(), 0.0, true, S.t64.ptr(), 1, 0, S.stream));
    const SpinorPtr te = S.t64.ptr();
    QCU_TRY(residuals_internal(S, S.xe.ptr(), S.xo.ptr(), S.be.ptr(), S.bo.ptr(), S.r64.ptr(), &te));
    trace.mark("x_e + true residual");
    bool again = false;
    for (int k = 0; k < nsys; ++k) {
      const double num = S.host_scal[2 * k], den = S.host_scal[2 * k + 1];
      res[k] = den > 0 ? sqrt(num / den) : sqrt(num);
      converged[k] = prm.legacy_stop ? (st[k].converged || converged[k]) : (res[k] <= prm.tol);
      const bool retry = active[k] && !prm.legacy_stop && !converged[k] && st[k].converged &&
                         total_iters[k] < max_iter && std::isfinite(res[k]);
      if (retry) target2[k] *= 0.01;  // tighten the Schur target and continue from x_o
      active[k] = retry ? 1 : 0;
      again = again || retry;
    }
    if (!again) break;
  }
  QCU_TRY(batch_to_systems(S.xe.ptr(), S.xo.ptr(), op, x_ext, S.stream));
  QCU_HIP(hipStreamSynchronize(S.stream));
  const double secs = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
  if (info) {
    for (int k = 0; k < nsys; ++k) {
      info[k].iters = total_iters[k];
      info[k].reliable_updates = total_rel[k];
      info[k].converged = converged[k];
      info[k].fallback = fallback[k];
      info[k].true_res = res[k];
      info[k].seconds = secs;
      info[k].restarts = restarts[k];
    }
  }
  return 0;
}

}  // namespace qcu
