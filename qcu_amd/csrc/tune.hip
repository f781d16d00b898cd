// tune.hip -- launch-shape autotuner and hop timing.
//
// For each (device, batch shape, precision) the tuner times the hop kernel
// with HIP events over a grid of block sizes, XCD-aware block orders and
// instruction-scheduling groupings, and keeps the fastest.  Results persist in
// a plain text cache file ("key block remap group" per line) so that later
// processes skip the search.
#include <atomic>
#include <cstdio>
#include <map>
#include <mutex>
#include <string>

#include "../../include/qcu.h"
#include "qcu_lattice.h"
#include "qcu_solver.h"
#include "qcu_tune.h"

namespace qcu {

namespace {
std::mutex g_tune_mu;
std::map<std::string, LaunchCfg> g_tuned;
std::atomic<unsigned long long> g_tune_gen{1};
}  // namespace

// changes whenever a tuned launch shape is set, so that captured solver
// graphs (which hold the launch shapes of their capture) are re-captured
unsigned long long tune_generation() { return g_tune_gen.load(); }

static void set_tuned(const std::string &key, LaunchCfg c) {
  c.automatic = false;
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned[key] = c;
  }
  ++g_tune_gen;
}

// back to the shape that the rule picks
static void set_automatic(const std::string &key) {
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    g_tuned.erase(key);
  }
  ++g_tune_gen;
}

static int valid_cfg(int block, int remap, int group) {
  QCU_CHECK((block == 64 || block == 128 || block == 256) && (remap == 0 || remap == 1) && group >= 0 && group <= 2,
            QCU_ERR_ARG, "launch shape: block 64, 128 or 256; remap 0 or 1; group 0, 1 or 2");
  return 0;
}

// the part of a batch's table key that is the same for every precision, formed
// once when the batch is built (asking the driver for the device costs more
// than a small hop)
std::string tune_base(const BatchOp &op) {
  static std::mutex mu;
  static std::map<int, std::string> names;  // device names, asked for once
  std::string k;
  {
    std::lock_guard<std::mutex> lk(mu);
    const int dev = current_device();
    auto it = names.find(dev);
    if (it == names.end()) {
      hipDeviceProp_t prop;
      if (dev >= 0 && hipGetDeviceProperties(&prop, dev) == hipSuccess) k = prop.gcnArchName;
      names[dev] = k;
    } else {
      k = it->second;
    }
  }
  char buf[96];
  for (const SegDesc &d : op.segs) {
    snprintf(buf, sizeof(buf), ":%dx%dx%dx%dr%d", 2 * d.g.lxh, d.g.ly, d.g.lz, d.g.lt, d.nrhs);
    k += buf;
  }
  return k;
}

std::string tune_key(const BatchOp &op, int prec) {
  char buf[32];
  snprintf(buf, sizeof(buf), ":p%d:c%d", prec, op.has_clover ? 1 : 0);
  return op.tune_base + buf;
}

static LaunchCfg find_cfg(const BatchOp &op, int prec) {
  {
    std::lock_guard<std::mutex> lk(g_tune_mu);
    auto it = g_tuned.find(tune_key(op, prec));
    if (it != g_tuned.end()) return it->second;
  }
  return rule_cfg(op.nvsites, prec);
}

LaunchCfg tuned_cfg(const BatchOp &op, int prec) {
  if (prec < P64 || prec > P16) return LaunchCfg();  // no such shape: hop() refuses the precision
  const unsigned long long gen = tune_generation();
  LaunchCfg c;
  if (!op.shapes.get(prec, gen, &c)) {
    c = find_cfg(op, prec);
    op.shapes.put(prec, gen, c);
  }
  return c;
}

// average milliseconds per launch of the hop kernel on resident fields
int bench_hop(const BatchOp &op, hipStream_t s, int prec, int clover, int xpay, int iters, const LaunchCfg &cfg,
              double *ms) {
  QCU_CHECK(prec >= 0 && prec <= 2 && iters > 0, QCU_ERR_ARG, "bad precision or iteration count");
  for (const Lattice *l : op.lats)
    QCU_CHECK((l->prec_mask >> prec) & 1, QCU_ERR_STATE, "links of the requested precision are not resident");
  const int n = (int)op.nvsites;
  Spinor a, b, c, g64;
  QCU_TRY(a.create(prec, n));
  QCU_TRY(b.create(prec, n));
  QCU_TRY(c.create(prec, n));
  QCU_TRY(g64.create(P64, n));
  QCU_TRY(gen_gauss(g64.data.p, (long)n * 12, 77, s));
  QCU_TRY(spinor_convert(op, a.ptr(), prec, g64.ptr(), s));
  QCU_TRY(spinor_convert(op, c.ptr(), prec, g64.ptr(), s));
  SpinorPtr none{};
  auto launch = [&](int k) {
    return hop(op, prec, (k & 1) ? a.ptr() : b.ptr(), (k & 1) ? b.ptr() : a.ptr(), k & 1, xpay ? EPI_XPAY : EPI_PLAIN,
               c.ptr(), RED_NONE, none, nullptr, nullptr, cfg, s, clover != 0);
  };
  for (int k = 0; k < 3; ++k) QCU_TRY(launch(k));
  hipEvent_t e0, e1;
  QCU_HIP(hipEventCreate(&e0));
  QCU_HIP(hipEventCreate(&e1));
  QCU_HIP(hipEventRecord(e0, s));
  for (int k = 0; k < iters; ++k) QCU_TRY(launch(k));
  QCU_HIP(hipEventRecord(e1, s));
  QCU_HIP(hipEventSynchronize(e1));
  float t = 0;
  QCU_HIP(hipEventElapsedTime(&t, e0, e1));
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  *ms = (double)t / iters;
  return 0;
}

static int tune_op(const BatchOp &op, hipStream_t s, int prec, double *best_ms, LaunchCfg *out) {
  const int clover = op.has_clover ? 1 : 0;
  const LaunchCfg rule = rule_cfg(op.nvsites, prec);
  LaunchCfg best;
  double bms = 0;
  QCU_TRY(fastest_shape(
      rule, hop_is_split(op, rule),
      [&](const LaunchCfg &c, double *ms) { return bench_hop(op, s, prec, clover, 1, 20, c, ms); }, &best, &bms));
  if (best.automatic)
    set_automatic(tune_key(op, prec));
  else
    set_tuned(tune_key(op, prec), best);
  if (best_ms) *best_ms = bms;
  if (out) *out = best;
  return 0;
}

}  // namespace qcu

using namespace qcu;

struct QcuBatch_s;
namespace qcu {
const BatchOp &batch_op(const QcuBatch_s *b);
hipStream_t batch_stream(const QcuBatch_s *b);
}  // namespace qcu

extern "C" {

int qcuTune(QcuLatticeHandle h, int prec, double *best_ms) {
  clear_error();
  QCU_CHECK(h, QCU_ERR_ARG, "null handle");
  QCU_CHECK(prec >= 0 && prec <= 2, QCU_ERR_ARG, "bad precision");
  QCU_CHECK(h->lat.gauge_loaded, QCU_ERR_STATE, "gauge field not loaded");
  return tune_op(h->lat.self, h->lat.stream, prec, best_ms, nullptr);
}

int qcuTuneSet(QcuLatticeHandle h, int prec, int block, int remap, int group) {
  clear_error();
  QCU_CHECK(h, QCU_ERR_ARG, "null handle");
  QCU_CHECK(h->lat.gauge_loaded, QCU_ERR_STATE, "gauge field not loaded");
  QCU_CHECK(prec >= 0 && prec <= 2, QCU_ERR_ARG, "bad precision");
  QCU_TRY(valid_cfg(block, remap, group));
  LaunchCfg c;
  c.block = block;
  c.remap = remap;
  c.group = group;
  set_tuned(tune_key(h->lat.self, prec), c);
  return 0;
}

int qcuBatchTuneSet(QcuBatchHandle h, int prec, int block, int remap, int group) {
  clear_error();
  QCU_CHECK(h, QCU_ERR_ARG, "null handle");
  QCU_CHECK(prec >= 0 && prec <= 2, QCU_ERR_ARG, "bad precision");
  QCU_TRY(valid_cfg(block, remap, group));
  LaunchCfg c;
  c.block = block;
  c.remap = remap;
  c.group = group;
  set_tuned(tune_key(batch_op(h), prec), c);
  return 0;
}

int qcuTuneGet(QcuLatticeHandle h, int prec, int *block, int *remap, int *group) {
  clear_error();
  QCU_CHECK(h && block && remap && group, QCU_ERR_ARG, "null argument");
  QCU_CHECK(prec >= 0 && prec <= 2, QCU_ERR_ARG, "bad precision");
  LaunchCfg c = tuned_cfg(h->lat.self, prec);
  *block = c.block;
  *remap = c.remap;
  *group = c.group;
  return 0;
}

int qcuBatchTune(QcuBatchHandle h, int prec, double *best_ms) {
  clear_error();
  QCU_CHECK(h, QCU_ERR_ARG, "null handle");
  QCU_CHECK(prec >= 0 && prec <= 2, QCU_ERR_ARG, "bad precision");
  return tune_op(batch_op(h), batch_stream(h), prec, best_ms, nullptr);
}

int qcuTuneSave(const char *path) {
  QCU_CHECK(path, QCU_ERR_ARG, "null path");
  FILE *f = fopen(path, "w");
  QCU_CHECK(f, QCU_ERR_ARG, std::string("cannot write ") + path);
  std::lock_guard<std::mutex> lk(g_tune_mu);
  for (auto &kv : g_tuned)
    fprintf(f, "%s %d %d %d\n", kv.first.c_str(), kv.second.block, kv.second.remap, kv.second.group);
  fclose(f);
  return 0;
}

int qcuTuneLoad(const char *path) {
  QCU_CHECK(path, QCU_ERR_ARG, "null path");
  FILE *f = fopen(path, "r");
  if (!f) return 0;  // no cache yet
  char key[512];
  int b, r, grp;
  std::lock_guard<std::mutex> lk(g_tune_mu);
  while (fscanf(f, "%511s %d %d %d", key, &b, &r, &grp) == 4) {
    if (b >= 64 && b <= 256 && b % 64 == 0 && (r == 0 || r == 1) && grp >= 0 && grp <= 2) {
      LaunchCfg c;
      c.block = b;
      c.remap = r;
      c.group = grp;
      c.automatic = false;
      g_tuned[key] = c;
    }
  }
  fclose(f);
  ++g_tune_gen;
  return 0;
}

}  // extern "C"
