// qcu_tune.h -- the hop kernel's launch shape without tuning, and the tuner's choice.
#pragma once
#include "qcu_internal.h"

namespace qcu {

// The rule for `nvsites` virtual sites: single-wave blocks refill a SIMD as soon as a
// wave ends (24^3x48 FP64 142 against 149 us in blocks of 256); large batches take
// longer blocks, which run as fast there and write fewer block partials.  The low
// precisions fence their directions in pairs (24^3x48 FP32 65 against 73 us
// unfenced), FP64 needs every load in flight (32^3x64 plain 282 against 288 us).
inline LaunchCfg rule_cfg(long long nvsites, int prec) {
  LaunchCfg c;
  c.block = nvsites <= (1 << 20) ? 64 : 256;
  c.group = prec == P64 ? 0 : 2;
  return c;
}

// The fastest of the rule's choice and the 18 shapes of one thread per site, by
// time(cfg, &ms); *best is automatic where that is the rule's.  split: the rule runs
// the kernel with eight waves per 64 sites; otherwise its shape is one of the 18 and
// is timed as the rule's only, so that noise between two timings of one launch does
// not decide what is kept.
template <class Time>
int fastest_shape(const LaunchCfg &rule, bool split, Time time, LaunchCfg *best, double *best_ms) {
  *best = rule;
  QCU_TRY(time(rule, best_ms));
  for (int group = 0; group < 3; ++group)
    for (int block = 64; block <= 256; block *= 2)
      for (int remap = 0; remap < 2; ++remap) {
        if (!split && block == rule.block && remap == rule.remap && group == rule.group) continue;
        LaunchCfg c;
        c.block = block;
        c.remap = remap;
        c.group = group;
        c.automatic = false;
        double ms = 0;
        QCU_TRY(time(c, &ms));
        if (ms < *best_ms) {
          *best_ms = ms;
          *best = c;
        }
      }
  return 0;
}

}  // namespace qcu
