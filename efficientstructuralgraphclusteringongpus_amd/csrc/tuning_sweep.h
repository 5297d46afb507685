// Coordinate descent over the planner knobs of one graph (sgc_dgraph_autotune),
// apart from the timing, which the caller does.
#pragma once

#include <stdint.h>

#include <initializer_list>

namespace sgc {

// Candidates are timed where their knob acts.  On a graph with filter stages a
// plain pass reads small_max_degree and hash_tables only, so the unit and tiny
// knobs, which act in passes that count every edge (with the core-check
// pruning, or when the filters' copies are not there), are timed in such
// passes; timed in plain ones, chance would pick them.  small_max_degree acts
// in both and must not slow either.
//
// measure(t, filters, &ms): the similarity time of a pass with the knobs t, a
// plain one or (filters false) one without filter stages; an error code or 0.
// filtered: whether plain passes have them.  *best starts as the defaults;
// *ms and *ms_default are times of plain passes.
template <class Tuning, class Measure>
int sweep_tuning(bool filtered, Measure measure, Tuning* best, double* ms, double* ms_default) {
  Tuning& cur = *best;
  double plain = 0, counted = 0;
  int rc = measure(cur, true, &plain);
  counted = plain;
  *ms_default = plain;
  auto split = [&]() { return filtered && cur.hash_tables; };
  if (!rc && split()) rc = measure(cur, false, &counted);
  // both: the knob acts with filters, too
  auto sweep = [&](auto knob, bool both, auto candidates) {
    for (const auto v : candidates) {
      if (rc || v == cur.*knob) continue;
      Tuning t = cur;
      t.*knob = v;
      double p = plain, c = counted;
      if (!split() || both) {
        rc = measure(t, true, &p);
        if (rc || !(p < plain)) continue;
        if (!split()) c = p;
      }
      if (split()) {
        rc = measure(t, false, &c);
        if (rc || !(both ? c <= counted : c < counted)) continue;
      }
      cur = t;
      plain = p;
      counted = c;
    }
  };
  sweep(&Tuning::large_unit_work, false, std::initializer_list<double>{2097152.0, 8388608.0, 33554432.0});
  sweep(&Tuning::small_max_degree, true, std::initializer_list<uint32_t>{128, 256, 512, 1024});
  sweep(&Tuning::small_unit_work, false, std::initializer_list<double>{65536.0, 262144.0, 1048576.0});
  if (!rc) {
    Tuning t = cur;
    t.hash_tables = 1 - cur.hash_tables;
    double p;
    rc = measure(t, true, &p);
    if (!rc && p < plain) cur = t, plain = counted = p;
  }
  sweep(&Tuning::tiny_work, false, std::initializer_list<uint32_t>{0, 1024, 2048, 4096});
  *ms = plain;
  return rc;
}

}  // namespace sgc
