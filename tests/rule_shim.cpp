// The granularity rule (device.hpp) as plain functions, for test_rule.py.
#include "../x-ted_amd/csrc/device.hpp"

using namespace xted;

extern "C" {

struct Rule {
  int lds_per_wave, max_cpl, min_waves, wide_cols, tail;
};
// One table: sides a and b, nesting heights of the row and the column keyroot,
// leaves of the column keyroot, its level's interior cells.
struct Table {
  int a, b, kd_r, kd_c, leaves_c;
  long long cells;
};

static ClassRule rule_of(const Rule& r) {
  return r.tail ? ClassRule{kLdsMaxTable, 1, 1 << 30, kLdsMaxTable, 16, kXLSeqRows}
                : ClassRule{r.lds_per_wave, r.min_waves, r.wide_cols, kLdsMaxTable, r.max_cpl,
                            kXLSeqRows};
}

int rule_class(const Rule* r, const Table* t, int force, long long* need) {
  const ClassRule rule = rule_of(*r);
  int64_t n = 0;
  auto own = [&](int k) { return t->leaves_c < xl_bw(k) ? t->leaves_c : xl_bw(k); };
  int cls = table_class(t->a, t->b, t->kd_r, t->kd_c, t->leaves_c, true, rule,
                        [&] { return (int64_t)t->cells; }, own, &n);
  cls = forced_class(force, cls, t->a, t->b, t->kd_r, t->kd_c, t->leaves_c, rule, own, &n);
  *need = n;
  return cls;
}

// A new context's settings: those of xted_set_tuning, then the tail rule's, the
// level placement's, the size bands', the light LDS and the tiny forms'.
void default_knobs(int* out) {
  const ClassRule r = kDefaultRule;
  const int v[] = {r.lds_per_wave,     r.max_cpl,         r.min_waves,   r.wide_cols, kDefaultTailPairs,
                   kDefaultLevelAlign, kDefaultSizeBands, kLightPerWave, r.tiny};
  for (int i = 0; i < 9; ++i) out[i] = v[i];
}

long long scan_need(int slots, int leaves_c, int kd_c, int w) {
  return scan_lds_need(slots, leaves_c, kd_c, w);
}

}  // extern "C"
