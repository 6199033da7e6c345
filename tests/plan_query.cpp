// The batched GEMMs' launch plans for the tests (tests/_plan.py): kai_batched_plan.h by g++.
#include "../kaillm_amd/csrc/kai_batched_plan.h"

// out: the fields of _plan.Plan
extern "C" void plan_mmqh(int type, int64_t n, int64_t k, int64_t m, int64_t *out) {
    const kai::MmqhPlan p = kai::mmqh_plan(type, n, k, m);
    const kai::MmqhConfig c = kai::mmqh_config(p.id, type);
    const kai::MmqhTail &t = p.tail;
    const int64_t v[] = {p.id, c.bn, c.bm, p.tiles_n, p.tiles_m, p.splits, p.split_stages, t.main, p.has_tail() ? t.splits : 0,
                         t.stages, t.r0, t.c0, t.rows, t.cols, p.rest,
                         static_cast<int64_t>(kai::mmqh_sums_bytes(type, n, k, m))};
    std::copy(std::begin(v), std::end(v), out);
}
extern "C" int plan_mmq6(int64_t n, int64_t k, int64_t m) { return kai::mmq6_plan(n, k, m); }
