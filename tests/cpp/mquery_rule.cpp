// mquery_rule.cpp -- the many-query decode's rule and plan (mquery_rule.hpp) for
// the tests.
#include "../../adaptq_amd/csrc/mquery_rule.hpp"

extern "C" int mq_takes(int n_heads, int nq, int max_n, int padded) {
  return aq::mq_pays(n_heads, nq, max_n, padded);
}

// splits, chunk, qgroups, qg, qblocks
extern "C" void mq_plan_of(int n_heads, int nq, int max_n, int *out) {
  const aq::MqPlan p = aq::mq_plan(n_heads, nq, max_n);
  out[0] = p.splits;
  out[1] = p.chunk;
  out[2] = p.qgroups;
  out[3] = p.qg;
  out[4] = p.qblocks;
}
