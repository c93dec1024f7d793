// The FFN's dispatch (credit_amd/csrc/ffn_plan.hpp) as the tests ask for it;
// built with g++ by tests/ffn_plan.py.
#include "../../credit_amd/csrc/ffn_plan.hpp"

// out: big, bm, slices, skew, held and its extra LDS of C[M, N] over K.
extern "C" void ffn_plan_query(int64_t M, int64_t N, int64_t K, int kn, int64_t* out) {
  const credit::ffn::GemmPlan p = credit::ffn::gemm_plan(M, N, K, kn != 0);
  out[0] = p.big;
  out[1] = p.bm;
  out[2] = p.slices;
  out[3] = p.skew;
  out[4] = p.held;
  out[5] = p.held ? credit::ffn::held_extra_lds((M / 128) * (N / 128), K / 64) : 0;
}
