// The host-side rules that choose a kernel (plan.hpp has no HIP types in it) behind plain C functions,
// for tests/test_plan_rules.py, which compiles this file with g++ and loads it.
#include "../../torch-xpu-ops_amd/csrc/kernels/plan.hpp"

using namespace rownorm;

extern "C" {

int rule_norm_bwd_reads_elements(int esize, int wsize, int G, int V, int rms, int64_t M, int64_t N) {
  return norm_bwd_reads_elements(esize, wsize, G, V, rms != 0, M, N) ? 1 : 0;
}

}  // extern "C"
