// The launch choices of 15642_moe_amd/csrc/plan.h as C functions for tests/test_plan.py.
#include "plan.h"

extern "C" {

int plan_router_k_parts(int T) { return moe::router_k_parts(T); }
int plan_router_waves(int T, int cus) { return moe::router_waves(T, cus); }

}
