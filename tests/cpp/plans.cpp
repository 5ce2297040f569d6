// The prefill kernels' cutting rules (csrc/plans.hpp) as plain C functions, for tests/test_plans.py.
#include "plans.hpp"

extern "C" {
void flash_plan_c(int T, int NQ, int NKV, int pos0, int kv_bf16, int n_cu, int64_t room, int* out, double* time) {
    const q35k::FlashPlan p = q35k::flash_plan(T, NQ, NKV, pos0, kv_bf16 != 0, n_cu, room);
    out[0] = p.piece;
    out[1] = p.pieces;
    out[2] = p.slots;
    *time = p.time;
}
}
