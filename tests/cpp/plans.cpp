// The prefill kernels' cutting rules (csrc/plans.hpp) as plain C functions, for tests/test_plans.py.
#include "plans.hpp"

extern "C" {
void flash_plan_c(int T, int NQ, int NKV, int pos0, int kv_bf16, int n_cu, int64_t room, int* out, double* time,
                  double* rounds) {
    const q35k::FlashPlan p = q35k::flash_plan(T, NQ, NKV, pos0, kv_bf16 != 0, n_cu, room);
    out[0] = p.piece;
    out[1] = p.pieces;
    out[2] = p.slots;
    *time = p.time;
    *rounds = p.rounds;
}
// out: image, piece, pieces, slots
void attn_room_c(int T, int NQ, int NKV, int pos0, int kv_bf16, int n_cu, int64_t floats, int* out, double* rounds) {
    const q35k::AttnRoom r = q35k::attn_prefill_room(T, NQ, NKV, pos0, kv_bf16 != 0, n_cu, floats);
    out[0] = r.image;
    out[1] = r.plan.piece;
    out[2] = r.plan.pieces;
    out[3] = r.plan.slots;
    *rounds = r.plan.rounds;
}
int share_slots_c(int T, int NQ, int NKV, int kv_bf16, int64_t max_ctx) {
    return q35k::attn_prefill_share_slots(T, NQ, NKV, kv_bf16 != 0, max_ctx);
}
// out: mr, nr, rt, ct, unit; 0 where the 128 x 128 tiles are the choice
int gemm_small_plan_c(int M, int N, int K, int swiglu, int path, int n_cu, int* out) {
    q35k::SmallPlan p{};
    if (!q35k::gemm_small_plan(M, N, K, swiglu != 0, path, n_cu, &p)) return 0;
    out[0] = p.mr;
    out[1] = p.nr;
    out[2] = p.rt;
    out[3] = p.ct;
    out[4] = p.unit;
    return 1;
}
int gemm_small_max_parts_c(int N) { return q35k::gemm_small_max_parts(N); }
}
