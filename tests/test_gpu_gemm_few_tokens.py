"""The projection GEMM's kernel for few tokens: every row of a product of M rows has the bits
it has among 1100 rows (which the 128 x 128 tiles compute, in the same order of sums), and is
within 1e-6 of float64 as the other GEMM tests ask (fp32 sums of K products in blocks of 512).
Sizes at the edges of its cut: one row, a row block and one more, ragged and single column
units, N not a multiple of 4, K below a step, ragged past a 512-deep block, several rounds."""
import numpy as np
import pytest

import pyq35
from helpers import bf16_bits, bf16_to_f32, rel_l2

pytestmark = pytest.mark.gpu
ALL = 1100


@pytest.mark.parametrize("N,K,resid", [(8224, 2048, False), (2048, 6144, True), (1024, 3584, True), (7168, 1024, False),
                                       (4102, 520, True), (130, 1000, False), (4, 8, False), (17, 40, True)])
@pytest.mark.parametrize("f16", [False, True])
def test_rows_do_not_depend_on_their_number(N, K, resid, f16):
    if f16 and K % 32:
        pytest.skip("the fp16 path needs K % 32 == 0")
    hip, lib = pyq35.Hip(), pyq35.lib
    rng = np.random.default_rng(N + K)
    X = rng.standard_normal((ALL, K)).astype(np.float32)
    W = bf16_bits(0.02 * rng.standard_normal((N, K)).astype(np.float32))
    R = rng.standard_normal((ALL, N)).astype(np.float32)
    ws = lib.q35_gemm_f16x2_workspace_bytes(ALL, N, K) if f16 else 4
    dX, dW, dY, dws = hip.upload(X), hip.upload(W), hip.malloc(ALL * N * 4), hip.malloc(ws)

    def product(M):
        hip.copy_in(dY, R)
        r = dY if resid else None
        if f16:
            pyq35.check(lib.q35_gemm_f16x2(dX, K, dW, M, N, K, r, N, dY, N, dws, ws, None))
        else:
            pyq35.check(lib.q35_gemm_bf16(dX, K, dW, M, N, K, r, N, dY, N, None))
        hip.sync()
        return hip.download(dY, (ALL, N))

    try:
        many = product(ALL)
        ref = X.astype(np.float64) @ bf16_to_f32(W).astype(np.float64).T + (R if resid else 0.0)
        assert rel_l2(many, ref) < 1e-6
        for M in (1, 15, 16, 17, 48, 77, 130, 300, 513):
            few = product(M)
            np.testing.assert_array_equal(few[:M], many[:M], err_msg=f"M={M}")
            np.testing.assert_array_equal(few[M:], R[M:], err_msg=f"M={M}: wrote past its rows")
    finally:
        for p in (dX, dW, dY, dws):
            hip.free(p)
