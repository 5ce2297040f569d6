"""Every tile form of the projection GEMM's kernel for few tokens, on each way its X operand can
lie: the rows of a product of M rows have the bits they have among 1100 rows, which the
128 x 128 tiles compute in the same order of sums. SIZES names one ragged and one other size per
tile form (tests/test_plans.py checks that they take it), (4, 4) at four K blocks a round being
the most LDS; 1024 and 1025 rows are the two sides of the dispatch. X split by its producer (the
in-projection and gate/up of a model's prefill) and the SwiGLU output's partial row maxima run
through a model: a GDN and an attention layer of the 0.8B- and 2B-shaped models."""
import numpy as np
import pytest

import pyq35
from helpers import bf16_bits, rel_l2

pytestmark = pytest.mark.gpu
ALL = 1100
# (three bf16 parts, two fp16 parts) -> tile form -> (M, N, K)
SIZES = {
    False: {(1, 1): [(10, 1024, 2048), (4, 1021, 2224)], (1, 2): [(115, 1021, 2048), (86, 1021, 2376)],
            (1, 3): [(141, 1024, 2048), (149, 1024, 2376)], (1, 5): [(34, 4102, 2048), (59, 4102, 2256)],
            (2, 2): [(207, 1022, 2048), (204, 1022, 2264)], (2, 3): [(276, 1021, 2048), (302, 1024, 2248)],
            (2, 4): [(404, 1021, 2048), (510, 1024, 2416)], (2, 5): [(101, 4099, 2048), (265, 4099, 2336)],
            (3, 3): [(360, 1021, 2048), (331, 1024, 3176)], (3, 5): [(643, 1021, 2048), (658, 1024, 3048)],
            (4, 3): [(519, 1021, 2048), (636, 1021, 2384)], (4, 4): [(814, 1021, 2048), (1024, 1024, 2048)]},
    True: {(1, 1): [(4, 1021, 2048), (47, 1024, 2208)], (1, 2): [(71, 1021, 2048), (86, 1021, 2368)],
           (1, 3): [(130, 1021, 2048), (138, 1024, 2496)], (1, 5): [(33, 4100, 2048), (40, 4099, 2240)],
           (2, 2): [(190, 1021, 2048), (187, 1024, 2240)], (2, 3): [(274, 1021, 2048), (320, 1024, 2304)],
           (2, 4): [(386, 1021, 2048), (438, 1024, 2432)], (2, 5): [(104, 4099, 2048), (108, 4368, 2208)],
           (3, 3): [(322, 1021, 2048), (334, 1024, 2336)], (3, 5): [(667, 1021, 2048), (670, 1021, 3168)],
           (4, 3): [(518, 1021, 2048), (523, 1024, 2432)], (4, 4): [(777, 1021, 2048), (847, 1021, 2336)]},
}


@pytest.mark.parametrize("f16,tile", [(f, t) for f in SIZES for t in SIZES[f]])
def test_tile(f16, tile):
    hip, lib = pyq35.Hip(), pyq35.lib
    for M, N, K in SIZES[f16][tile]:
        rng = np.random.default_rng(N + K)
        X = rng.standard_normal((ALL, K)).astype(np.float32)
        R = rng.standard_normal((ALL, N)).astype(np.float32)
        ws = lib.q35_gemm_f16x2_workspace_bytes(ALL, N, K) if f16 else 4
        bufs = [hip.upload(X), hip.upload(bf16_bits(0.02 * rng.standard_normal((N, K)).astype(np.float32))), hip.upload(R),
                hip.malloc(ws)]
        dX, dW, dY, dws = bufs

        def product(M):
            hip.copy_in(dY, R)  # the residual, in place
            if f16:
                pyq35.check(lib.q35_gemm_f16x2(dX, K, dW, M, N, K, dY, N, dY, N, dws, ws, None))
            else:
                pyq35.check(lib.q35_gemm_bf16(dX, K, dW, M, N, K, dY, N, dY, N, None))
            hip.sync()
            return hip.download(dY, (ALL, N))

        try:
            many, few = product(ALL), product(M)
            np.testing.assert_array_equal(few[:M], many[:M], err_msg=f"{M} x {N} x {K}")
            np.testing.assert_array_equal(few[M:], R[M:], err_msg=f"{M} x {N} x {K}: wrote past its rows")
            if M == 1024:
                np.testing.assert_array_equal(product(1025)[:1025], many[:1025])
        finally:
            for p in bufs:
                hip.free(p)


@pytest.mark.parametrize("name", ["0.8b", "2b"])
def test_model_layers(tmp_path, name):
    """Hidden states after each layer: the same bits whatever the number of tokens (the GDN layer's
    kernel for up to 36 tokens sums in another order: there within 1e-6)."""
    d = pyq35.dims_for(name)
    d.n_layers_total, d.attn_interval, d.vocab_size = 2, 2, 1024
    pyq35.synth_write_model(str(tmp_path), d, seed=3, std=0.02)
    ids = pyq35.synth_token_ids(7, d.vocab_size, ALL)
    m = pyq35.Model(str(tmp_path), ALL + 8)

    def layers(n):
        m.reset()
        return m.extend(ids[:n], want_logits=False, want_trace=True)[1]

    many = layers(ALL)
    for n in (1, 9, 16, 17, 33, 36):
        few = layers(n)
        assert max(rel_l2(few[t, l], many[t, l]) for t in range(n) for l in range(2)) < 1e-6, n
    for n in (37, 48, 49, 64, 97, 130, 145, 192, 209, 256, 300, 400, 500, 640, 769, 1000, 1024, 1025):
        np.testing.assert_array_equal(layers(n), many[:n], err_msg=f"{n} tokens")
    m.close()
