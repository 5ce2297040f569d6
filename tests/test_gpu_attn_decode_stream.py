"""Attention decode of GQA groups of 4 over fp32 caches too long for the Infinity Cache, many
heads x layers in one launch (the vector kernel), against the same layers one launch each (the
matrix cores, compared with the oracle elsewhere): both sides of the line in heads and positions."""
import ctypes as C

import numpy as np
import pytest

import pyq35
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu
HD = 256


@pytest.mark.parametrize("nkv,layers,pos", [(4, 5, 6499), (4, 5, 6498), (10, 2, 6600), (19, 1, 7000)])
def test_layers_together_and_one_by_one(nkv, layers, pos):
    hip, rng, nq, maxc = pyq35.Hip(), np.random.default_rng(pos + nkv), 4 * nkv, pos + 2
    f = lambda *n: rng.standard_normal(n, dtype=np.float32)  # noqa: E731
    n = layers * nkv * maxc * HD
    one = f(2, n // layers)  # one layer's keys and values; the others' are shifted by a few rows
    k, v = (np.concatenate([np.roll(x, 3 * HD * i) for i in range(layers)]) for x in one)
    up = {x: hip.upload(a) for x, a in dict(k=k, v=v, qg=f(layers, nq, 2 * HD), kn=f(layers, nkv, HD), vn=f(layers, nkv, HD),
                                            w=0.1 * f(layers, HD)).items()}
    out = hip.malloc(4 * layers * nq * HD)

    def run(first, count):
        at = lambda x, per: up[x] + 4 * first * per  # noqa: E731
        a = pyq35.AttnDecodeArgs(q_heads=nq, kv_heads=nkv, head_dim=HD, rotary_dim=64, pos=pos, max_context=maxc, n_layers=count,
                                 rope_theta=1e7, eps=1e-6, qg=at("qg", nq * 2 * HD), k_new=at("kn", nkv * HD),
                                 v_new=at("vn", nkv * HD), q_norm=at("w", HD), k_norm=at("w", HD),
                                 k_cache=at("k", nkv * maxc * HD), v_cache=at("v", nkv * maxc * HD), out=out + 4 * first * nq * HD)
        a.workspace_bytes = pyq35.lib.q35_attn_decode_workspace_bytes(C.byref(a))
        a.workspace = hip.malloc(a.workspace_bytes)
        pyq35.check(pyq35.lib.q35_attn_decode(C.byref(a), None))
        hip.sync()
        hip.free(a.workspace)
        return hip.download(out, (layers, nq, HD)), hip.download(up["k"], (layers, nkv, maxc, HD))[:, :, pos]

    together, row = run(0, layers)
    for i in range(layers):
        single, row1 = run(i, 1)
        assert max(rel_l2(together[i, h], single[i, h]) for h in range(nq)) < REL_L2
        np.testing.assert_allclose(row[i], row1[i], rtol=2e-6, atol=2e-6)
    for p in list(up.values()) + [out]:
        hip.free(p)
