"""Attention prefill of few tokens on a long context, where the kernel splits a block's keys into
pieces and merges them: against the oracle (the bar of the other attention tests), without
room for the partial outputs, and through the model against decoding the same tokens one by
one. Sizes: one token, a block of 128 (64 with a bf16 cache) rows and one more, tokens that
straddle a tile, pieces some rows have no key in, groups that do not divide the block."""
import numpy as np
import pytest

import pyq35
import test_gpu_kv_bf16 as kv16
import test_gpu_prefill as pf
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu

SHAPES = [(2, 1, 1, 2047), (2, 1, 1, 2048), (16, 2, 17, 2200), (8, 2, 32, 2080), (8, 2, 33, 4000), (6, 2, 50, 3001),
          (2, 2, 300, 2500), (16, 1, 9, 6100)]


@pytest.fixture(scope="module")
def hip():
    return pyq35.Hip()


@pytest.mark.parametrize("nq,nkv,T,pos0", SHAPES)
def test_split_keys_vs_oracle(hip, nq, nkv, T, pos0):
    out, ref, *_ = pf.run_attn_prefill(hip, nq, nkv, T, pos0, seed=T + pos0)
    whole, *_ = pf.run_attn_prefill(hip, nq, nkv, T, pos0, seed=T + pos0, ws_min=True)
    for t in range(T):
        assert rel_l2(out[t], ref[t]) < REL_L2 and rel_l2(whole[t], ref[t]) < REL_L2, f"token {t}"


@pytest.mark.parametrize("nq,nkv,T,pos0", SHAPES)
def test_split_keys_vs_oracle_bf16(hip, nq, nkv, T, pos0):
    kv16.test_attn_prefill_bf16(hip, nq, nkv, T, pos0)


@pytest.mark.parametrize("name,kv", [("tiny_gqa", 4), ("tiny", 2)])
def test_model_extend_on_a_long_context(tmp_path, name, kv):
    d = pyq35.dims_for(name)
    pyq35.synth_write_model(str(tmp_path), d, seed=3, std=0.02)
    ids = pyq35.synth_token_ids(5, d.vocab_size, 21)
    logits = []
    for block in (True, False):
        m = pyq35.Model(str(tmp_path), 3100, kv_bytes_per_elem=kv)
        m.fill_synthetic(3000, seed=9)
        logits.append(m.extend(ids)[0] if block else np.stack([m.step(int(i))[0] for i in ids]))
        m.close()
    # a bf16 row may round the other way: the bar of the bf16-cache model tests
    bar = REL_L2 if kv == 4 else 2e-4
    for t in range(len(ids)):
        assert rel_l2(logits[0][t], logits[1][t]) < bar, f"token {t}"
