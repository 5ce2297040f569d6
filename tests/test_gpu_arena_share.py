"""The prompt arena's room for the attention's partial outputs (68 MB): only where a context is
long enough for its keys to be cut, and made when the context grows to that; a context that
grows keeps its prompts working, with blocks as large as before, and their results."""
import numpy as np
import pytest

import pyq35
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu
SLOT = 16 * 258 * 4


def arena(m):
    return m.budget()["prompt_arena_bytes"]


@pytest.mark.parametrize("kv", [4, 2])
def test_no_room_where_nothing_is_cut(model_dirs, kv):
    size = {}
    for ctx in (1024, 2048, 2049, 4096):
        m = pyq35.Model(model_dirs["tiny"], ctx, kv_bytes_per_elem=kv, prefill_block=64)
        size[ctx] = arena(m)
        m.close()
    # uncut: at most the tile image of an fp32 cache (3 KB a position of the one kv head)
    assert 0 <= size[2048] - size[1024] <= (1024 * 3072 + 256 if kv == 4 else 0) and size[2048] < size[2049]
    assert size[2048] < 32 << 20
    # 64 tokens of 2 heads are one block of 128 rows or two of 64: 8 slots a piece of 128 or fewer
    assert size[4096] - size[2048] <= 8 * 128 * SLOT


@pytest.mark.parametrize("planned", [True, False])
def test_room_after_the_context_grows(model_dirs, planned):
    ids = pyq35.synth_token_ids(5, 1024, 40)
    m = pyq35.Model(model_dirs["tiny"], 1000, prefill_block=64 if planned else 0)
    m.set_prefill_block(64)
    m.prefill(ids, want_logits=False)
    before = arena(m)
    m.reserve_context(4096)
    m.fill_synthetic(4000, seed=9)
    got = m.extend(ids)[0]
    m.set_prefill_block(16)   # smaller blocks: the same arena
    m.set_position(0)
    m.extend(ids, want_logits=False)
    grown = arena(m)
    m.close()
    fresh = pyq35.Model(model_dirs["tiny"], 4096, prefill_block=64)
    fresh.fill_synthetic(4000, seed=9)
    ref = fresh.extend(ids)[0]
    assert before < grown == arena(fresh)
    fresh.close()
    np.testing.assert_array_equal(got, ref)
    assert rel_l2(got, ref) < REL_L2


@pytest.mark.parametrize("kv", [4, 2])
@pytest.mark.parametrize("T", [700, 1500])
def test_long_turn_on_a_long_context(tmp_path, T, kv):
    """16 / 2 heads at 8000 positions, a turn in one block whose best cut (more than 5000 slots) is
    larger than the 4096 that the arena sets aside, against decoding it token by token."""
    d = pyq35.dims_for("tiny")
    d.n_layers_total, d.attn_interval, d.attn_q_heads, d.attn_kv_heads = 2, 2, 16, 2
    pyq35.synth_write_model(str(tmp_path), d, seed=3, std=0.02)
    ids = pyq35.synth_token_ids(11, d.vocab_size, T)
    logits = []
    for block in (T, 0):
        m = pyq35.Model(str(tmp_path), 8000 + T, kv_bytes_per_elem=kv, prefill_block=block)
        m.fill_synthetic(8000, seed=9)
        logits.append(m.extend(ids)[0] if block else np.stack([m.step(int(i))[0] for i in ids]))
        m.close()
    # a bf16 row may round the other way: the bar of the bf16-cache model tests
    bar = REL_L2 if kv == 4 else 2e-4
    assert max(rel_l2(a, b) for a, b in zip(*logits)) < bar
