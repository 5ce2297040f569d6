"""Attention decode of GQA groups of 4 on the matrix cores, fp32 and bf16 caches, against the
oracle at the bars of the other decode tests: splits shorter than a tile of 16 positions, one
past it, ragged over the four waves, a single split, rotary widths that do and do not take this
kernel, and a bf16 cache off its 16-byte alignment (which takes the vector kernel)."""
import ctypes as C

import numpy as np
import pytest

import pyq35
import test_gpu_kv_bf16 as kv16
import test_gpu_mixers as mix
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    return pyq35.Hip()


@pytest.mark.parametrize("pos,n_splits", [(0, 1), (15, 1), (16, 1), (65, 1), (130, 2), (9, 4), (1000, 7), (4099, 64)])
def test_splits(hip, pos, n_splits):
    for nq, nkv in ((8, 2), (4, 1)):
        out, ref, krow, kref, vrow, vref = mix.run_attn(hip, nq, nkv, pos, pos + 2, n_splits, seed=pos + nq)
        assert rel_l2(out, ref) < REL_L2
        np.testing.assert_allclose(krow, kref, rtol=2e-6, atol=2e-6)
        np.testing.assert_array_equal(vrow, vref)
        kv16.run_attn_decode_bf16(hip, nq, nkv, pos, pos + 2, n_splits, seed=pos + nq)


@pytest.mark.parametrize("rot", [0, 18, 32, 256])
def test_rotary_widths(hip, rot):
    out, ref, *_ = mix.run_attn(hip, 8, 2, 200, 201, 3, seed=rot, rot=rot)
    assert rel_l2(out, ref) < REL_L2


def test_bf16_layers(hip):
    kv16.run_attn_decode_bf16(hip, 8, 2, 777, 800, 0, seed=3, layers=3)


def test_bf16_cache_alignment(hip):
    """The same cache 16-byte aligned and 8 bytes off: equal within the bar."""
    rng = np.random.default_rng(5)
    pos, maxc, n = 300, 304, 2 * 304 * 256
    bits = [kv16.cache_bits(rng, (2, maxc, 256), pos).ravel() for _ in range(2)]
    up = lambda a: hip.upload(a.astype(np.float32))  # noqa: E731
    qg, kn, vn, w = up(rng.standard_normal(8 * 512)), up(rng.standard_normal(512)), up(rng.standard_normal(512)), up(np.zeros(256))
    outs, bufs = [], [qg, kn, vn, w]
    for off in (0, 4):
        k, v = (hip.upload(np.concatenate([np.zeros(off, np.uint16), b, np.zeros(8, np.uint16)])) for b in bits)
        a = pyq35.AttnDecodeArgs(q_heads=8, kv_heads=2, head_dim=256, rotary_dim=64, pos=pos, max_context=maxc, kv_dtype=1,
                                 rope_theta=1e7, eps=1e-6, qg=qg, k_new=kn, v_new=vn, q_norm=w, k_norm=w,
                                 k_cache=k + 2 * off, v_cache=v + 2 * off)
        a.workspace_bytes = pyq35.lib.q35_attn_decode_workspace_bytes(C.byref(a))
        a.workspace, a.out = hip.malloc(a.workspace_bytes), hip.malloc(8 * 256 * 4)
        pyq35.check(pyq35.lib.q35_attn_decode(C.byref(a), None))
        hip.sync()
        outs.append(hip.download(a.out, 8 * 256))
        bufs += [k, v, a.workspace, a.out]
    for p in bufs:
        hip.free(p)
    assert n == bits[0].size and rel_l2(outs[0], outs[1]) < REL_L2
