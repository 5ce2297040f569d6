"""GDN prefill of few tokens (one launch, token by token) against the oracle's sequential
recurrence at the bars of the other GDN prefill tests: one token, less than a conv run and one
more, positions that move the ring's slots, continuing, v-heads = 2 k-heads, the raw readout, and
a state off its 16-byte alignment (chunked kernels, the same result within the bar); 47, 48 and 49
tokens run the chunked kernels (the 36-token limit of the one launch: test_gpu_gdn_edges.py)."""
import ctypes as C

import numpy as np
import pytest

import oracle_py as op
import pyq35
from helpers import REL_L2, rel_l2, ring_from_window, window_from_ring

pytestmark = pytest.mark.gpu
D = 128


def run(hip, kh, vh, T, pos0, seed, gated=True, misalign=0):
    rng = np.random.default_rng(seed)
    d = pyq35.default_dims(gdn_k_heads=kh, gdn_v_heads=vh)
    conv, vd = (2 * kh + vh) * D, vh * D
    f = lambda *n: rng.standard_normal(n).astype(np.float32)  # noqa: E731
    qkv, z, ba = f(T, conv), f(T, vd), f(T, 2 * vh)
    cw, alog, dtb, nw = 0.5 * f(conv, 4), f(vh), f(vh), 1 + 0.1 * f(D)
    win, S = f(conv, 3), 0.1 * f(vh, D, D)
    up = [hip.upload(x) for x in (qkv, z, ba, cw, alog, dtb, nw, ring_from_window(win, pos0))]
    st = hip.malloc(S.nbytes + 16)
    hip.copy_in(st + misalign, S)
    a = pyq35.GdnPrefillArgs(n_tokens=T, pos0=pos0, k_heads=kh, v_heads=vh, head_dim_k=D, head_dim_v=D, conv_kernel=4,
                             eps=d.rms_norm_eps, qkv=up[0], z=up[1], b=up[2], a=up[2] + 4 * vh, ld_qkv=conv, ld_z=vd,
                             ld_ba=2 * vh, conv_w=up[3], A_log=up[4], dt_bias=up[5], norm_w=up[6] if gated else None,
                             conv_ring=up[7], state=st + misalign)
    a.workspace_bytes = pyq35.lib.q35_gdn_prefill_workspace_bytes(C.byref(a))
    a.workspace, a.out = hip.malloc(a.workspace_bytes), hip.malloc(4 * T * vd)
    pyq35.check(pyq35.lib.q35_gdn_prefill(C.byref(a), None))
    hip.sync()
    out, ring, Sd = hip.download(a.out, (T, vd)), hip.download(up[7], (4, conv)), hip.download(st + misalign, S.shape)
    for p in up + [st, a.workspace, a.out]:
        hip.free(p)
    Sr, ref = S.copy(), np.zeros((T, vd), np.float32)
    for t in range(T):
        raw, full = op.gdn_core(d, qkv[t], z[t], ba[t, :vh], ba[t, vh:], cw, alog, dtb, nw, win, Sr)
        ref[t] = full if gated else raw
    np.testing.assert_array_equal(window_from_ring(ring, pos0 + T), win)
    assert rel_l2(Sd, Sr) < REL_L2 and max(rel_l2(out[t], ref[t]) for t in range(T)) < REL_L2


@pytest.mark.parametrize("kh,vh,T,pos0,gated", [
    (16, 16, 1, 0, True), (16, 16, 3, 0, True), (2, 2, 4, 1, True), (2, 2, 5, 6, True), (2, 4, 31, 3, True), (1, 2, 47, 100, True),
    (16, 16, 48, 5, True), (2, 2, 49, 5, True), (2, 2, 17, 2, False)])
def test_few_tokens_vs_oracle(kh, vh, T, pos0, gated):
    run(pyq35.Hip(), kh, vh, T, pos0, seed=T + kh, gated=gated)


def test_unaligned_state():
    run(pyq35.Hip(), 2, 2, 9, 4, seed=1, misalign=8)
