"""Attention prefill of few tokens on a long context in workspaces that have room for part of
what the kernel would take: the keys are cut to the room there is. Every result is within the
bar of the other attention tests of the unsplit kernel's (which those compare with the oracle),
and other sums than the unsplit ones show that the keys were cut."""
import ctypes as C

import numpy as np
import pytest

import pyq35
from helpers import REL_L2, rel_l2

pytestmark = pytest.mark.gpu
SLOT = 16 * 258 * 4  # bytes of the partial outputs of 16 rows
HD = 256


class Turn:
    """n tokens at pos0 on a cache of normal keys and values; run(room) with the least workspace
    and `room` bytes more."""

    def __init__(self, hip, nq, nkv, T, pos0, bf16):
        rng = np.random.default_rng(T + pos0)
        self.hip, self.T, self.nq = hip, T, nq
        f = lambda *n: rng.standard_normal(n).astype(np.float32)  # noqa: E731
        ld, maxc = 2 * (nq + nkv) * HD, pos0 + T + 3
        cut = (lambda x: (x.view(np.uint32) >> 16).astype(np.uint16)) if bf16 else (lambda x: x)
        self.kv = [cut(f(nkv, maxc, HD)) for _ in range(2)]
        self.cache = [hip.upload(x) for x in self.kv]
        self.bufs = [hip.upload(f(T, ld)), hip.upload(0.1 * f(HD)), hip.malloc(T * nq * HD * 4)]
        self.args = pyq35.AttnPrefillArgs(
            n_tokens=T, pos0=pos0, q_heads=nq, kv_heads=nkv, head_dim=HD, rotary_dim=64, kv_dtype=int(bf16), max_context=maxc,
            rope_theta=1e7, eps=1e-6, qkv=self.bufs[0], ld_qkv=ld, q_norm=self.bufs[1], k_norm=self.bufs[1],
            k_cache=self.cache[0], v_cache=self.cache[1], out=self.bufs[2])
        self.least = nq * T * HD * 4 + 256
        self.image = 0 if bf16 else nkv * ((pos0 + T + 31) // 32) * 32 * 3072
        self.room = pyq35.lib.q35_attn_prefill_workspace_bytes(C.byref(self.args)) - self.least  # for all of it

    def run(self, room):
        n = self.least + room
        for p, x in zip(self.cache, self.kv):
            self.hip.copy_in(p, x)
        self.args.workspace, self.args.workspace_bytes = self.hip.malloc(n), n
        pyq35.check(pyq35.lib.q35_attn_prefill(C.byref(self.args), None))
        self.hip.sync()
        out = self.hip.download(self.bufs[2], (self.T, self.nq * HD))
        self.hip.free(self.args.workspace)
        return out

    def close(self):
        for p in self.bufs + self.cache:
            self.hip.free(p)


def same(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


@pytest.mark.parametrize("nq,nkv,T,pos0", [(2, 1, 300, 6000), (8, 2, 70, 2500), (6, 2, 33, 9000)])
@pytest.mark.parametrize("bf16", [False, True])
def test_keys_are_cut_to_the_room(nq, nkv, T, pos0, bf16):
    t = Turn(pyq35.Hip(), nq, nkv, T, pos0, bf16)
    try:
        slots = (t.room - t.image) // SLOT  # of the plan without bounds
        assert slots > 8
        whole, full = t.run(0), t.run(t.room)
        assert not same(whole, full) and rel_l2(full, whole) < REL_L2
        groups = -(-T * (nq // nkv) // (64 if bf16 else 128)) * nkv * (4 if bf16 else 8)  # slots of one piece of all blocks
        for k in (slots - 1, slots // 2, 2 * groups, 2 * groups - 1):
            part = t.run(t.image + k * SLOT)
            assert rel_l2(part, whole) < REL_L2, k
            if k >= 2 * groups:  # room for two pieces or more
                assert not same(part, whole), k
        assert same(t.run((2 * groups - 1) * SLOT), whole)  # one piece is no cut
    finally:
        t.close()
