"""The GDN prefill's forms at the sizes where one hands over to the next, against the oracle's
sequential recurrence at the bars of the other GDN prefill tests. Blocks of up to 36 tokens run
token by token in one launch: the whole 36 and the first chunked size, with one v-head per k-head
(the ring is written by the same launch) and more (a launch of its own), gated and raw. More than
32 v-heads, whole eights of them: the state scan's workgroups go head by head; 40 and 48 heads
beside 33, which keep their order."""
import pytest

import pyq35
from test_gpu_gdn_few_tokens import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kh,vh,T,pos0,gated", [
    (16, 16, 35, 2, True), (16, 16, 36, 1, True), (16, 16, 37, 0, True), (2, 4, 36, 3, True), (1, 2, 36, 2, True),
    (2, 4, 37, 5, True), (1, 3, 36, 7, True), (2, 2, 36, 4, False), (2, 4, 36, 6, False), (2, 4, 1, 3, True),
    (1, 2, 3, 5, True)])
def test_last_block_token_by_token(kh, vh, T, pos0, gated):
    run(pyq35.Hip(), kh, vh, T, pos0, seed=5 * T + vh, gated=gated)


@pytest.mark.parametrize("kh,vh,T,pos0", [(10, 40, 70, 1), (16, 48, 200, 2), (11, 33, 130, 3)])
def test_many_heads(kh, vh, T, pos0):
    run(pyq35.Hip(), kh, vh, T, pos0, seed=T)
