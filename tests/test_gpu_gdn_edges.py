"""The GDN prefill against the oracle's sequential recurrence at the bars of the other GDN prefill
tests: more than 32 v-heads, whole eights of them (the state scan's workgroups go head by head), 40
and 48 heads beside 33, which keep their order."""
import pytest

import pyq35
from test_gpu_gdn_few_tokens import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kh,vh,T,pos0", [(10, 40, 70, 1), (16, 48, 200, 2), (11, 33, 130, 3)])
def test_many_heads(kh, vh, T, pos0):
    run(pyq35.Hip(), kh, vh, T, pos0, seed=T)
