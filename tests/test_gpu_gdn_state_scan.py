"""The chunked GDN prefill's state scan against the oracle's sequential recurrence, at the bars of
the other GDN prefill tests: one chunk, whole and ragged last chunks, odd and even numbers of
chunks (the scan runs them in pairs), one v-head, 3 v-heads, v-heads = 2 k-heads, a state off its
16-byte alignment; the conv ring is compared exactly."""
import pytest

import pyq35
from test_gpu_gdn_few_tokens import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kh,vh,T,pos0,gated,misalign", [
    (1, 1, 49, 2, True, 0), (1, 1, 64, 0, True, 0), (3, 3, 65, 1, True, 0), (2, 4, 128, 5, True, 0), (2, 2, 129, 6, False, 0),
    (1, 2, 193, 7, True, 0), (16, 16, 257, 3, True, 0), (2, 2, 100, 4, True, 4)])
def test_state_scan_vs_oracle(kh, vh, T, pos0, gated, misalign):
    run(pyq35.Hip(), kh, vh, T, pos0, seed=T + vh, gated=gated, misalign=misalign)
