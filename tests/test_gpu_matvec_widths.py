"""The matvec at the widths of the 0.8B shape (1024 and 3584, whose chunk count is a compile-time
constant) against the oracle, at the bars of the other matvec tests: fewer rows than a workgroup's,
a last partial workgroup, and both sides of the line (8192 rows) where a wave takes two rows; 3576,
the width below, takes the general kernel."""
import numpy as np
import pytest

import oracle_py as op
import pyq35
from helpers import bf16_bits, rel_l2

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [1024, 3584, 3576])
@pytest.mark.parametrize("rows", [1, 7, 1025, 8191, 8193])
def test_matvec_width(rows, cols):
    rng = np.random.default_rng(rows + cols)
    hip = pyq35.Hip()
    W = bf16_bits(rng.standard_normal((rows, cols)).astype(np.float32) * 0.02)
    x = rng.standard_normal(cols).astype(np.float32)
    dW, dx, dy = hip.upload(W), hip.upload(x), hip.malloc(rows * 4)
    pyq35.check(pyq35.lib.q35_matmul_bf16(dW, dx, dy, rows, cols, None))
    hip.sync()
    y, ref = hip.download(dy, rows), op.matmul_bf16(W, x)
    for p in (dW, dx, dy):
        hip.free(p)
    assert rel_l2(y, ref) < 1e-6
    np.testing.assert_allclose(y, ref, rtol=1e-4, atol=1e-5 * np.abs(ref).max())
