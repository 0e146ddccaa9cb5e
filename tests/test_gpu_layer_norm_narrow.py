"""LayerNorm over narrow rows (several rows per wave up to 128 values) and the
first wider ones, ragged row counts, against 64 bits.
"""
import numpy as np
import pytest

import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [32, 64, 96, 128, 160, 192, 224, 256, 288])
@pytest.mark.parametrize("rows", [1, 15, 16, 17, 1000])
def test_layer_norm_narrow(ctx, n, rows):
    rng = np.random.default_rng(n + rows)
    x = (rng.standard_normal((rows, n)) * 2 + 0.3).astype(np.float32)
    w, b = rng.standard_normal(n).astype(np.float32), rng.standard_normal(n).astype(np.float32)
    y = ctx.buffer(rows * n * 4)
    ctx.layer_norm(ctx.to_device(x), rows, n, 1e-5, ctx.to_device(w), ctx.to_device(b), y)
    ctx.sync()
    c = x.astype(np.float64) - x.astype(np.float64).mean(-1, keepdims=True)
    ref = c / np.sqrt((c * c).mean(-1, keepdims=True) + 1e-5) * w + b
    # four roundings of 2^-24 and the rounded mean and scale
    assert orc.rel_l2(y.download(np.float32, (rows, n)), ref) <= 5e-7
