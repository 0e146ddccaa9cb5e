"""The device's ggml_gelu computes x / (1 + e^(−2u)) and keeps the result only
where fp16 rounds both ends of an error interval alike (gelu_tanh_half,
csrc/s3e_internal.h).  Restated here, over every fp16 input: with the
exponential and the reciprocal off by one unit in the last place either way, a
kept result is the entry of ggml's table, and few inputs in use need the table.
The device's own results over every fp16 input: test_gpu_frame_products.py.
"""
import numpy as np

import oracle_lib as orc

F = np.float32


def _ulp(v, by):
    return v if by == 0 else np.nextafter(v, F(np.inf if by > 0 else 0))


def _kept(x, de, dr):
    """The formula in float32 (fma as one rounding of the float64 value): (kept, its fp16 bits)."""
    x64 = x.astype(np.float64)
    p = ((x * x).astype(np.float64) * np.float64(F(-0.10294324)) + np.float64(F(-2.30220819))).astype(F)
    with np.errstate(over="ignore"):
        e = _ulp(np.exp2((x * p).astype(np.float64)).astype(F), de)
        r = _ulp((1.0 / (F(1) + e).astype(np.float64)).astype(F), dr)
    y = x * r
    eps = (np.abs(y).astype(np.float64) * np.float64(F(6e-7)) + (np.abs(x) * F(1.3e-7)).astype(np.float64)).astype(F)
    lo, hi = (y - eps).astype(np.float16).view(np.uint16), (y + eps).astype(np.float16).view(np.uint16)
    return lo == hi, lo


def test_kept_results_are_the_table():
    bits = np.arange(65536, dtype=np.uint32).astype(np.uint16)
    x = bits.view(np.float16).astype(F)
    use = np.abs(x) <= 10  # (values just inside ±10 round to them)
    x, bits = x[use], bits[use]
    table = np.empty(65536, np.uint16)
    orc.LIB.orc_gelu_tanh_table(orc.ptr(table))
    for de in (-1, 0, 1):
        for dr in (-1, 0, 1):
            kept, half = _kept(x, de, dr)
            wrong = kept & (half != table[bits])
            assert not wrong.any(), (de, dr, x[wrong][:4])


def test_few_lookups():
    x = np.random.default_rng(0).standard_normal(200000).astype(np.float16).astype(F)
    assert (~_kept(x, 0, 0)[0]).mean() < 0.01
