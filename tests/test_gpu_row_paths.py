"""s3e_mul_mat's ways through the device by row count and shape.

Products of few rows convert X inside the kernel where that is cheaper: bit
for bit the product of rows converted beforehand, on either side of the rule.  Above, few tiles split K into ranges,
and fp16 products then stage up to six stages at once: against the product in
64 bits, where sums of K fp32 products in any order stay within 1e-6 relative
L2 (2^-24 per sum, averaged over K ≤ 4736).
"""
import ctypes

import numpy as np
import pytest

import oracle_lib as orc
import s3e
from test_zz_no_alloc import _Graphs

pytestmark = pytest.mark.gpu

TYPES = [orc.Q4_0, orc.Q4_1, orc.Q8_0, orc.F16]
VDT = {orc.Q4_0: s3e.TYPE_Q8_0, orc.Q8_0: s3e.TYPE_Q8_0, orc.Q4_1: s3e.TYPE_Q8_1, orc.F16: s3e.TYPE_F16}


def _inputs(ctx, t, M, N, K, seed):
    rng = np.random.default_rng(seed)
    W = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    X = rng.standard_normal((M, K)).astype(np.float32)
    X[:, : 32] *= 0 if M % 2 else 1  # a block of zeros: scale 0
    bias = rng.standard_normal(N).astype(np.float32)
    wb = orc.to_weight_bytes(t, W)
    return wb, X, bias, ctx.weight(t, K, N, wb)


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M,N,K", [(1, 33, 32), (7, 1024, 1024), (32, 96, 160), (33, 130, 4736), (64, 4736, 1024)])
def test_rows_converted_in_the_product(ctx, t, M, N, K):
    _, X, bias, w = _inputs(ctx, t, M, N, K, M + N)
    Xd, Bd, Y0, Y = ctx.to_device(X), ctx.to_device(bias), ctx.buffer(M * N * 4), ctx.buffer(M * N * 4)
    planes = (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
    q, d, s = ctx.buffer(M * K * 2), ctx.buffer(planes), ctx.buffer(planes)
    print(t, M, N, K, flush=True)
    ctx.quantize_rows(VDT[t], Xd, M, K, q, d, s)
    ctx.mul_mat_q(w, q, d, s, M, Y0, Bd)
    ctx.mul_mat(w, Xd, M, Y, Bd)
    ctx.sync()
    assert np.array_equal(Y.download(np.float32, (M, N)), Y0.download(np.float32, (M, N)))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M,N,K", [(1, 33, 32), (7, 130, 224), (16, 96, 1056), (33, 64, 160), (64, 40, 96)])
@pytest.mark.parametrize("at,value", [(4, 2100.0), (1, 3e4), (8, 7e4), (16, 1e7)])
def test_large_values_at_the_end_of_a_row(ctx, t, M, N, K, at, value):
    # the last stage reaches past K: what it reads there must weigh nothing,
    # also where a scale or a sum of the row's last values would be infinite
    wb, X, _, w = _inputs(ctx, t, M, N, K, M + K)
    X[:, -at:] = 0
    X[:, K - at : K - at + 4] = value
    Xd, Y0, Y = ctx.to_device(X), ctx.buffer(M * N * 4), ctx.buffer(M * N * 4)
    planes = (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
    q, d, s = ctx.buffer(M * K * 2), ctx.buffer(planes), ctx.buffer(planes)
    print(t, M, N, K, at, value, flush=True)
    ctx.quantize_rows(VDT[t], Xd, M, K, q, d, s)
    ctx.mul_mat_q(w, q, d, s, M, Y0)
    ctx.mul_mat(w, Xd, M, Y)
    ctx.sync()
    got, want = Y.download(np.float32, (M, N)), Y0.download(np.float32, (M, N))
    assert np.array_equal(got, want, equal_nan=True)
    if value == 2100.0:
        assert np.isfinite(got).all() and orc.rel_l2(got, orc.mul_mat(t, wb, N, K, X)) <= 1e-6


@pytest.mark.parametrize("M,K", [(1, 128), (33, 640), (66, 2176)])
def test_fp6_codes_are_the_int8_codes(ctx, M, K):
    # E3M2 codes of q = 16·h + l, h = (q + 8) >> 4: no negative zeros, whatever the values
    rng = np.random.default_rng(K)
    X = rng.standard_normal((M, K)).astype(np.float32)
    X[0, 32:64] = np.where(np.arange(32) % 2, -1e-40, 1e-40)  # 127 / maximum is infinite: every code of it
    X[-1, 5], X[-1, 70], X[-1, 96:] = np.nan, np.inf, 0
    Mt, planes = (M + 63) // 64 * 64, (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
    q6, q8, d6, d8 = ctx.buffer(3 * Mt * K // 2), ctx.buffer(M * K), ctx.buffer(planes), ctx.buffer(planes)
    Xd = ctx.to_device(X)
    print(M, K, flush=True)
    ctx.quantize_rows(s3e.TYPE_Q8_0_F6X2, Xd, M, K, q6, d6, None)
    ctx.quantize_rows(s3e.TYPE_Q8_0, Xd, M, K, q8, d8, None)
    ctx.sync()
    words = q6.download(np.uint64, (Mt // 64, K // 128, 4, 2, 3, 64)).transpose(0, 5, 1, 2, 3, 4)  # row, stage, block, part, word
    bits = np.unpackbits(np.ascontiguousarray(words).view(np.uint8).reshape(Mt, K // 32, 2, 24), axis=-1, bitorder="little")
    code = (bits.reshape(Mt, K // 32, 2, 32, 6) << np.arange(6)).sum(-1)[:M]
    value = np.array([0, 1, 2, 3, 4, 5, 6, 7, 8], np.int64)
    table = np.full(64, 99, np.int64)
    table[[0, 12, 16, 18, 20, 21, 22, 23, 24]] = value
    table[[44, 48, 50, 52, 53, 54, 55, 56]] = -value[1:]
    want = q8.download(np.int8, (M, K)).astype(np.int64).reshape(M, K // 32, 32)
    tiny = np.zeros(want.shape, bool)
    tiny[0, 1] = True
    got = 16 * table[code[:, :, 0]] + table[code[:, :, 1]]
    assert np.array_equal(got[~tiny], want[~tiny])
    assert set(want[tiny]) == {-1, 0} and np.array_equal(table[code[:, :, 1]][tiny], want[tiny]) and (code[:, :, 0][tiny] == 32).all()


@pytest.mark.parametrize("t", [orc.Q4_0, orc.Q4_1, orc.Q8_0])
@pytest.mark.parametrize("M,N,K", [(1, 33, 32), (16, 96, 224), (64, 64, 256), (65, 96, 256)])
def test_blocks_of_nan_stay_nan(ctx, t, M, N, K):
    # single values that are not numbers are passed over, as ggml's maximum does; a block of nothing else is not
    _, X, _, w = _inputs(ctx, t, M, N, K, M + K)
    X[0, K - 32 :] = np.nan
    X[M // 2, 3] = np.nan
    Xd, Y0, Y = ctx.to_device(X), ctx.buffer(M * N * 4), ctx.buffer(M * N * 4)
    planes = (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
    q, d, s = ctx.buffer(M * K * 2), ctx.buffer(planes), ctx.buffer(planes)
    print(t, M, N, K, flush=True)
    ctx.quantize_rows(VDT[t], Xd, M, K, q, d, s)
    ctx.mul_mat_q(w, q, d, s, M, Y0)
    ctx.mul_mat(w, Xd, M, Y)
    ctx.sync()
    got, want = Y.download(np.float32, (M, N)), Y0.download(np.float32, (M, N))
    assert np.isnan(got[0]).all() and np.isfinite(got[1:]).all()
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("M", [1, 15, 16, 63, 65])
@pytest.mark.parametrize("K", [128, 1152])
def test_fp6_conversion_leaves_rows_past_m(ctx, M, K):
    X = np.random.default_rng(M + K).standard_normal((M, K)).astype(np.float32)
    Mt, Mp, G = (M + 63) // 64 * 64, (M + 127) // 128 * 128, K // 128
    q, d = np.full(3 * Mt * K // 2, 0xA5, np.uint8), np.full(G * Mp * 4, 0xA5A5, np.uint16)
    qd, dd = ctx.to_device(q), ctx.to_device(d)
    print(M, K, flush=True)
    ctx.quantize_rows(s3e.TYPE_Q8_0_F6X2, ctx.to_device(X), M, K, qd, dd, None)
    ctx.sync()
    words = qd.download(np.uint64, (Mt // 64, G, 4, 2, 3, 64)).transpose(0, 5, 1, 2, 3, 4).reshape(Mt, -1)
    scales = dd.download(np.uint16, (G, Mp, 4)).transpose(1, 0, 2).reshape(Mp, -1)
    assert (words[M:] == 0xA5A5A5A5A5A5A5A5).all() and (scales[M:] == 0xA5A5).all()
    want = np.abs(X.reshape(M, -1, 32)).max(-1) / np.float32(127)
    assert np.array_equal(scales[:M].view(np.float16), want.astype(np.float16))


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("M,N,K,shift", [(1, 256, 256, 0), (7, 256, 256, 0), (64, 256, 256, 0), (16, 96, 160, 0), (16, 160, 96, 0),
                                         (33, 256, 256, 5000), (200, 256, 256, 0)])
def test_output_over_input(ctx, t, M, N, K, shift):
    # Y over X, or starting `shift` floats into it
    _, X, bias, w = _inputs(ctx, t, M, N, K, M + N)
    Xd, Bd, Y = ctx.to_device(X), ctx.to_device(bias), ctx.buffer(M * N * 4)
    both = ctx.buffer((shift + M * max(N, K)) * 4)
    over = s3e.DeviceView(both.ptr + 4 * shift, M * N * 4)
    print(t, M, N, K, shift, flush=True)
    ctx.mul_mat(w, Xd, M, Y, Bd)
    both.upload(X)
    ctx.mul_mat(w, both, M, over, Bd)
    ctx.sync()
    got = both.download(np.float32, shift + M * N)[shift:].reshape(M, N)
    assert np.array_equal(got, Y.download(np.float32, (M, N)))


@pytest.mark.parametrize("t", TYPES + [orc.F32])
@pytest.mark.parametrize("M,N,K", [(65, 128, 512), (65, 96, 1024), (129, 1024, 4736), (1601, 1024, 4736),
                                   (200, 130, 2080), (2048, 1024, 448), (1984, 1024, 64), (2049, 1024, 1056)])
def test_split_products(ctx, t, M, N, K):
    wb, X, bias, w = _inputs(ctx, t, M, N, K, M + K)
    Y = ctx.buffer(M * N * 4)
    print(t, M, N, K, flush=True)
    ctx.mul_mat(w, ctx.to_device(X), M, Y, ctx.to_device(bias))
    ctx.sync()
    pick = np.unique(np.r_[0:3, M // 2 : M // 2 + 3, M - 3 : M])  # rows are independent: the oracle takes a few
    if t == orc.F32:
        ref = X[pick].astype(np.float64) @ wb.view(np.float32).reshape(N, K).astype(np.float64).T + bias
    else:
        ref = orc.mul_mat(t, wb, N, K, X[pick]).astype(np.float64) + bias
    got = Y.download(np.float32, (M, N))
    assert np.isfinite(got).all()
    assert orc.rel_l2(got[pick], ref) <= 1e-6


@pytest.mark.parametrize("M", [6144, 6145, 8064, 8193])
def test_fp16_tiles_by_rounds(ctx, M):
    # 384 tiles of 128 x 128 run in 64-row tiles, 392 to 512 wide, 520 in 64-row tiles
    N, K = 1024, 512
    wb, X, bias, w = _inputs(ctx, orc.F16, M, N, K, M)
    Y = ctx.buffer(M * N * 4)
    print(M, flush=True)
    ctx.mul_mat(w, ctx.to_device(X), M, Y, ctx.to_device(bias))
    ctx.sync()
    ref = X.astype(np.float16).astype(np.float64) @ wb.view(np.float16).reshape(N, K).astype(np.float64).T + bias
    assert orc.rel_l2(Y.download(np.float32, (M, N)), ref) <= 1e-6


@pytest.mark.parametrize("t", [orc.Q8_0, orc.F16])
def test_captured_product_sums_in_one_range(ctx, t):
    # a graph must not hold the context's workspace: its replays may run beside other calls
    M, N, K = 300, 512, 1024
    _, X, bias, w = _inputs(ctx, t, M, N, K, 5)
    Xd, Bd = ctx.to_device(X), ctx.to_device(bias)
    planes = (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
    q, d, s = ctx.buffer(M * K * 2), ctx.buffer(planes), ctx.buffer(planes)
    ctx.quantize_rows(VDT[t], Xd, M, K, q, d, s)
    ref, got = ctx.buffer(M * N * 4), ctx.buffer(M * N * 4)
    ctx.mul_mat_q(w, q, d, s, M, ref, Bd)
    ctx.sync()
    want = ref.download(np.float32, (M, N))
    gr = _Graphs()
    g, ex = gr.capture(ctx.stream, lambda: ctx.mul_mat_q(w, q, d, s, M, got, Bd))
    try:
        first = None
        for rep in range(3):
            got.upload(np.full((M, N), np.nan, np.float32))
            assert gr.h.hipGraphLaunch(ex, ctx.stream) == 0
            ctx.sync()
            out = got.download(np.float32, (M, N))
            first = out if first is None else first
            assert np.array_equal(out, first) and orc.rel_l2(out, want) <= 1e-6, rep
            ctx.mul_mat_q(w, q, d, s, M, ref, Bd)  # eager work on the workspace between replays
            ctx.sync()
    finally:
        gr.h.hipGraphExecDestroy(ex)
        gr.h.hipGraphDestroy(g)


@pytest.mark.parametrize("t", [orc.Q4_0, orc.F16])
def test_captured_small_product_beside_large_ones(ctx, t):
    # a captured product of up to 64 rows keeps its partial sums where no larger product writes
    gr = _Graphs()
    gr.h.hipStreamCreateWithFlags.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_uint]
    gr.h.hipStreamSynchronize.argtypes = gr.h.hipStreamDestroy.argtypes = [ctypes.c_void_p]
    other = ctypes.c_void_p()
    assert gr.h.hipStreamCreateWithFlags(ctypes.byref(other), 1) == 0  # hipStreamNonBlocking
    ops = []
    for M, N, K in ((32, 256, 2048), (300, 512, 2048)):  # 4 K ranges; 4 or 8
        _, X, bias, w = _inputs(ctx, t, M, N, K, M)
        Xd, Bd, Y = ctx.to_device(X), ctx.to_device(bias), ctx.buffer(M * N * 4)
        planes = (K + 127) // 128 * 4 * ((M + 127) // 128 * 128) * 2
        q, d, s = ctx.buffer(M * K * 2), ctx.buffer(planes), ctx.buffer(planes)
        ctx.quantize_rows(VDT[t], Xd, M, K, q, d, s)
        ctx.mul_mat_q(w, q, d, s, M, Y, Bd)
        ctx.sync()
        ops.append((M, N, Y, Y.download(np.float32, (M, N)), (w, q, d, s, M, Y, Bd)))
    (M0, N0, Y0, want0, small), (M1, N1, Y1, want1, large) = ops
    g, ex = gr.capture(ctx.stream, lambda: ctx.mul_mat_q(*small))
    try:
        for rep in range(10):
            Y0.upload(np.full((M0, N0), np.nan, np.float32))
            Y1.upload(np.full((M1, N1), np.nan, np.float32))
            for _ in range(4):
                ctx.mul_mat_q(*large)
                assert gr.h.hipGraphLaunch(ex, other) == 0
            ctx.sync()
            assert gr.h.hipStreamSynchronize(other) == 0
            assert np.array_equal(Y0.download(np.float32, (M0, N0)), want0), rep
            assert np.array_equal(Y1.download(np.float32, (M1, N1)), want1), rep
    finally:
        gr.h.hipGraphExecDestroy(ex)
        gr.h.hipGraphDestroy(g)
        gr.h.hipStreamDestroy(other)


def test_first_large_product_allocates_nothing(ctx):
    # a context's first split product, while another stream's capture (global mode) is open: an allocation would end it
    M, N, K = 300, 96, 1024
    c = s3e.Context(0)
    rng = np.random.default_rng(8)
    W, X = (rng.standard_normal(n).astype(np.float32) for n in ((N, K), (M, K)))
    w, Xd, Y = c.weight(orc.F32, K, N, orc.to_weight_bytes(orc.F32, W)), c.to_device(X), c.buffer(M * N * 4)
    x1, q1 = ctx.to_device(X), ctx.buffer(M * K * 2)
    made = []

    def calls():
        c.mul_mat_q(w, Xd, None, None, M, Y)
        ctx.quantize_rows(s3e.TYPE_F16, x1, M, K, q1, None, None)
        made.append(s3e.Context(0))

    gr = _Graphs()
    try:
        g, ex = gr.capture(ctx.stream, calls)
        gr.h.hipGraphExecDestroy(ex)
        gr.h.hipGraphDestroy(g)
        c.sync()
        assert orc.rel_l2(Y.download(np.float32, (M, N)), X.astype(np.float64) @ W.T.astype(np.float64)) <= 1e-6
    finally:
        for b in (w, Xd, Y):
            b.free()
        for x in (c, *made):
            x.close()


def test_f32_noalloc_products_overlap(ctx):
    # two contexts at once: F32 products convert nothing and keep their partial sums apart
    c = s3e.Context(0)
    calls = []
    try:
        for i, x in enumerate((ctx, c)):
            M, N, K = 300 + i, 512, 1024
            _, X, bias, w = _inputs(x, orc.F32, M, N, K, 20 + i)
            Y = x.buffer(M * N * 4)
            args = (w, x.to_device(X), M, Y, x.to_device(bias))
            x.mul_mat_noalloc(*args)
            x.sync()
            calls.append((x, args, Y, Y.download(np.float32, (M, N))))
        for rep in range(5):
            for x, args, Y, want in calls:
                Y.upload(np.full(want.shape, np.nan, np.float32))
            for _ in range(8):
                for x, args, Y, want in calls:
                    x.mul_mat_noalloc(*args)
            for x, args, Y, want in calls:
                x.sync()
                assert np.array_equal(Y.download(np.float32, want.shape), want), rep
        calls[1][1][0].free()
    finally:
        c.close()
