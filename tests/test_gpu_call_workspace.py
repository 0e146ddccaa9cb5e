"""s3e_mul_mat and s3e_flash_attn_ext keep their converted operands in one
workspace per context.  What an earlier call of another size, weight type or
operator left there must not show in a later call's result (bit for bit the
result of a context of its own), calls above the workspace's bound take
memory of their own, and threads that share a context take turns.
"""
import threading

import numpy as np
import pytest

import oracle_lib as orc
import s3e

pytestmark = pytest.mark.gpu


def _mul_mat(c, t, M, N, K, seed):
    rng = np.random.default_rng(seed)
    W = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    X = rng.standard_normal((M, K)).astype(np.float32)
    w, Y = c.weight(t, K, N, orc.to_weight_bytes(t, W)), c.buffer(M * N * 4)
    c.mul_mat(w, c.to_device(X), M, Y)
    c.sync()
    return Y.download(np.float32, (M, N))


def _attn(c, prec, D, nq, nkv, seed):
    rng = np.random.default_rng(seed)
    q, k, v = (rng.standard_normal((2, n, D)).astype(np.float32) for n in (nq, nkv, nkv))
    O = c.buffer(nq * 2 * D * 4)
    nb = [(1, D, n * D, 2 * n * D) for n in (nq, nkv, nkv)]
    c.flash_attn_ext(c.to_device(q), nb[0], c.to_device(k), nb[1], c.to_device(v), nb[2], D, nq, nkv, 2, 1, 0.125, O,
                     prec=prec)
    c.sync()
    return O.download(np.float32, (nq, 2, D))


CALLS = [
    (_mul_mat, (orc.F16, 300, 96, 4736, 1)),      # large values, no scale planes
    (_mul_mat, (orc.Q8_0, 65, 96, 160, 2)),       # K past its last whole stage
    (_attn, (s3e.PREC_F32, 64, 130, 33, 3)),
    (_mul_mat, (orc.Q4_1, 7, 130, 96, 4)),        # small-M kernel
    (_attn, (s3e.PREC_DEFAULT, 256, 40, 1000, 5)),
    (_mul_mat, (orc.Q4_0, 129, 256, 1024, 6)),    # fp6 pairs
    (_attn, (s3e.PREC_F32, 96, 1, 17, 7)),
    (_mul_mat, (orc.Q4_0, 70, 40, 96, 8)),        # int8 codes
]


def _alone(call):
    c = s3e.Context(0)
    out = call[0](c, *call[1])
    c.close()
    return out


def test_calls_share_the_workspace():
    ref = [_alone(call) for call in CALLS]
    c = s3e.Context(0)
    for order in (range(len(CALLS)), reversed(range(len(CALLS)))):
        for i in order:
            fn, args = CALLS[i]
            print(fn.__name__, args, flush=True)
            assert np.array_equal(fn(c, *args), ref[i]), args
    c.close()


def test_threads_take_turns():
    ref = [_alone(CALLS[i]) for i in (0, 1)]
    c, got = s3e.Context(0), {}

    def work(i):
        got[i] = [CALLS[i][0](c, *CALLS[i][1]) for _ in range(8)]

    threads = [threading.Thread(target=work, args=(i,)) for i in (0, 1)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in (0, 1):
        assert len(got.get(i, ())) == 8 and all(np.array_equal(g, ref[i]) for g in got[i])
    c.close()


def test_above_the_bound(ctx):
    # 140 000 rows of 4096 as fp16 are 1.15 GB, above the 1 GiB kept; the rows repeat, so the small product's rows do
    M0, M, N, K = 1000, 140000, 32, 4096
    rng = np.random.default_rng(9)
    W = (rng.standard_normal((N, K)) * 0.02).astype(np.float32)
    X = rng.standard_normal((M0, K)).astype(np.float32)
    w, Y0, Y = ctx.weight(orc.F16, K, N, orc.to_weight_bytes(orc.F16, W)), ctx.buffer(M0 * N * 4), ctx.buffer(M * N * 4)
    ctx.mul_mat(w, ctx.to_device(X), M0, Y0)
    big = ctx.to_device(np.tile(X, (M // M0, 1)))
    ctx.mul_mat(w, big, M, Y)
    ctx.sync()
    ref, out = Y0.download(np.float32, (M0, N)), Y.download(np.float32, (M // M0, M0, N))
    big.free()
    # the two may run tiles of another shape: sums of 4096 fp32 products in another order
    assert max(orc.rel_l2(o, ref) for o in out) <= 1e-6
