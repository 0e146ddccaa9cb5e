"""The products inside a Hiera block and a memory-attention layer, alone: the
attention's projection and one MLP weight are zero, so what comes out is the
product under test.
"""
import contextlib
import os

import numpy as np
import pytest

import oracle_lib as orc
import s3e
from model_patch import patched

pytestmark = pytest.mark.gpu

# Sums in fp32 that tell the K ranges they were formed in: 2^24 in the first
# 512, 1 + 1 (in different stages) in the second, -2^24 in the third.  Ranges
# of 512 added in order give (2^24 + 2) - 2^24 = 2; where the ones meet 2^24
# one at a time both are lost (ties to even) and the sum is 0.
BIG, ONES, BACK = 0, (512, 576), 1024


def _hidden(n, off):
    """fc1 biases (fc1's weight is zero) whose activations are 16384 at BIG and BACK, 16 at ONES, else 0."""
    b = np.full(n, off, np.float32)
    b[[BIG, BACK]] = 16384
    b[list(ONES)] = 16
    return b


def _weights(n_out, n_hidden):
    w = np.zeros((n_out, n_hidden), np.float32)
    w[:, BIG], w[:, BACK], w[:, list(ONES)] = 1024, -1024, 1 / 16
    return w


@contextlib.contextmanager
def _state(ctx, path):
    gm = s3e.Model(ctx, path)
    st = s3e.State(ctx, gm)
    try:
        yield st
    finally:  # also where an assertion holds on to the frame: before the context goes
        st.free()
        gm.free()


@pytest.fixture(scope="module")
def hiera_file(tmpdir_session):
    path = os.path.join(str(tmpdir_session), "products.ggml")
    s3e.synth_write_sam2(path, "hiera_t", img_size=1024, ftype="f16", seed=4, stages=(1, 1, 2, 2), global_idx=())
    return path


@pytest.mark.parametrize("block,side,dim", [(3, 64, 384), (5, 32, 768)])
def test_hiera_fc2_sums_in_ranges_of_512(ctx, hiera_file, tmpdir_session, block, side, dim):
    # 192 tiles in 3 ranges, 96 tiles in 6
    path, p = os.path.join(str(tmpdir_session), f"fc2_{block}.ggml"), f"hiera.blocks.{block}."
    patched(hiera_file, path, {
        p + "attn.proj.weight": 0, p + "attn.proj.bias": 0, p + "mlp.fc1.weight": 0, p + "mlp.fc1.bias": _hidden(4 * dim, -100),
        p + "mlp.fc2.weight": _weights(dim, 4 * dim), p + "mlp.fc2.bias": 0})
    T = side * side
    x, y = ctx.to_device(np.zeros((T, dim), np.float32)), ctx.buffer(T * dim * 4)
    print("hiera block", block, flush=True)
    with _state(ctx, path) as st:
        st.hiera_block(block, x, side, side, y)
        ctx.sync()
        assert (y.download(np.float32, (T, dim)) == 2).all()


def test_memory_attention_linear2_sums_in_ranges_of_512(ctx, tmpdir_session):
    # 4096 rows: 128 tiles in 4 ranges.  The norm at the end shows even channels (2, or 0) against odd ones (1)
    src, path = (os.path.join(str(tmpdir_session), n) for n in ("ma.ggml", "ma_ranges.ggml"))
    p = "mem_attn.layers.0."
    s3e.synth_write_sam2(src, "hiera_t", img_size=64, ftype="f16", seed=13, mem_attn_layers=1, embed_dim=32, stages=(1, 1, 1, 1),
                         global_idx=(), window_spec=(4, 4, 2, 2), bkg=(2, 2))
    w = _weights(256, 2048)
    w[1::2] = 0
    w[1::2, ONES[0]] = 1 / 16
    patched(src, path, {
        p + "sa.out_proj.weight": 0, p + "sa.out_proj.bias": 0, p + "ca.out_proj.weight": 0, p + "ca.out_proj.bias": 0,
        p + "linear1.weight": 0, p + "linear1.bias": _hidden(2048, 0), p + "linear2.weight": w, p + "linear2.bias": 0,
        "mem_attn.norm.weight": 1, "mem_attn.norm.bias": 0})
    N, M = 4096, 64
    zero = ctx.to_device(np.zeros((N, 256), np.float32))
    rope = ctx.to_device(np.ones((N, 128, 2), np.float32))
    out = ctx.buffer(N * 256 * 4)
    print("memory attention", flush=True)
    with _state(ctx, path) as st:
        st.mem_attn(zero, zero, N, zero, zero, M, M, rope, None, out)
        ctx.sync()
        y = out.download(np.float32, (N, 256))
        assert (y[:, ::2] > 0.9).all() and (y[:, 1::2] < -0.9).all()


@pytest.mark.parametrize("ft", ["q8_0", "q4_1", "f16"])
@pytest.mark.parametrize("M", [12, 1200])
def test_nan_key_reaches_every_output(ctx, tmpdir_session, ft, M):
    # one memory token is NaN: with few keys (one range) as with many, no output hides it
    path = os.path.join(str(tmpdir_session), f"ma_nan_{ft}.ggml")
    s3e.synth_write_sam2(path, "hiera_t", img_size=64, ftype=ft, seed=13, std=0.05, random_affine=True, mem_attn_layers=1, embed_dim=32,
                         stages=(1, 1, 1, 1), global_idx=(), window_spec=(4, 4, 2, 2), bkg=(2, 2))
    N, rng = 25, np.random.default_rng(M)
    prompt = rng.standard_normal((M, 64)).astype(np.float32)
    curr, zero = ctx.to_device(rng.standard_normal((N, 256)).astype(np.float32)), ctx.to_device(np.zeros((max(M, N), 256), np.float32))
    rope = ctx.to_device(np.tile(np.float32([1, 0]), (N, 128, 1)))
    print(ft, M, flush=True)
    with _state(ctx, path) as st:
        for bad in (False, True):
            if bad:
                prompt[M // 2] = np.nan
            out = ctx.buffer(N * 256 * 4)
            st.mem_attn(curr, zero, N, ctx.to_device(prompt), zero, M, M, rope, None, out)
            ctx.sync()
            y = out.download(np.float32, (N, 256))
            assert np.isnan(y).all() if bad else np.isfinite(y).all()


def test_gelu_of_every_fp16_value(ctx, tmpdir_session):
    """fc1 + ggml_gelu of an F16 file, bit for bit ggml's fp16 table: every fp16 value below 16 in size, and values that
    round to ±10 from inside."""
    src, path = (os.path.join(str(tmpdir_session), n) for n in ("gelu.ggml", "gelu_all.ggml"))
    s3e.synth_write_sam2(src, "hiera_t", img_size=256, ftype="f16", seed=5, stages=(1, 1, 1, 1), global_idx=())
    T, C, U, first = 4096, 96, 20, 2
    # token t's first normalised channel is a[t]: each fp16 mantissa of [1, 2) and 0 .. 1023 / 1024, both signs
    a = np.concatenate([1 + np.arange(1024) / 1024, np.arange(1024) / 1024])
    a = np.concatenate([a, -a]).astype(np.float32)
    x = np.zeros((T, C), np.float32)  # (mean 0 and variance 1; channels first .. first + U - 1 stay 0)
    x[:, 0], x[:, 1] = a, -a
    fill = C - first - U
    x[:, first + U :] = np.sqrt((C - 2 * a.astype(np.float64) ** 2) / fill)[:, None] * np.where(np.arange(fill) % 2, 1, -1)
    # hidden unit j is a·2^(3 - j) (exact), the last two a·8 ∓ 0.001; fc2 puts unit j into channel first + j
    scale = np.float32(2.0) ** np.r_[3:-15:-1, 3, 3].astype(np.float32)
    bias = np.zeros(4 * C, np.float32)
    bias[U - 2 : U] = -0.001, 0.001
    w1, w2 = np.zeros((4 * C, C), np.float32), np.zeros((C, 4 * C), np.float32)
    w1[:U, 0] = scale
    w2[first + np.arange(U), np.arange(U)] = 1
    p = "hiera.blocks.0."
    patched(src, path, {
        p + "attn.proj.weight": 0, p + "attn.proj.bias": 0, p + "norm2.weight": 1, p + "norm2.bias": 0, p + "mlp.fc1.weight": w1,
        p + "mlp.fc1.bias": bias, p + "mlp.fc2.weight": w2, p + "mlp.fc2.bias": 0})
    normed = orc.layer_norm(x, 1e-6)[:, 0].astype(np.float16)
    assert np.array_equal(normed, a.astype(np.float16))
    pre = normed.astype(np.float32)[:, None] * scale + bias[:U]
    seen = np.unique(np.abs(pre.astype(np.float16)).view(np.uint16))
    assert np.array_equal(seen[seen < np.float16(15.99).view(np.uint16)], np.arange(np.float16(15.99).view(np.uint16)))
    y = ctx.buffer(T * C * 4)
    print("gelu", flush=True)
    with _state(ctx, path) as st:
        st.hiera_block(0, ctx.to_device(x), 64, 64, y)
        ctx.sync()
        got = y.download(np.float32, (T, C))[:, first : first + U]
    want = orc.gelu_tanh(pre).astype(np.float16).astype(np.float32)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("img", [416, 1024])
def test_fpn_products_on_split_fp16_weights(ctx, tmpdir_session, img):
    """The F32 laterals of a quantized file, fp16 pairs on either side: few tiles (six stages in flight) and many, ragged
    rows, K from 96 to 768.  2^-22 per operand and fp32 sums."""
    path = os.path.join(str(tmpdir_session), "fpn.ggml")
    s3e.synth_write_sam2(path, "hiera_t", img_size=1024, ftype="q8_0", seed=6, std=0.05, random_affine=True, stages=(1, 1, 1, 1),
                         global_idx=(), scalp=0)
    files = orc.read_model_file(path)
    gm = s3e.Model(ctx, path)
    st = s3e.State(ctx, gm, img)
    try:
        chw = np.random.default_rng(img).standard_normal((3, img, img)).astype(np.float32)
        st.encode_chw(ctx.to_device(chw))
        ctx.sync()
        for i in (0, 1, 3):  # level 2 also takes level 3 from above
            w, b = (files[f"fpn.convs.{3 - i}." + n][2].astype(np.float64) for n in ("weight", "bias"))
            rows, K = (img // (4 << i)) ** 2, 96 << i
            x, y = st.tensor(f"hiera_stage_{i}").reshape(rows, K), st.tensor(f"neck_trk_{i}").reshape(rows, 256)
            ref = x.astype(np.float64) @ w.reshape(256, K).T + b
            err = orc.rel_l2(y, ref)
            print(img, i, rows, K, err, flush=True)
            assert err <= 1e-6
    finally:
        st.free()
        gm.free()
