"""Prompt attention on the matrix cores and its combines, bit for bit with the host oracle.

Groups of 1 to 64 query heads a KV head (rows a workgroup takes: 64 down to 1) and one past that,
rows on both sides of a workgroup's block, contexts whose combine is one batch, several, and more
than 64 chunks, more heads than a fused row holds, and values a row must not see that are not
finite.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle.host_model import inverse_frequencies
from oracle import reference as R
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def attend(host, heads, kv, d, m, past, spoil=None, slab=None, schedule=0, scale=None):
    """(ctx, xq, xs) of the GPU and of the oracle for one seeded prompt."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    from nanocompile_amd.kernels import attention_workspace_bytes, float_bits
    print(f"attention heads={heads}/{kv} d={d} m={m} past={past} slab={slab} schedule={schedule}", flush=True)
    rng = np.random.default_rng(heads + 3 * m + 7 * past)
    cap = past + m + 3
    qkv = rng.standard_normal((m, (heads + 2 * kv) * d)).astype(np.float32)
    kc, vc = (rng.standard_normal((kv, cap, d)).astype(np.float32) for _ in "kv")
    if spoil:
        spoil(qkv, kc, vc)
    inv, scale = inverse_frequencies(d, 1e6), float(np.float32(d ** -0.5 if scale is None else scale))
    dq, dk, dv, dinv = (DeviceArray.from_host(a) for a in (qkv, kc, vc, inv))
    expected = host.rope_append_attention(qkv, kc, vc, inv, heads, kv, d, past, scale)
    hip.call("nc_rope_append", [dq, dk, dv, dinv], [m, heads, kv, d, past, cap])
    nbytes = attention_workspace_bytes(heads, d, slab or m, past + m)
    work, ctx = DeviceArray((nbytes // 4,), np.float32), DeviceArray((m, heads * d), np.float32)
    xq, xs = DeviceArray((m, heads * d), np.int8), DeviceArray((m,), np.float32)
    hip.call("nc_attention", [ctx, dq, dk, dv, None, work, xq, xs],
             [m, heads, kv, d, past, cap, float_bits(scale), nbytes, schedule])
    hip.sync()
    return ctx.numpy(), xq.numpy(), xs.numpy(), expected


@pytest.mark.parametrize("heads,kv,d,m,past", [
    (3, 3, 64, 130, 0), (14, 2, 64, 10, 57), (14, 2, 64, 19, 500), (33, 1, 64, 5, 61), (64, 1, 32, 3, 130),
    (66, 1, 16, 4, 60), (17, 17, 16, 70, 64), (6, 2, 64, 9, 4090), (4, 2, 32, 600, 7),
    # small groups with enough rows for the matrix cores
    (3, 3, 64, 300, 200), (17, 17, 16, 70, 300), (6, 2, 64, 40, 4050), (2, 2, 32, 521, 100), (8, 2, 16, 130, 400)])
@pytest.mark.parametrize("slab", [None, 4])
def test_prompt_attention(gpu, host, heads, kv, d, m, past, slab):
    ctx, xq, xs, expected = attend(host, heads, kv, d, m, past, slab=slab)
    assert np.array_equal(bits(ctx), bits(expected))
    eq, es = R.quantize_token(expected)
    assert np.array_equal(xq, eq) and np.array_equal(bits(xs), bits(es))


@pytest.mark.parametrize("m,past", [(30, 50), (70, 0)])
def test_values_a_row_must_not_see(gpu, host, m, past):
    """An infinite value of a later key reaches no earlier row; the rows that see it agree with the oracle."""
    heads, kv, d, at = 14, 2, 64, 23

    def spoil(qkv, kc, vc):
        qkv[at, (heads + kv) * d + 5] = np.inf              # the value of KV head 0's key past + at
    ctx, _, _, expected = attend(host, heads, kv, d, m, past, spoil)
    assert np.isfinite(ctx[:at]).all()
    assert np.array_equal(bits(ctx[:at]), bits(expected[:at]))
    assert np.array_equal(np.isnan(ctx), np.isnan(expected))
    assert np.array_equal(ctx[~np.isnan(ctx)], expected[~np.isnan(ctx)])


@pytest.mark.parametrize("heads,kv,d,schedule", [*((14, 2, 64, s) for s in (1, 2, 3, 4)), (8, 8, 64, 0), (66, 1, 16, 0)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_values_no_schedule_may_see(gpu, host, heads, kv, d, schedule, bad):
    """Every schedule, and groups the matrix cores do not take: an infinite or NaN value of each later key of
    a chunk (every remainder of a row's keys by four) reaches no earlier row."""
    m, past = 26, 50
    spoiled = {16: 2, 19: 0, 21: 3, 22: 1}                      # row: element (keys 66, 69, 71, 72)

    def spoil(qkv, kc, vc):
        for row, e in spoiled.items():
            qkv[row, (heads + kv) * d + e] = bad                # a value of KV head 0
    ctx, xq, xs, expected = attend(host, heads, kv, d, m, past, spoil, schedule=schedule)
    first = min(spoiled)
    assert np.isfinite(ctx[:first]).all()
    assert np.array_equal(bits(ctx[:first]), bits(expected[:first]))
    assert np.array_equal(np.isnan(ctx), np.isnan(expected))
    assert np.array_equal(ctx[~np.isnan(ctx)], expected[~np.isnan(ctx)])


def test_not_a_number_scores(gpu, host):
    """A key with a NaN makes every row that sees it NaN, and no other."""
    heads, kv, d, m, past, at = 14, 2, 64, 40, 30, 17

    def spoil(qkv, kc, vc):
        qkv[at, heads * d] = np.nan                         # the key of KV head 0 at past + at
    ctx, _, _, expected = attend(host, heads, kv, d, m, past, spoil)
    assert np.array_equal(np.isnan(ctx), np.isnan(expected)) and np.isnan(ctx[at:, :d]).all()
    assert np.array_equal(bits(ctx[:at]), bits(expected[:at]))


@pytest.mark.parametrize("past", [447, 448, 520, 4095, 4096, 9000, 16383])
def test_decode_combine_over_long_contexts(gpu, host, past):
    """Decode attention where its combine takes one wave's batch, several of four waves', and the most keys."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    from nanocompile_amd.kernels import attention_workspace_bytes, float_bits
    heads, kv, d, cap = 14, 2, 64, past + 1
    print(f"decode past={past}", flush=True)
    rng = np.random.default_rng(past)
    qkv = rng.standard_normal((1, (heads + 2 * kv) * d)).astype(np.float32)
    kc, vc = (rng.standard_normal((kv, cap, d)).astype(np.float32) for _ in "kv")
    inv, scale = inverse_frequencies(d, 1e6), float(np.float32(d ** -0.5))
    dq, dk, dv, dinv = (DeviceArray.from_host(a) for a in (qkv, kc, vc, inv))
    expected = host.rope_append_attention(qkv, kc, vc, inv, heads, kv, d, past, scale)
    nbytes = attention_workspace_bytes(heads, d, 1, cap)
    work, ctx = DeviceArray((nbytes // 4,), np.float32), DeviceArray((1, heads * d), np.float32)
    pos = DeviceArray.from_host(np.array([past], np.int64))
    for where in (None, pos):
        hip.call("nc_attention_decode", [ctx, dq, dk, dv, dinv, where, None, work],
                 [heads, kv, d, past if where is None else 0, cap, float_bits(scale), nbytes])
        hip.sync()
        assert np.array_equal(bits(ctx.numpy()), bits(expected)), where is not None
