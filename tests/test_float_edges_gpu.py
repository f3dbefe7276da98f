"""The multi-row kernels at the ends of float32: subnormal sums, infinities and NaN.

Their bits rest on the matrix cores rounding each product or fused multiply-add once and keeping
subnormals. Here nothing larger shares a dot product with the subnormal terms, so a flushed one shows
in the output. NaN: the same outputs are NaN as in the reference's order, and the LM head's argmax
(which orders a NaN by its sign) is that of its one-row kernels.
"""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import bits
from tests.test_attention_rows_gpu import attend
from tests.test_head_rows_gpu import in_order

pytestmark = pytest.mark.gpu

TINY = [1e-42, 3e-41, 1e-39, 2e-38]              # subnormal whole; around the smallest normal


def head(x, w):
    """The LM head of rows x by table w (argmax keys a row by atomic maximum), and its row indices."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    (m, h), v = x.shape, len(w)
    packed, y = DeviceArray((-(-v // 64) * 64, h), np.float32), DeviceArray((m, v), np.float32)
    best, index = DeviceArray((m,), np.uint64), DeviceArray((m,), np.int64)
    hip.call("nc_pack_rows64", [packed, DeviceArray.from_host(w)], [v, h])
    hip.call("nc_argmax_clear", [best], [m])
    hip.call("nc_lm_head", [y, best, DeviceArray.from_host(x), packed], [m, v, h, 0, 0])
    hip.call("nc_argmax_index", [index, best], [m, 0])
    hip.sync()
    return y.numpy(), index.numpy()


# rows by table rows by width that take 4 and 16 rows a wave
HEADS = [(5, 40000, 64), (2, 100000, 60), (17, 65537, 64), (40, 46000, 68)]


@pytest.mark.parametrize("m,v,h", HEADS)
def test_head_of_subnormal_products(gpu, m, v, h):
    rng = np.random.default_rng(m)
    x = rng.standard_normal((m, h)).astype(np.float32)
    size = np.array(TINY, np.float32)[np.arange(m) % 4, None]
    w = rng.standard_normal((v, h)).astype(np.float32)
    w *= np.float32(1e-10)
    x = (x * (size / np.float32(1e-10))).astype(np.float32)
    print(f"head subnormal m={m} v={v} h={h}", flush=True)
    expected = in_order(x, w)
    assert (np.abs(expected[0]) < 1e-38).all() and (expected[0] != 0).any()
    y, index = head(x, w)
    assert np.array_equal(bits(y), bits(expected)) and np.array_equal(index, expected.argmax(1))


@pytest.mark.parametrize("m,v,h", HEADS)
def test_head_of_infinities_and_nan(gpu, m, v, h):
    rng = np.random.default_rng(m)
    x, w = (rng.standard_normal(s).astype(np.float32) for s in ((m, h), (v, h)))
    minus = np.array([0xFFC00001], np.uint32).view(np.float32)[0]
    x[0, 3] = 0.0
    x[1, 5] = np.inf
    w[7, 3], w[v - 3, 0], w[v - 2, 1], w[v - 1, 2], w[100, 9] = np.inf, np.nan, minus, -np.inf, np.inf
    print(f"head nan m={m} v={v} h={h}", flush=True)
    with np.errstate(all="ignore"):
        expected = in_order(x, w)
    y, index = head(x, w)
    assert np.array_equal(np.isnan(y), np.isnan(expected))
    assert np.array_equal(bits(y)[~np.isnan(y)], bits(expected)[~np.isnan(expected)])
    for row in range(min(m, 5)):
        one, at = head(x[row:row + 1], w)
        assert np.array_equal(bits(y[row]) >> 31, bits(one[0]) >> 31), row      # a NaN's sign too
        assert index[row] == at[0], row


INT8 = [(33, 731, 40), (17, 1433, 136), (40, 601, 160), (7, 33, 552), (24, 896, 896), (300, 200, 896)]


@pytest.mark.parametrize("m,n,k", INT8)
def test_int8_of_subnormal_sums(gpu, host, m, n, k):
    from nanocompile_amd import kernels
    rng = np.random.default_rng(m + k)
    x = (rng.standard_normal((m, k)) * np.array(TINY)[np.arange(m) % 4, None] / 64).astype(np.float32)
    q = rng.integers(-127, 128, (n, k), dtype=np.int8)
    s = np.exp2(rng.integers(0, 3, n)).astype(np.float32)                      # exact: the sums' own bits
    print(f"int8 subnormal m={m} n={n} k={k}", flush=True)
    expected = host.matmul_i8_f32(x, q, s)
    assert (np.abs(expected[0]) < 1e-38).all() and (expected[0] != 0).any()
    assert np.array_equal(bits(kernels.matmul_i8(x, q, s).numpy()), bits(expected))


@pytest.mark.parametrize("m,n,k", INT8)
def test_int8_of_infinities_and_nan(gpu, host, m, n, k):
    from nanocompile_amd import kernels
    rng = np.random.default_rng(m + k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    q = rng.integers(-127, 128, (n, k), dtype=np.int8)
    q[n // 2, 3] = 0
    x[0, 3], x[1, k - 1], x[2, 0], x[2, 32 % k] = np.inf, np.nan, np.inf, -np.inf
    s = rng.random(n, dtype=np.float32)
    expected, got = host.matmul_i8_f32(x, q, s), kernels.matmul_i8(x, q, s).numpy()
    assert np.isnan(expected[0, n // 2]) and np.isnan(expected[1]).all()
    assert np.array_equal(np.isnan(got), np.isnan(expected))
    assert np.array_equal(bits(got)[~np.isnan(got)], bits(expected)[~np.isnan(expected)])


@pytest.mark.parametrize("m,n,k", [(500, 33, 32), (17, 1000, 160), (33, 700, 640), (24, 896, 896)])
def test_vnni_of_subnormal_and_unusual_scales(gpu, host, m, n, k):
    """Block scales that are subnormal, infinite (times a zero Dp4 too) and NaN."""
    from nanocompile_amd import kernels
    rng = np.random.default_rng(m + k)
    xq, q = (rng.integers(-127, 128, s, dtype=np.int8) for s in ((m, k), (n, k)))
    xs = (rng.random((m, k // 32)) * np.array(TINY)[np.arange(m) % 4, None] / 100).astype(np.float32)
    off = np.zeros((m, 1), np.float32)
    xs[4, 0], xs[5, -1], xs[6, 0] = np.inf, np.nan, np.inf
    xq[6, :32] = 0
    s = np.ones(n, np.float32)
    expected, got = host.matmul_i8_vnni(xq, xs, off, q, s, 32), kernels.matmul_i8_vnni(xq, xs, off, q, s, 32).numpy()
    assert (np.abs(expected[0]) < 1e-38).all() and (expected[0] != 0).any() and np.isnan(expected[6]).all()
    assert np.array_equal(np.isnan(got), np.isnan(expected))
    assert np.array_equal(bits(got)[~np.isnan(got)], bits(expected)[~np.isnan(expected)])


@pytest.mark.parametrize("heads,kv,d,m,past", [(14, 2, 64, 19, 100), (2, 2, 32, 530, 70), (64, 1, 16, 3, 130)])
def test_attention_over_subnormal_values(gpu, host, heads, kv, d, m, past):
    """Values whose weighted sums are subnormal, and scores whose chains are (a scale brings them back)."""
    def values(qkv, kc, vc):
        qkv[:, (heads + kv) * d:] *= np.float32(1e-40)
        vc *= np.float32(1e-40)
    ctx, xq, xs, expected = attend(host, heads, kv, d, m, past, values)
    assert (np.abs(expected) < 1e-38).all() and (expected != 0).any()
    assert np.array_equal(bits(ctx), bits(expected))

    def scores(qkv, kc, vc):
        qkv[:, :(heads + kv) * d] *= np.float32(1e-21)
        kc *= np.float32(1e-21)
    ctx, xq, xs, expected = attend(host, heads, kv, d, m, past, scores, scale=1e38)
    assert np.array_equal(bits(ctx), bits(expected))
    even = attend(host, heads, kv, d, m, past, scores, scale=0.0)[3]
    assert not np.array_equal(bits(even), bits(expected))                      # the scores mattered
