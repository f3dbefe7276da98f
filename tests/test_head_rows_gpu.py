"""nc_lm_head over several rows of x, bit for bit with the reference's order.

The oracle is the order itself (lower.py:255-269: k in order, the product rounded, then the add),
one numpy float32 operation at a time. Sizes sit on both sides of every line of the dispatch
(one-row kernels, 4 and 16 rows a wave), with widths that are not whole stages of 64 and tables
that are not whole blocks of 64 rows.
"""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import bits

pytestmark = pytest.mark.gpu


def in_order(x, w):
    acc = np.zeros((x.shape[0], w.shape[0]), np.float32)
    for k in range(x.shape[1]):
        acc += x[:, k, None] * w[None, :, k]
    return acc


@pytest.mark.parametrize("m,v,h", [
    (2, 38400, 68),            # 4 rows a wave: two rows of four, one piece past a stage
    (5, 16000, 896),           # a remainder of one row
    (1200, 1, 64),             # one table row; one stage exactly
    (17, 65537, 60),           # 16 rows a wave: a remainder of one, no whole stage, one row past a block
    (16, 131071, 132),         # the last block short, rows not a multiple of 4 (no 16-byte stores)
    (333, 6400, 128),
    (2, 90000, 68),            # 4 rows a wave of a narrow table: two rows of four, one piece past a stage
    (7, 25500, 132),           # rows of the table not a whole block, x one row short of two fours
    (10805, 1, 64),            # one table row, three of four waves without work
])
@pytest.mark.parametrize("epilogue", [False, True])
def test_rows_match_the_reference_order(gpu, m, v, h, epilogue):
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    rng = np.random.default_rng(m * 7 + h)
    x = rng.standard_normal((m, h)).astype(np.float32)
    w = (rng.standard_normal((v, h)) * 0.02).astype(np.float32)
    x[0, :8] = [0.0, -0.0, 1e-30, -1e-38, 1e-42, 3e38, -3e38, 1.0]          # products below and above the normals
    w[0, :8] = [-1.0, 2.0, 1e-12, 1e-3, 1.0, 1e-30, 1e-30, -0.0]
    bias = rng.standard_normal(v).astype(np.float32) if epilogue else None
    residual = rng.standard_normal((m, v)).astype(np.float32) if epilogue else None
    packed = DeviceArray((-(-v // 64) * 64, h), np.float32)
    hip.call("nc_pack_rows64", [packed, DeviceArray.from_host(w)], [v, h])
    y = DeviceArray((m, v), np.float32)
    keys, index = DeviceArray((m, -(-v // 64)), np.uint64), DeviceArray((m,), np.int64)
    operands = [None if a is None else DeviceArray.from_host(a) for a in (bias, residual)]
    hip.call("nc_lm_head", [y, keys, DeviceArray.from_host(x), packed, None, *operands], [m, v, h, 0, 1])
    hip.call("nc_argmax_index", [index, keys], [m, -(-v // 64)])
    hip.sync()
    plain = in_order(x, w)
    expected = plain if not epilogue else residual + (plain + bias)
    assert np.array_equal(bits(y.numpy()), bits(expected))
    assert np.array_equal(index.numpy(), plain.argmax(1))
    # one key a row by atomic maximum, no logits
    best = DeviceArray((m,), np.uint64)
    hip.call("nc_argmax_clear", [best], [m])
    hip.call("nc_lm_head", [None, best, DeviceArray.from_host(x), packed], [m, v, h, 0, 0])
    hip.call("nc_argmax_index", [index, best], [m, 0])
    hip.sync()
    assert np.array_equal(index.numpy(), plain.argmax(1))
