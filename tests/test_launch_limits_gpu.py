"""Calls whose workgroups would not fit one dimension of a grid (2^32 threads), a few rows of each against the oracle.

Long outputs over short dot products: gigabytes written in well under a second.
"""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import bits

pytestmark = pytest.mark.gpu


def test_argmax_keys_of_a_large_table(gpu):
    """65,535 rows by 1,048,576 table rows, keys only: every row's argmax, rows spread over the call checked."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    m, v, h = 65535, 1 << 20, 4
    print(f"lm_head m={m} v={v} h={h}", flush=True)
    rng = np.random.default_rng(5)
    x = rng.standard_normal((m, h)).astype(np.float32)
    w = rng.standard_normal((v, h)).astype(np.float32)
    packed, keys = DeviceArray((v, h), np.float32), DeviceArray((m, v // 64), np.uint64)
    index = DeviceArray((m,), np.int64)
    hip.call("nc_pack_rows64", [packed, DeviceArray.from_host(w)], [v, h])
    hip.call("nc_lm_head", [None, keys, DeviceArray.from_host(x), packed], [m, v, h, 0, 1])
    hip.call("nc_argmax_index", [index, keys], [m, v // 64])
    hip.sync()
    got = index.numpy()
    for row in (0, 1, 15, 16, 32767, 65519, 65520, 65534):
        acc = np.zeros(v, np.float32)
        for k in range(h):
            acc += x[row, k] * w[:, k]
        assert got[row] == acc.argmax(), row
    assert len(set(got.tolist())) > 1


def rows_of(array, rows):
    """Rows of a matrix on the device."""
    n = array.shape[1]
    return np.stack([array.view((n,), offset_bytes=4 * n * int(r)).numpy() for r in rows])


def test_vnni_of_many_outputs(gpu, host):
    """65,535 rows by 65,537 weight rows (2^32 outputs and more), the first and last rows bit for bit."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    from oracle import reference as R
    m, n, k = 65535, 65537, 32
    print(f"matmul_i8_vnni m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(6)
    rows = [0, 1, 7, 8, 40000, 65527, 65528, 65534]
    xq = rng.integers(-127, 128, (m, k), dtype=np.int8)
    xs, off = (rng.random((m, 1), dtype=np.float32) for _ in "so")
    q, s = R.quantize_int8((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    y = DeviceArray((m, n), np.float32)
    packed = DeviceArray.from_host(np.zeros(16, np.int8))        # no whole 128: the packed weights are not read
    hip.call("nc_matmul_i8_vnni", [y, *map(DeviceArray.from_host, (xq, xs, off)), packed,
                                   *map(DeviceArray.from_host, (q, s))], [m, n, k, 32])
    hip.sync()
    expected = host.matmul_i8_vnni(xq[rows], xs[rows], off[rows], q, s, 32)
    assert np.array_equal(bits(rows_of(y, rows)), bits(expected))


def test_int8_of_many_outputs(gpu, host):
    """65,535 rows by 131,073 weight rows (2^33 outputs and more), the first and last rows bit for bit."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    from nanocompile_amd.kernels import pack_chains
    from oracle import reference as R
    m, n, k = 65535, 131073, 32
    print(f"matmul_i8 m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(7)
    rows = [0, 1, 15, 16, 40000, 65519, 65520, 65534]
    x = rng.standard_normal((m, k)).astype(np.float32)
    q, s = R.quantize_int8((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    y = DeviceArray((m, n), np.float32)
    hip.call("nc_matmul_i8", [y, *map(DeviceArray.from_host, (x, pack_chains(q), q, s))], [m, n, k])
    hip.sync()
    assert np.array_equal(bits(rows_of(y, rows)), bits(host.matmul_i8_f32(x[rows], q, s)))
