"""Calls whose workgroups do not fit one dimension of a grid (2^32 threads), a few rows of each against the oracle.

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
