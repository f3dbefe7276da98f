"""The reference's int8 modes over several rows (matrix-core kernels), bit for bit with the host C oracle.

Sizes sit on both sides of the dispatch's lines and at the edges of the tiles: rows and weight
rows that are not whole tiles of 16, widths with blocks past the last whole stage of 128, groups
of 8 past the last whole block of 32, and the smallest widths each kernel takes.
"""

from __future__ import annotations

import numpy as np
import pytest

from oracle import reference as R
from tests.conftest import bits

pytestmark = pytest.mark.gpu


def operands(m, n, k):
    rng = np.random.default_rng(m + 3 * n + 5 * k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[rng.random(x.shape) < 0.01] *= 20
    x[0, :6] = [0.0, -0.0, 1e-38, -1e-42, 1e30, -1e-30]
    q, s = R.quantize_int8((rng.standard_normal((n, k)) * 0.02).astype(np.float32))
    return rng, x, q, s


SHAPES = [(1, 17, 32), (17, 33, 40), (5, 100, 104), (16, 16, 128), (33, 31, 136), (18, 50, 216), (1, 70, 1000),
          (40, 500, 160), (256, 2001, 96), (23, 896, 896), (24, 896, 4864), (130, 3900, 896)]


@pytest.mark.parametrize("m,n,k", SHAPES)
def test_matmul_i8_rows(gpu, host, m, n, k):
    from nanocompile_amd import hip, kernels
    from nanocompile_amd.hip import DeviceArray
    print(f"matmul_i8 m={m} n={n} k={k}", flush=True)
    rng, x, q, s = operands(m, n, k)
    expected = host.matmul_i8_f32(x, q, s)
    assert np.array_equal(bits(kernels.matmul_i8(x, q, s).numpy()), bits(expected))
    bias, residual = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    got = kernels.matmul_i8(x, q, s, bias=bias, residual=residual).numpy()
    assert np.array_equal(bits(got), bits(residual + (expected + bias)))
    if k in (896, 4864):
        h, gate = DeviceArray((m, n), np.float32), DeviceArray.from_host(residual)
        want = DeviceArray((m, n), np.float32)
        hip.call("nc_matmul_i8_silu", [h, DeviceArray.from_host(x), DeviceArray.from_host(kernels.pack_chains(q)),
                                       DeviceArray.from_host(q), DeviceArray.from_host(s), gate], [m, n, k])
        hip.call("nc_silu_mul", [want, gate, DeviceArray.from_host(expected)], [m * n])
        hip.sync()
        assert np.array_equal(bits(h.numpy()), bits(want.numpy()))


def test_matmul_i8_rows_unaligned_operands(gpu, host):
    """x 4 bytes past a 16-byte boundary takes the kernel that reads it an element at a time."""
    from nanocompile_amd import hip, kernels
    from nanocompile_amd.hip import DeviceArray
    m, n, k = 20, 70, 160
    _, x, q, s = operands(m, n, k)
    room = DeviceArray((m * k + 1,), np.float32)
    room.upload(np.concatenate([[0], x.reshape(-1)]).astype(np.float32))
    y = DeviceArray((m, n), np.float32)
    hip.call("nc_matmul_i8", [y, room.ptr + 4, DeviceArray.from_host(kernels.pack_chains(q)),
                              DeviceArray.from_host(q), DeviceArray.from_host(s)], [m, n, k])
    hip.sync()
    assert np.array_equal(bits(y.numpy()), bits(host.matmul_i8_f32(x, q, s)))
