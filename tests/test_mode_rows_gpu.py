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
          (40, 500, 160), (256, 2001, 96), (23, 896, 896), (24, 896, 4864), (130, 3900, 896),
          # the matrix cores' least outputs and widths, every remainder of a width by 128 and by 32
          (257, 97, 32), (33, 731, 40), (5, 4803, 104), (6, 4001, 128), (17, 1433, 136), (18, 1351, 216), (40, 601, 160),
          (16, 16, 640), (4, 17, 520), (7, 33, 552), (19, 50, 744), (1, 31, 3096), (2, 20, 1560), (3, 5, 512)]


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


@pytest.mark.parametrize("m,n,k", [(20, 70, 160), (20, 1300, 160), (30, 900, 896)])
def test_matmul_i8_rows_unaligned_operands(gpu, host, m, n, k):
    """x 4 bytes past a 16-byte boundary takes the kernel that reads it an element at a time."""
    from nanocompile_amd import hip, kernels
    from nanocompile_amd.hip import DeviceArray
    _, x, q, s = operands(m, n, k)
    room = DeviceArray((m * k + 1,), np.float32)
    room.upload(np.concatenate([[0], x.reshape(-1)]).astype(np.float32))
    y = DeviceArray((m, n), np.float32)
    hip.call("nc_matmul_i8", [y, room.ptr + 4, DeviceArray.from_host(kernels.pack_chains(q)),
                              DeviceArray.from_host(q), DeviceArray.from_host(s)], [m, n, k])
    hip.sync()
    assert np.array_equal(bits(y.numpy()), bits(host.matmul_i8_f32(x, q, s)))


@pytest.mark.parametrize("m,n,k", [(500, 33, 32), (17, 1000, 96), (9, 1801, 128), (40, 500, 160), (33, 700, 640),
                                   (129, 130, 1248), (18, 896, 896), (24, 896, 4864), (130, 3900, 896)])
@pytest.mark.parametrize("block", [32, 64])
def test_matmul_i8_vnni_rows(gpu, host, m, n, k, block):
    from nanocompile_amd import hip, kernels
    from nanocompile_amd.hip import DeviceArray
    if k % block:
        pytest.skip("not a whole number of blocks")
    print(f"matmul_i8_vnni m={m} n={n} k={k} block={block}", flush=True)
    rng, x, q, s = operands(m, n, k)
    xq, xs, off = R.quantize_blocks(x, block)
    expected = host.matmul_i8_vnni(xq, xs, off, q, s, block)
    assert np.array_equal(bits(kernels.matmul_i8_vnni(xq, xs, off, q, s, block).numpy()), bits(expected))
    bias, residual = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    got = kernels.matmul_i8_vnni(xq, xs, off, q, s, block, bias=bias, residual=residual).numpy()
    assert np.array_equal(bits(got), bits(residual + (expected + bias)))
    if k in (896, 4864):
        h, gate = DeviceArray((m, n), np.float32), DeviceArray.from_host(residual)
        want = DeviceArray((m, n), np.float32)
        up = [xq, xs, off, kernels.pack_chains_vnni(q), q, s]
        hip.call("nc_matmul_i8_vnni_silu", [h, *map(DeviceArray.from_host, up), gate], [m, n, k, block])
        hip.call("nc_silu_mul", [want, gate, DeviceArray.from_host(expected)], [m * n])
        hip.sync()
        assert np.array_equal(bits(h.numpy()), bits(want.numpy()))


@pytest.mark.parametrize("k", [32, 64, 96, 992, 1024, 1056, 4864])
@pytest.mark.parametrize("aligned", [True, False])
def test_block_quantizer_rows(gpu, k, aligned):
    """Four elements a lane on 16-byte rows, one a lane off them: zeros, NaN, infinities, ties, signed zeros."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    m = 5
    rng = np.random.default_rng(k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[0, :32] = 0.0
    x[1, 7], x[2, k - 1], x[3, 3] = np.nan, -np.inf, -0.0
    x[4, :32] = np.tile([127.0, -0.5, 0.5, 63.5], 8)
    room = DeviceArray((m * k + 1,), np.float32)
    room.upload(np.concatenate([[0], x.reshape(-1)] if not aligned else [x.reshape(-1), [0]]).astype(np.float32))
    xq, xs, off = DeviceArray((m, k), np.int8), DeviceArray((m, k // 32), np.float32), DeviceArray((m,), np.float32)
    hip.call("nc_quantize_blocks", [xq, xs, off, room.ptr + (0 if aligned else 4)], [m, k, 32])
    hip.sync()
    eq, es, eoff = R.quantize_blocks(x, 32)
    finite = [0, 3, 4]
    assert np.array_equal(xq.numpy()[finite], eq[finite])
    assert np.array_equal(bits(xs.numpy()[finite]), bits(es[finite]))
    assert np.array_equal(bits(off.numpy()[finite]), bits(eoff[finite, 0]))
    assert np.array_equal(np.isnan(xs.numpy()), np.isnan(es)) and np.array_equal(np.isinf(xs.numpy()), np.isinf(es))


@pytest.mark.parametrize("k", [32, 96, 1024, 1056])
def test_block_quantizer_rows_agree(gpu, k):
    """The two routes' bytes, scales and offsets over NaN and infinite elements at every place of a block."""
    from nanocompile_amd import hip
    from nanocompile_amd.hip import DeviceArray
    m = 128
    rng = np.random.default_rng(k)
    x = rng.standard_normal((m, k)).astype(np.float32)
    for i, bad in enumerate([np.nan, np.inf, -np.inf, -0.0]):
        x[32 * i + np.arange(32), np.arange(32) + 32 * (i % (k // 32))] = bad
    room = DeviceArray((m * k + 1,), np.float32)
    got = []
    for at in (0, 4):
        room.upload(np.concatenate([x.reshape(-1), [0]] if at == 0 else [[0], x.reshape(-1)]).astype(np.float32))
        outs = DeviceArray((m, k), np.int8), DeviceArray((m, k // 32), np.float32), DeviceArray((m,), np.float32)
        hip.call("nc_quantize_blocks", [*outs, room.ptr + at], [m, k, 32])
        hip.sync()
        got.append([o.numpy() for o in outs])
    assert np.array_equal(got[0][0], got[1][0])
    for a, b in zip(got[0][1:], got[1][1:]):
        assert np.array_equal(np.isnan(a), np.isnan(b)) and np.array_equal(bits(a)[~np.isnan(a)], bits(b)[~np.isnan(b)])
    assert np.isnan(got[0][1]).any() and np.isinf(got[0][1]).any()
