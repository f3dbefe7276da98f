"""The library's own tile for long k loops, on both sides of each line, against the smallest tile bit for bit."""

from __future__ import annotations

import numpy as np
import pytest

from tests.conftest import bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [(1000, 1000, 2048), (1025, 1000, 2048), (320, 2600, 2064), (70, 6336, 2048)])
def test_default_tiles_for_long_k(gpu, m, n, k):
    from nanocompile_amd import kernels
    print(f"default tile m={m} n={n} k={k}", flush=True)
    rng = np.random.default_rng(m + n)
    i8 = lambda *shape: rng.integers(-127, 128, shape, dtype=np.int8)              # noqa: E731
    f32 = lambda *shape: rng.random(shape, dtype=np.float32) * np.float32(1e-2)    # noqa: E731
    xq, xs, q, s, q2, s2 = i8(m, k), f32(m), i8(n, k), f32(n), i8(n, k), f32(n)
    one = kernels.matmul_i8_token(xq, xs, q, s).numpy()
    assert np.array_equal(bits(one), bits(kernels.matmul_i8_token(xq, xs, q, s, schedule=18).numpy()))
    pair = kernels.matmul_i8_token_swiglu(xq, xs, q, s, q2, s2).numpy()
    assert np.array_equal(bits(pair), bits(kernels.matmul_i8_token_swiglu(xq, xs, q, s, q2, s2, schedule=18).numpy()))
