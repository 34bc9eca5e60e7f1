"""int8 convolutions at tile counts where the launch shape changes: counts that
are no multiple of 8 (workgroups without a tile) up to three per CU and past it.
Integer sums and specified roundings: bit-exact against the oracle."""
import ctypes as C

import numpy as np
import pytest

import oracle
from acfun_amd import capi

pytestmark = pytest.mark.gpu

CASES = [  # N, H, W, Cin, Cout, ks, stride, act
    (1, 7, 7, 3, 16, 1, 1, 0),        # one tile
    (2, 13, 11, 48, 77, 3, 2, 1),     # 4, both ragged
    (3, 15, 9, 17, 130, 5, 1, 2),     # 21, padded channels
    (1, 9, 30, 16, 650, 7, 2, 1),     # 22
    (4, 29, 37, 64, 301, 3, 2, 1),    # 90 tiles of 64 x 64
    (1, 65, 63, 32, 65, 1, 1, 0),     # 130 of them, one live column in half
    (5, 57, 56, 24, 128, 3, 1, 1),    # 500
    (1, 112, 113, 40, 250, 1, 1, 1),  # 792: past three per CU
]


@pytest.mark.parametrize("N,H,W,Cin,Cout,ks,stride,act", CASES)
@pytest.mark.parametrize("zero", [False, True])
def test_conv_int8_tile_counts(N, H, W, Cin, Cout, ks, stride, act, zero):
    rng = np.random.default_rng(N * 131 + H * 17 + Cin + Cout)
    pad = ks // 2
    x = rng.standard_normal((N, H, W, Cin)).astype(np.float32)
    if zero:
        x[:] = 0
    wq = rng.integers(-128, 128, (ks * ks * Cin, Cout)).astype(np.int8)
    ws = rng.uniform(0.005, 0.05, Cout).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    oh, ow = (H + 2 * pad - ks) // stride + 1, (W + 2 * pad - ks) // stride + 1
    got = np.full((N, oh, ow, Cout), np.nan, np.float32)
    p = lambda a: C.c_void_p(a.ctypes.data)  # noqa: E731
    capi.lib().acfun_conv2d_int8(p(x), N, H, W, Cin, p(wq), p(ws), p(b), ks, ks, Cout, stride, pad,
                                 0.0, p(got), act)
    want = oracle.conv2d_int8(x, wq, ws, b, ks, ks, Cout, stride, pad, act)
    assert np.array_equal(got, want), capi.last_error()
