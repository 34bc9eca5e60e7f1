"""int8 convolutions at tile counts where the launch shape changes: counts that
are no multiple of 8 (workgroups without a tile) up to three per CU and past it, and
weight matrices either side of the preparation's two forms.  Integer sums and specified roundings: bit-exact against the oracle."""
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
    (1, 7, 7, 512, 230, 3, 1, 1),     # 2^20 weights and more: four channels per
    (1, 6, 5, 1031, 1023, 1, 1, 0),   # preparation block, the last block ragged
    (1, 5, 4, 700, 168, 3, 2, 1),     # (1,058,400 of them; 168 / 4 is whole)
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


@pytest.mark.parametrize("K,N", [(4096, 256), (4095, 256), (4099, 259), (8192, 128), (8256, 127)])
def test_gemm_int8_prepared_by_fours(K, N):
    """The weight preparation of a plain product: rows, not taps, to the dword."""
    rng = np.random.default_rng(K + N)
    A = rng.integers(0, 256, (3, K)).astype(np.uint8)
    B = rng.integers(-128, 128, (K, N)).astype(np.int8)
    got = np.full((3, N), -1, np.int32)
    p = lambda a: C.c_void_p(a.ctypes.data)  # noqa: E731
    capi.lib().acfun_gemm_int8(3, N, K, p(A), p(B), p(got))
    assert np.array_equal(got, oracle.gemm_int8(A, B)), capi.last_error()
