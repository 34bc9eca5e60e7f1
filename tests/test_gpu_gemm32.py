"""The persistent fp32 GEMM / implicit-GEMM kernel (k_gemm32p) where its tile
list, its chunk cursor and its deferred stores can go wrong: tile counts just
past the CU count (most workgroups run one tile, a few two), K of a single
ragged chunk up to several, ragged M and N, and convolutions whose taps
change in the middle of a tile.  Against the f64 product; the bound is
fp32 accumulation over K terms, sqrt(K) * 2^-24 on each output's scale, taken
four times."""
import numpy as np
import pytest

import oracle
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _tol(K):
    return 4 * np.sqrt(K) * 2.0 ** -24 + 2.0 ** -22


@pytest.mark.parametrize("M,N", [(64 * 257, 64), (64 * 300 - 1, 68), (2113, 516), (64 * 1025, 64)])
@pytest.mark.parametrize("K", [4, 32, 36, 64, 132])
def test_gemm_tile_lists(gpu, rng, M, N, K):
    torch = pytest.importorskip("torch")
    g = torch.Generator().manual_seed(int(rng.integers(1 << 30)))
    a, b, bias = (torch.rand(s, generator=g) * 2 - 1 for s in ((M, K), (K, N), (N,)))
    ta, tb, tbias = (t.cuda() for t in (a, b, bias))
    y = torch.full((M + 1, N), 7.0, device="cuda")       # one row past C stays untouched
    torch.cuda.synchronize()
    for act in (0, 1):
        assert gpu.acfun_dev_gemm_epi(M, N, K, ta.data_ptr(), tb.data_ptr(), y.data_ptr(),
                                      tbias.data_ptr(), act, None) == 0
        assert gpu.acfun_sync() == 0
        want = a.double() @ b.double() + bias.double()
        want = want.relu() if act else want
        got = y.cpu()
        assert rel_err(got[:M].numpy(), want.numpy()) < _tol(K)
        assert bool((got[M] == 7.0).all())


@pytest.mark.parametrize("N,H,W,Cin,ks,Cout,s,p", [
    (27, 50, 50, 64, 3, 68, 2, 1),      # two chunks per tap, ragged M and Cout, 528 tiles
    (21, 41, 43, 64, 3, 64, 1, 0),      # no padding
    (2, 96, 96, 128, 1, 100, 1, 1),     # 1x1 with a border of padding only
])
def test_conv_tile_lists(gpu, rng, N, H, W, Cin, ks, Cout, s, p):
    torch = pytest.importorskip("torch")
    x = rng.uniform(0, 1, (N, H, W, Cin)).astype(np.float32)
    K = ks * ks * Cin
    w = (rng.standard_normal((K, Cout)) / np.sqrt(K)).astype(np.float32)
    OH, OW = oracle.out_hw(H, W, ks, ks, s, p)
    assert -(-N * OH * OW // 64) * -(-Cout // 64) >= 512
    tx, tw = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    y = torch.full((N, OH, OW, Cout), float("nan"), device="cuda")
    torch.cuda.synchronize()
    assert gpu.acfun_dev_conv2d(tx.data_ptr(), N, H, W, Cin, tw.data_ptr(), None, ks, ks, Cout, s,
                                p, 1, y.data_ptr(), 0, None) == 0
    assert gpu.acfun_sync() == 0
    want = oracle.conv2d_f64(x, w, None, ks, ks, Cout, s, p, 1, 0)
    assert rel_err(y.cpu().numpy(), want) < _tol(K)
