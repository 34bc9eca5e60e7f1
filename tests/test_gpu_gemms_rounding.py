"""Rounding error of k_gemms's long reductions against the f64 product.  Adding n
products in fp32 one after another leaves a relative error (2-norm, random
terms) of about 0.72 * 2^-24 * sqrt(n / 6): each of the n sums rounds by at most
half an ulp of a partial sum whose square grows linearly.  The kernel adds 256 at
a time and then the K / 256 partial sums (and the waves' four); the bound is that
with a fifth on top.  Four waves with a chain of K / 4 each are past it from
K = 2048 on."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _bound(K):
    return 1.2 * 0.72 * 2.0 ** -24 * np.sqrt((256 + K / 256 + 4) / 6)


def _error(got, want):
    return float((got.double() - want).norm() / want.norm())


@pytest.mark.parametrize("M,N,K", [
    (1, 1000, 2048), (64, 1000, 2048), (16, 512, 6144), (64, 256, 4096),   # whole blocks
    (100, 130, 3000), (4, 1024, 4095), (256, 4096, 2050),                  # a ragged end
    (1500, 1024, 4096),                                                    # 64 x 64 tiles on eight waves
])
def test_gemm_rounding(gpu, M, N, K):
    torch = pytest.importorskip("torch")
    g = torch.Generator().manual_seed(M + N + K)
    a, b = torch.randn((M, K), generator=g), torch.randn((K, N), generator=g)
    ta, tb, y = a.cuda(), b.cuda(), torch.empty((M, N), device="cuda")
    torch.cuda.synchronize()
    assert gpu.acfun_dev_gemm_epi(M, N, K, ta.data_ptr(), tb.data_ptr(), y.data_ptr(), None, 0, None) == 0
    assert gpu.acfun_sync() == 0
    assert _error(y.cpu(), a.double() @ b.double()) < _bound(K)


@pytest.mark.parametrize("N,H,W,Cin,ks,Cout,s", [
    (1, 7, 7, 512, 3, 512, 1), (2, 12, 76, 487, 3, 16, 2), (2, 88, 65, 80, 5, 41, 2),
    (1, 14, 14, 1024, 1, 512, 2)])
def test_conv_rounding(gpu, N, H, W, Cin, ks, Cout, s):
    torch = pytest.importorskip("torch")
    K, p = ks * ks * Cin, ks // 2
    g = torch.Generator().manual_seed(Cin + Cout)
    x, w = torch.randn((N, H, W, Cin), generator=g), torch.randn((K, Cout), generator=g)
    tx, tw = x.cuda(), w.cuda()
    oh, ow = (H + 2 * p - ks) // s + 1, (W + 2 * p - ks) // s + 1
    y = torch.empty((N, oh, ow, Cout), device="cuda")
    torch.cuda.synchronize()
    assert gpu.acfun_dev_conv2d(tx.data_ptr(), N, H, W, Cin, tw.data_ptr(), None, ks, ks, Cout, s, p,
                                1, y.data_ptr(), 0, None) == 0
    assert gpu.acfun_sync() == 0
    want = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2),
                                      w.double().view(ks, ks, Cin, Cout).permute(3, 2, 0, 1), stride=s,
                                      padding=p).permute(0, 2, 3, 1)
    assert _error(y.cpu(), want) < _bound(K)
