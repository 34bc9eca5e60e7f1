"""k_gemms (small tiles, K split between a workgroup's waves, any alignment) as
its rule picks the tile, against the f64 product: one row, one column, K below,
at and just past its 16-deep blocks and their split over the waves, rows and
columns one past a tile, GEMM operands that start 4 bytes past a 16-byte
boundary, and convolutions whose taps change within a wave's run.  (The rule
picks few of the tiles at these sizes; test_gpu_gemms_forced.py runs each in
every mode.)  Inputs past the operands are NaN, so a read that leaks into an
output shows.  The bound is fp32 accumulation over K terms, sqrt(K) * 2^-24 on
the output's scale, taken four times."""
import numpy as np
import pytest

import oracle
from acfun_amd import capi
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def _tol(K):
    return 4 * np.sqrt(K) * 2.0 ** -24 + 2.0 ** -22


def _padded(t, torch, off):
    """t inside a NaN buffer, `off` floats past its 256-byte aligned start."""
    buf = torch.full((t.numel() + off + 64,), float("nan"), device="cuda")
    buf[off:off + t.numel()] = t.reshape(-1).cuda()
    return buf, buf.data_ptr() + 4 * off


@pytest.mark.parametrize("M,N", [(1, 1), (1, 1000), (17, 15), (16, 64), (49, 512), (65, 131),
                                 (333, 777), (999, 500), (2065, 260)])
@pytest.mark.parametrize("K", [1, 5, 16, 63, 64, 65, 300, 1333])
@pytest.mark.parametrize("off", [0, 1])
def test_gemm_small_tiles(gpu, rng, M, N, K, off):
    torch = pytest.importorskip("torch")
    g = torch.Generator().manual_seed(int(rng.integers(1 << 30)))
    a, b, bias = (torch.rand(s, generator=g) * 2 - 1 for s in ((M, K), (K, N), (N,)))
    ka, pa = _padded(a, torch, off)
    kb, pb = _padded(b, torch, off)
    kbias, pbias = _padded(bias, torch, off)
    y = torch.full((M * N + 8,), 7.0, device="cuda")
    torch.cuda.synchronize()
    act = K & 1
    assert gpu.acfun_dev_gemm_epi(M, N, K, pa, pb, y.data_ptr() + 4 * off, pbias, act, None) == 0
    assert gpu.acfun_sync() == 0
    want = a.double() @ b.double() + bias.double()
    want = want.relu() if act else want
    got = y.cpu().numpy()
    assert rel_err(got[off:off + M * N].reshape(M, N), want.numpy()) < _tol(K)
    assert np.all(got[:off] == 7.0) and np.all(got[off + M * N:] == 7.0)


@pytest.mark.parametrize("N,H,W,Cin,ks,Cout,s,p", [
    (1, 14, 14, 256, 3, 256, 1, 1), (1, 7, 7, 512, 3, 512, 1, 1), (2, 9, 11, 16, 3, 20, 1, 1),
    (1, 14, 14, 512, 3, 512, 2, 1), (3, 13, 10, 48, 5, 33, 2, 2), (1, 28, 28, 512, 1, 100, 2, 0),
    (16, 57, 30, 80, 3, 80, 2, 1), (1, 3, 3, 16, 3, 4, 1, 1), (2, 12, 12, 32, 8, 24, 3, 4),
    # any channel count: taps padded to 4 channels, several taps in a 16-deep block
    (1, 9, 8, 1, 3, 5, 2, 1), (2, 13, 11, 3, 5, 17, 2, 2), (1, 14, 9, 5, 4, 7, 3, 0),
    (1, 45, 10, 248, 3, 32, 1, 1), (1, 24, 11, 28, 7, 32, 2, 3), (3, 12, 7, 37, 3, 33, 1, 1),
    (2, 9, 9, 143, 1, 20, 2, 0), (1, 10, 10, 12, 8, 64, 1, 4)])
def test_conv_small_tiles(gpu, rng, N, H, W, Cin, ks, Cout, s, p):
    torch = pytest.importorskip("torch")
    x = rng.uniform(0, 1, (N, H, W, Cin)).astype(np.float32)
    K = ks * ks * Cin
    w = (rng.standard_normal((K, Cout)) / np.sqrt(K)).astype(np.float32)
    OH, OW = oracle.out_hw(H, W, ks, ks, s, p)
    kx, px = _padded(torch.from_numpy(x), torch, 0)
    kw, pw = _padded(torch.from_numpy(w), torch, 0)
    y = torch.full((N, OH, OW, Cout), float("nan"), device="cuda")
    torch.cuda.synchronize()
    assert gpu.acfun_dev_conv2d(px, N, H, W, Cin, pw, None, ks, ks, Cout, s, p, 1, y.data_ptr(), 1,
                                None) == 0
    assert gpu.acfun_sync() == 0
    want = oracle.conv2d_f64(x, w, None, ks, ks, Cout, s, p, 1, 1)
    assert rel_err(y.cpu().numpy(), want) < _tol(K)


def test_infinities_and_nan_stay_in_their_row(gpu):
    """0 * inf is NaN in the product's own terms only: the rows beside an
    infinite and a NaN row, and K's cleared tail, stay finite."""
    torch = pytest.importorskip("torch")
    M, N, K = 40, 24, 37
    a = torch.rand((M, K), generator=torch.Generator().manual_seed(3))
    b = torch.rand((K, N), generator=torch.Generator().manual_seed(4))
    a[7] = float("inf")
    a[21] = float("nan")
    ta, tb, y = a.cuda(), b.cuda(), torch.zeros((M, N), device="cuda")
    torch.cuda.synchronize()
    assert gpu.acfun_dev_gemm_epi(M, N, K, ta.data_ptr(), tb.data_ptr(), y.data_ptr(), None, 0, None) == 0
    assert gpu.acfun_sync() == 0
    got, want = y.cpu(), (a.double() @ b.double()).float()
    assert bool(torch.isinf(got[7]).all()) and bool(torch.isnan(got[21]).all())
    keep = [i for i in range(M) if i not in (7, 21)]
    assert rel_err(got[keep].numpy(), want[keep].numpy()) < _tol(K)


@pytest.mark.parametrize("N,H,W,Cin,ks,Cout,s,kernel", [
    (33, 83, 65, 16, 3, 224, 2, "k_gemm_f32"),      # 11 tiles of 64 x 64 per CU, K of 144
    (60, 51, 51, 16, 5, 96, 2, "k_gemms"),          # 5 of them, K of 400
    (60, 84, 84, 16, 5, 64, 2, "k_gemms"),          # 6.5 of them in one column
])
def test_many_tiles_keep_the_faster_kernel(gpu, N, H, W, Cin, ks, Cout, s, kernel):
    """Large convolutions of few channels: k_gemm_f32's 128 x 128 tiles."""
    torch = pytest.importorskip("torch")
    K, p = ks * ks * Cin, ks // 2
    g = torch.Generator().manual_seed(Cout)
    x, w = torch.rand((N, H, W, Cin), generator=g), torch.randn((K, Cout), generator=g) / K ** 0.5
    OH, OW = oracle.out_hw(H, W, ks, ks, s, p)
    tx, tw, y = x.cuda(), w.cuda(), torch.full((N, OH, OW, Cout), float("nan"), device="cuda")
    torch.cuda.synchronize()
    gpu.acfun_prof_enable(1)
    assert gpu.acfun_dev_conv2d(tx.data_ptr(), N, H, W, Cin, tw.data_ptr(), None, ks, ks, Cout, s, p, 1,
                                y.data_ptr(), 0, None) == 0
    assert gpu.acfun_sync() == 0
    ran = {name for _, name in capi.prof_report()[0]}
    gpu.acfun_prof_enable(0)
    want = torch.nn.functional.conv2d(x.double().permute(0, 3, 1, 2), w.double().view(ks, ks, Cin, Cout)
                                      .permute(3, 2, 0, 1), stride=s, padding=p).permute(0, 2, 3, 1)
    assert rel_err(y.cpu().numpy(), want.numpy()) < _tol(K)
    assert ran == {kernel}
