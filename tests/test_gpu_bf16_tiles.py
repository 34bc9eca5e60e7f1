"""acfun_gemm_bf16's tiles (64, 128 with one or several per CU, 256) at their
edges: M and N that end 16 past a tile, K below, at and past a chunk, more
stages than chunks.  Against the f64 product of the rounded operands (the
16-aligned region; M and N are multiples of 16 here); the bound is fp32
accumulation over K terms, sqrt(K) * 2^-24 on the output's scale, taken four
times."""
import numpy as np
import pytest

from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


def tile(torch, M, N, K):
    """The launcher's choice: 64, "128 alone" on its CU, 128 or 256, by its fit of
    the busiest CU's time."""
    cus = torch.cuda.get_device_properties(0).multi_processor_count
    k = -(-K // 128) * 128

    def per_cu(b):
        return -(-(-(-M // b) * -(-N // b)) // cus)

    n = per_cu(128)
    us = {64: 3 + per_cu(64) * k * 0.0040, 128: 3 + (k * 0.0090 if n < 2 else n * k * 0.0075),
          256: 4 + per_cu(256) * k * 0.0262}
    if us[256] < us[128] and us[256] < us[64]:
        return 256
    return 64 if us[64] <= us[128] else "128 alone" if n < 2 else 128


@pytest.mark.parametrize("M,N,K,which", [
    (16, 16, 1, 64), (80, 144, 128, 64), (144, 80, 129, 64), (272, 528, 640, 64),
    (1040, 2064, 1100, "128 alone"), (1936, 2032, 384, "128 alone"), (1824, 2048, 128, "128 alone"),
    (1936, 2064, 384, 128), (3008, 2000, 300, 128), (2064, 4112, 130, 128), (4112, 3856, 1030, 128),
    (4080, 4000, 520, 256), (4080, 3856, 1030, 256), (3856, 4096, 640, 256),
])
def test_bf16_tiles(gpu, rng, M, N, K, which):
    torch = pytest.importorskip("torch")
    assert tile(torch, M, N, K) == which
    g = torch.Generator().manual_seed(int(rng.integers(1 << 30)))
    a, b = (torch.rand(s, generator=g) * 2 - 1 for s in ((M, K), (K, N)))
    ta, tb = a.cuda(), b.cuda()
    y = torch.full((M + 1, N), 7.0, device="cuda")        # one row past C stays untouched
    torch.cuda.synchronize()
    assert gpu.acfun_dev_gemm_bf16(M, N, K, ta.data_ptr(), tb.data_ptr(), y.data_ptr(), None) == 0
    assert gpu.acfun_sync() == 0
    want = a.bfloat16().double() @ b.bfloat16().double()
    got = y.cpu()
    assert rel_err(got[:M].numpy(), want.numpy()) < 4 * np.sqrt(K) * 2.0 ** -24 + 2.0 ** -22
    assert bool((got[M] == 7.0).all())
