"""A loaded model's 3x3 layers keep their F(2,3) filter transform, so the direct
convolution has less to save than in a call that makes the transform: with few
output tiles, more than 32 output channels and at most 48 input channels the
layer stays on the unit kernel, elsewhere it is multiplied directly.  Either way
the transform is made at most once, and a call outside a model multiplies
directly.  Against the f64 convolution."""
import numpy as np
import pytest

import oracle
from acfun_amd import acfun0, capi
from tests.helpers import rel_err

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,H,W,Cin,Cout,kernel", [
    (6, 28, 32, 16, 48, "k_wino23"), (13, 14, 12, 16, 160, "k_wino23"), (4, 28, 32, 48, 48, "k_gemms"),
    (14, 24, 24, 48, 48, "k_wino23"), (41, 14, 14, 64, 64, "k_gemms"), (18, 32, 14, 24, 32, "k_gemms"),
    (12, 10, 10, 48, 96, "k_gemms")])
def test_kept_transform(gpu, rng, tmp_path, N, H, W, Cin, Cout, kernel):
    torch = pytest.importorskip("torch")
    w = (rng.standard_normal((9 * Cin, Cout)) * np.sqrt(2 / (9 * Cin))).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    x = rng.uniform(0, 1, (N, H, W, Cin)).astype(np.float32)
    path = str(tmp_path / "m.acfun")
    acfun0.write(path, Cin, H, W, [("conv", 3, 3, Cout, 1, 1, w, b)], version=2)
    m = gpu.acfun_model_load_ex(path.encode(), 0)
    assert m, capi.last_error()
    tx, tw, tb = (torch.from_numpy(a).cuda() for a in (x, w, b))
    y = torch.full((N, H, W, Cout), float("nan"), device="cuda")
    want = oracle.conv2d_f64(x, w, b, 3, 3, Cout, 1, 1, 1, 0)
    torch.cuda.synchronize()
    seen = []
    try:
        for _ in range(2):
            gpu.acfun_prof_enable(1)
            assert gpu.acfun_dev_model_infer_batch(m, N, tx.data_ptr(), y.data_ptr(), None) > 0
            assert gpu.acfun_sync() == 0
            seen.append({name: n for (_, name), (n, _) in capi.prof_report()[0].items()})
            gpu.acfun_prof_enable(0)
            assert rel_err(y.cpu().numpy(), want) < 1e-3
        gpu.acfun_prof_enable(1)
        assert gpu.acfun_dev_conv2d(tx.data_ptr(), N, H, W, Cin, tw.data_ptr(), tb.data_ptr(), 3, 3, Cout,
                                    1, 1, 1, y.data_ptr(), 0, None) == 0
        assert gpu.acfun_sync() == 0
        call = {name for _, name in capi.prof_report()[0]}
    finally:
        gpu.acfun_prof_enable(0)
        gpu.acfun_model_destroy(m)
    assert all(set(s) - {"k_wino_filter_t"} == {kernel} for s in seen), seen
    assert seen[0].get("k_wino_filter_t", 0) == (kernel == "k_wino23") and "k_wino_filter_t" not in seen[1]
    assert call == {"k_gemms"} and rel_err(y.cpu().numpy(), want) < 1e-3
