"""Child process of tests/test_gpu_gemms_forced.py (run as a script; the switches
are read once per process).

  python tests/gpu_gemms_forced.py tiles   -- with ACFUN_GEMMS naming a tile of
      k_gemms, GEMMs and convolutions (channel counts that are and are not
      multiples of 16) at the edges of that tile, with operands 0 and 4 bytes past
      a 16-byte boundary inside NaN-filled buffers, an infinity and a NaN in one
      pixel, and a fused residual;
  python tests/gpu_gemms_forced.py which   -- prints the kernel that each of WHICH
      ran.

Prints each case before its call, and "forced ok" at the end."""
import os
import sys
import tempfile

import numpy as np

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)

import torch  # noqa: E402

import oracle  # noqa: E402
from acfun_amd import acfun0, capi  # noqa: E402
from tests.helpers import rel_err  # noqa: E402

# M, N, K: single rows and columns, tiles ending one past and one short, K from
# less than a block to several folds per wave, a ragged end or none
GEMMS = [(1, 1, 1), (17, 15, 5), (16, 64, 64), (33, 17, 300), (65, 131, 37), (130, 70, 1333),
         (64, 64, 2560), (49, 100, 4099), (1, 77, 6200), (200, 33, 16)]
# N, H, W, Cin, ks, Cout, stride, pad
CONVS = [(1, 9, 11, 16, 3, 20, 1, 1), (2, 14, 13, 48, 5, 33, 2, 2), (1, 7, 7, 512, 3, 70, 1, 1),
         (1, 28, 20, 64, 1, 100, 2, 0), (2, 12, 12, 32, 8, 24, 3, 4), (3, 30, 9, 80, 3, 130, 2, 1),
         (1, 9, 8, 1, 3, 5, 2, 1), (2, 13, 11, 3, 5, 17, 2, 2), (1, 14, 9, 5, 4, 7, 3, 0),
         (1, 20, 10, 248, 3, 66, 1, 1), (1, 24, 11, 28, 7, 132, 2, 3), (3, 12, 7, 37, 3, 33, 1, 1),
         (2, 9, 9, 143, 1, 20, 2, 0), (1, 10, 10, 487, 3, 65, 2, 1)]
# a product, an FC layer, a layer with a tile per CU, a strided and a 3x3/1
# convolution, the smallest unaligned calls and one just past them
WHICH = {"gemm": (196, 256, 512), "fc": (64, 1000, 2048), "gemm256": (1024, 1024, 1024),
         "conv": (1, 14, 14, 256, 3, 256, 2, 1), "conv3x3": (1, 14, 14, 256, 3, 256, 1, 1), "tiny": (9, 79, 16), "tiny1x1": (3, 21, 28, 16, 1, 16, 2, 0),
         "past": (17, 79, 16)}


def _tol(K):
    return 4 * np.sqrt(K) * 2.0 ** -24 + 2.0 ** -22


def _padded(t, off):
    """t inside a NaN buffer, `off` floats past its 256-byte aligned start."""
    buf = torch.full((t.numel() + off + 64,), float("nan"), device="cuda")
    buf[off:off + t.numel()] = t.reshape(-1).cuda()
    return buf, buf.data_ptr() + 4 * off


def _ran(L):
    ran = {name for _, name in capi.prof_report()[0]}
    L.acfun_prof_enable(0)
    return ran


def gemm(L, M, N, K, off, want_kernel):
    g = torch.Generator().manual_seed(M + N + K)
    a, b, bias = (torch.rand(s, generator=g) * 2 - 1 for s in ((M, K), (K, N), (N,)))
    (ka, pa), (kb, pb), (kc, pc) = (_padded(t, off) for t in (a, b, bias))
    y = torch.full((M * N + 8,), 7.0, device="cuda")
    torch.cuda.synchronize()
    L.acfun_prof_enable(1)
    assert L.acfun_dev_gemm_epi(M, N, K, pa, pb, y.data_ptr() + 4 * off, pc, K & 1, None) == 0, capi.last_error()
    assert L.acfun_sync() == 0, capi.last_error()
    ran = _ran(L)
    assert want_kernel is None or ran == {want_kernel}, ran
    want = a.double() @ b.double() + bias.double()
    want = (want.relu() if K & 1 else want).numpy()
    got = y.cpu().numpy()
    err = rel_err(got[off:off + M * N].reshape(M, N), want)
    assert err < _tol(K), err
    assert np.all(got[:off] == 7.0) and np.all(got[off + M * N:] == 7.0)
    return ran


def conv(L, N, H, W, Cin, ks, Cout, s, p, off, want_kernel, odd=None):
    rng = np.random.default_rng(Cin * 31 + Cout)
    K = ks * ks * Cin
    x = rng.uniform(0, 1, (N, H, W, Cin)).astype(np.float32)
    if odd is not None:
        x[N - 1, H // 2, W // 2] = odd
    w = (rng.standard_normal((K, Cout)) / np.sqrt(K)).astype(np.float32)
    b = rng.standard_normal(Cout).astype(np.float32)
    OH, OW = oracle.out_hw(H, W, ks, ks, s, p)
    (kx, px), (kw, pw), (kb, pb) = (_padded(torch.from_numpy(t), off) for t in (x, w, b))
    y = torch.full((N * OH * OW * Cout + 8,), 7.0, device="cuda")
    torch.cuda.synchronize()
    L.acfun_prof_enable(1)
    assert L.acfun_dev_conv2d(px, N, H, W, Cin, pw, pb, ks, ks, Cout, s, p, 1, y.data_ptr() + 4 * off, 0,
                              None) == 0, capi.last_error()
    assert L.acfun_sync() == 0, capi.last_error()
    ran = _ran(L)
    assert want_kernel is None or ran == {want_kernel}, ran
    with np.errstate(invalid="ignore"):
        want = oracle.conv2d_f64(x, w, b, ks, ks, Cout, s, p, 1, 0).ravel()
    got = y.cpu().numpy()
    assert np.all(got[:off] == 7.0) and np.all(got[off + want.size:] == 7.0)
    got = got[off:off + want.size]
    fin = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fin) and (odd is None) == bool(fin.all())
    err = rel_err(got[fin], want[fin])
    assert err < _tol(K), err
    return ran


def residual(L, H, W, Cin, Cout, stride):
    """1x1 convolutions A and B of the input, A's output added in B's epilogue, ReLU."""
    rng = np.random.default_rng(Cin + Cout)
    x = rng.uniform(0, 1, (2, H, W, Cin)).astype(np.float32)
    ws = [(rng.standard_normal((Cin, Cout)) / np.sqrt(Cin)).astype(np.float32) for _ in range(2)]
    bs = [rng.standard_normal(Cout).astype(np.float32) for _ in range(2)]
    ca, cb = (("conv", 1, 1, Cout, stride, 0, w, b) for w, b in zip(ws, bs))
    with tempfile.TemporaryDirectory() as d:
        path = os.path.join(d, "m.acfun")
        acfun0.write(path, Cin, H, W, [ca, ("input", -1), cb, ("add", 0, 1)], version=2)
        m = L.acfun_model_load_ex(path.encode(), 0)
    assert m, capi.last_error()
    want = [oracle.conv2d_f64(x, w, b, 1, 1, Cout, stride, 0, 1, 0) for w, b in zip(ws, bs)]
    want = np.maximum(want[0] + want[1], 0)
    tx, y = torch.from_numpy(x).cuda(), torch.full(want.shape, float("nan"), device="cuda")
    torch.cuda.synchronize()
    L.acfun_prof_enable(1)
    assert L.acfun_dev_model_infer_batch(m, 2, tx.data_ptr(), y.data_ptr(), None) > 0, capi.last_error()
    assert L.acfun_sync() == 0, capi.last_error()
    kernels, layers = capi.prof_report()
    L.acfun_prof_enable(0)
    L.acfun_model_destroy(m)
    assert {n for _, n in kernels} == {"k_gemms"}, kernels
    assert any(lay["residual"] >= -1 for lay in layers), layers
    err = rel_err(y.cpu().numpy(), want)
    assert err < 2 * _tol(Cin), err


def main():
    L = capi.lib()
    assert L.acfun_backend() == 4, capi.last_error()
    if sys.argv[1] == "which":
        for name, shape in WHICH.items():
            ran = (gemm if len(shape) == 3 else conv)(L, *shape, 0, None)
            print("ran", name, "+".join(sorted(ran)), flush=True)
    else:
        for off in (0, 1):
            for case in GEMMS:
                print("gemm", case, off, flush=True)
                gemm(L, *case, off, "k_gemms")
            for case in CONVS:
                print("conv", case, off, flush=True)
                conv(L, *case, off, "k_gemms")
        for odd in (np.inf, np.nan):
            for case in CONVS:
                print("conv", case, odd, flush=True)
                conv(L, *case, 0, "k_gemms", odd)
        for case in ((9, 10, 64, 36, 1), (9, 7, 100, 132, 1), (17, 10, 64, 68, 2)):
            print("residual", case, flush=True)
            residual(L, *case)
    print("forced ok", flush=True)


if __name__ == "__main__":
    main()
