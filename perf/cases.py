"""Timed workloads of libacfun_amd.so: what a user of the convolution / GEMM
path has it do, through the C ABI's device-pointer entry points.

listed() holds the fixed workloads, draw(rng) makes others of the same ranges,
prepare()/run() build and run one, work() gives the bytes and operations it
cannot do without, exact() its result in 64 bits and tolerance() how far a
correct fp32 / bf16 implementation may be from another.
"""
import math
import os
import tempfile

import numpy as np
import torch

from acfun_amd import acfun0, capi


def listed():
    return [
        # A square fp32 product: the reference's own GEMM benchmark size.
        dict(name="gemm_1024", kind="gemm", M=1024, N=1024, K=1024, bias=False, act=0),
        # A fully connected layer with no size a multiple of 4 (bias + ReLU):
        # the shapes a caller has who never heard of tiles.
        dict(name="gemm_ragged", kind="gemm", M=999, N=777, K=1333, bias=True, act=1),
        # The bf16 product at the large end of its use.
        dict(name="gemm_bf16_4096", kind="gemm_bf16", M=4096, N=4096, K=4096),
        # The 3x3/1 layer of a ResNet's first stage, batch 32 (Winograd F(2,3)).
        dict(name="conv3x3_56", kind="conv", N=32, H=56, W=56, Cin=64, Cout=64, ks=3, stride=1,
             act=1),
        # The same layer on a twice as large image (Winograd F(4,3)).
        dict(name="conv3x3_112", kind="conv", N=8, H=112, W=112, Cin=64, Cout=64, ks=3, stride=1,
             act=1),
        # A strided 3x3 layer between two ResNet stages, batch 64 (implicit GEMM).
        dict(name="conv3x3s2_56", kind="conv", N=64, H=56, W=56, Cin=128, Cout=128, ks=3,
             stride=2, act=1),
        # Quantized 1x1 and 3x3 layers, float in and out, weights as the caller keeps them.
        dict(name="int8_1x1_28", kind="conv_int8", N=32, H=28, W=28, Cin=256, Cout=512, ks=1,
             stride=1, act=1),
        dict(name="int8_3x3_28", kind="conv_int8", N=32, H=28, W=28, Cin=128, Cout=128, ks=3,
             stride=1, act=1),
        # A mobile network's depthwise layer with its pool: bound by memory.
        dict(name="dw_pool_112", kind="dw_pool", N=32, H=112, W=112, C=96, stride=2),
        # A small grouped layer with its pool: the smallest call.
        dict(name="group_pool_14", kind="group_pool", N=32, H=14, W=14, groups=6, cin=4, cout=8),
        # A ResNet-50-style model on one image: what an interactive caller waits for.
        dict(name="model_fp32_b1", kind="model", N=1, H=224, int8=False),
        # The same model, int8 convolutions, on a batch of 64: offline throughput.
        dict(name="model_int8_b64", kind="model", N=64, H=224, int8=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _channels(rng, lo, hi):
    """Channel counts: two in three a multiple of 16, as networks have them."""
    c = _log(rng, lo, hi)
    return max(16, (c + 8) // 16 * 16) if rng.random() < 2 / 3 else c


def draw(rng):
    kind = rng.choice(["gemm", "gemm_bf16", "conv", "conv", "conv_int8", "conv_int8", "dw_pool",
                       "group_pool", "model"])
    if kind == "gemm":
        return dict(kind=kind, M=_log(rng, 1, 2048), N=_channels(rng, 16, 2048),
                    K=_channels(rng, 16, 4096), bias=rng.random() < 0.5, act=rng.randint(0, 1))
    if kind == "gemm_bf16":
        return dict(kind=kind, M=_log(rng, 64, 4096), N=_channels(rng, 64, 4096),
                    K=_channels(rng, 64, 4096))
    if kind in ("conv", "conv_int8"):
        ks = rng.choice([1, 3, 3, 5, 7] if kind == "conv" else [1, 1, 3, 3])
        c = dict(kind=kind, N=_log(rng, 1, 64), H=_log(rng, 7, 120), W=_log(rng, 7, 120),
                 Cin=_channels(rng, 3, 512), Cout=_channels(rng, 16, 512), ks=ks,
                 stride=rng.choice([1, 1, 2]), act=rng.randint(0, 1))
        while c["N"] > 1 and (work(c)["flops"] > 3e10 or work(c)["bytes"] > 5e8):
            c["N"] = c["N"] // 2
        while work(c)["flops"] > 3e10:
            c["H"], c["W"] = c["H"] // 2 + 3, c["W"] // 2 + 3
            c["Cin"] = max(3, c["Cin"] // 2)
        return c
    if kind == "dw_pool":
        c = dict(kind=kind, N=_log(rng, 1, 64), H=_log(rng, 14, 120), W=_log(rng, 14, 120),
                 C=_channels(rng, 8, 512), stride=rng.randint(1, 2))
        while c["N"] > 1 and work(c)["bytes"] > 5e8:
            c["N"] = c["N"] // 2
        return c
    if kind == "group_pool":
        return dict(kind=kind, N=_log(rng, 1, 64), H=_log(rng, 7, 56), W=_log(rng, 7, 56),
                    groups=rng.randint(2, 8), cin=rng.choice([3, 4, 4, 8, 8, 16]),
                    cout=rng.choice([4, 8, 8, 16, 10]))
    int8 = rng.random() < 0.5
    H = rng.randint(96, 256)
    most = (64 if int8 else 16) * (224 / H) ** 2
    return dict(kind="model", N=min(64, _log(rng, 1, most)), H=H, int8=int8)


# ------------------------------------------------------------------ inputs
_stream = None


def _queue():
    """The caller's stream: one for the whole program."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda") * std


def _out(n, k, stride, pad):
    return (n + 2 * pad - k) // stride + 1


def _inputs(case, seed):
    """The case's device tensors.  Activations are a ReLU's output, weights He-normal."""
    g, k = _gen(seed), case["kind"]
    if k in ("gemm", "gemm_bf16"):
        M, N, K = case["M"], case["N"], case["K"]
        t = dict(a=_normal(g, (M, K)), b=_normal(g, (K, N), 1 / math.sqrt(K)))
        t["bias"] = _normal(g, (N,), 0.1) if case.get("bias") else None
        return t
    if k in ("conv", "conv_int8"):
        K = case["ks"] ** 2 * case["Cin"]
        t = dict(x=_normal(g, (case["N"], case["H"], case["W"], case["Cin"])).relu_(),
                 w=_normal(g, (K, case["Cout"]), math.sqrt(2 / K)),
                 bias=_normal(g, (case["Cout"],), 0.1))
        if k == "conv_int8":  # per-channel symmetric weights, as a quantized checkpoint holds them
            t["ws"] = t["w"].abs().amax(0) / 127
            t["w"] = (t["w"] / t["ws"]).round().clamp(-127, 127).to(torch.int8)
        return t
    if k == "dw_pool":
        return dict(x=_normal(g, (case["N"], case["H"], case["W"], case["C"])).relu_(),
                    w=_normal(g, (case["C"], 3, 3), 0.3), bias=_normal(g, (case["C"],), 0.1))
    if k == "group_pool":
        G, ci, co = case["groups"], case["cin"], case["cout"]
        return dict(x=_normal(g, (case["N"], case["H"], case["W"], G * ci)).relu_(),
                    w=_normal(g, (G, 9 * ci, co), math.sqrt(2 / (9 * ci))),
                    bias=_normal(g, (G * co,), 0.1))
    return dict(x=torch.rand((case["N"], case["H"], case["H"], 3), generator=g, device="cuda"))


def _records(case, seed):
    """The model up to its logits (no softmax)."""
    inC, inH, inW, recs = acfun0.resnet50(np.random.default_rng(seed), in_hw=case["H"])
    return inC, inH, inW, recs[:-1]


class _Model:
    """A loaded model; its handle goes with the object."""

    def __init__(self, case, seed):
        fd, path = tempfile.mkstemp(suffix=".acfun")
        os.close(fd)
        try:
            acfun0.write(path, *_records(case, seed), version=2)
            self.lib = capi.lib()
            self.h = self.lib.acfun_model_load_ex(path.encode(), 1 if case["int8"] else 0)
        finally:
            os.unlink(path)
        if not self.h:
            raise RuntimeError(capi.last_error())
        self.sync = torch.cuda.synchronize

    def __del__(self):
        if getattr(self, "h", None):
            self.sync()
            self.lib.acfun_model_destroy(self.h)


def prepare(case, seed):
    lib, q, t, k = capi.lib(), _queue(), _inputs(case, seed), case["kind"]
    s = q.cuda_stream
    p = {n: (v.data_ptr() if v is not None else None) for n, v in t.items()}
    good = 0
    if k == "gemm":
        y = torch.empty((case["M"], case["N"]), device="cuda")
        call = (lib.acfun_dev_gemm_epi, case["M"], case["N"], case["K"], p["a"], p["b"],
                y.data_ptr(), p["bias"], case["act"], s)
    elif k == "gemm_bf16":
        y = torch.empty((case["M"], case["N"]), device="cuda")
        call = (lib.acfun_dev_gemm_bf16, case["M"], case["N"], case["K"], p["a"], p["b"],
                y.data_ptr(), s)
    elif k in ("conv", "conv_int8"):
        pad = case["ks"] // 2
        y = torch.empty((case["N"], _out(case["H"], case["ks"], case["stride"], pad),
                         _out(case["W"], case["ks"], case["stride"], pad), case["Cout"]),
                        device="cuda")
        x = (p["x"], case["N"], case["H"], case["W"], case["Cin"])
        shape = (case["ks"], case["ks"], case["Cout"], case["stride"], pad)
        if k == "conv":
            call = (lib.acfun_dev_conv2d, *x, p["w"], p["bias"], *shape, 1, y.data_ptr(),
                    case["act"], s)
        else:
            call = (lib.acfun_dev_conv2d_int8, *x, p["w"], p["ws"], p["bias"], *shape,
                    y.data_ptr(), case["act"], s)
    elif k == "dw_pool":
        oh, ow = (_out(case[n], 3, case["stride"], 1) for n in "HW")
        y = torch.empty((case["N"], _out(oh, 3, 2, 1), _out(ow, 3, 2, 1), case["C"]),
                        device="cuda")
        call = (lib.acfun_dev_conv2d_dw_maxpool, p["x"], case["N"], case["H"], case["W"],
                case["C"], p["w"], p["bias"], 3, 3, case["stride"], 1, 1, 3, 2, 1, y.data_ptr(),
                0, s)
    elif k == "group_pool":
        G = case["groups"]
        y = torch.empty((case["N"], _out(case["H"], 3, 2, 1), _out(case["W"], 3, 2, 1),
                         G * case["cout"]), device="cuda")
        call = (lib.acfun_dev_conv2d_g_maxpool, p["x"], case["N"], case["H"], case["W"],
                G * case["cin"], p["w"], p["bias"], 3, 3, G * case["cout"], 1, 1, G, 1, 3, 2, 1,
                y.data_ptr(), 0, s)
    else:
        t["model"] = _Model(case, seed)
        y = torch.empty((case["N"], 1000), device="cuda")
        call = (lib.acfun_dev_model_infer_batch, t["model"].h, case["N"], p["x"], y.data_ptr(), s)
        good = 1000
    q.wait_stream(torch.cuda.current_stream())
    return dict(call=call[0], args=call[1:], good=good, y=y, keep=t)


def run(state):
    if state["call"](*state["args"]) != state["good"]:
        raise RuntimeError(capi.last_error())
    return state["y"]


# ------------------------------------------------------------------ work
def _conv_flops(N, H, W, Cin, Cout, ks, stride, wino=True):
    """Products and sums of a convolution by the algorithm its sizes get: the
    Winograd forms' transform-domain products where the path uses one."""
    pad = ks // 2
    if wino and ks == 3 and stride == 1 and min(H, W) >= 3 and min(Cin, Cout) >= 4:
        if min(H, W) >= 112 and min(Cin, Cout) >= 64:
            return 2 * N * -(-H // 4) * -(-W // 4) * 36 * Cin * Cout
        return 2 * N * -(-H // 2) * -(-W // 2) * 16 * Cin * Cout
    return 2 * N * _out(H, ks, stride, pad) * _out(W, ks, stride, pad) * ks * ks * Cin * Cout


def _model_work(case):
    """(flops, parameters) of the model's convolutions and head."""
    N, h, wino = case["N"], _out(case["H"], 7, 2, 3), not case["int8"]
    fl, params = _conv_flops(N, case["H"], case["H"], 3, 64, 7, 2), 147 * 64
    h, cin = _out(h, 3, 2, 1), 64
    for stage, blocks in enumerate((3, 4, 6, 3)):
        mid = 64 << stage
        for b in range(blocks):
            st = 2 if b == 0 and stage else 1
            o = _out(h, 3, st, 1)
            fl += _conv_flops(N, h, h, cin, mid, 1, 1) + _conv_flops(N, h, h, mid, mid, 3, st, wino)
            fl += _conv_flops(N, o, o, mid, 4 * mid, 1, 1)
            params += cin * mid + 9 * mid * mid + 4 * mid * mid
            if b == 0:
                fl += _conv_flops(N, o, o, cin, 4 * mid, 1, 1)
                params += 4 * cin * mid
            h, cin = o, 4 * mid
    return fl + 2 * N * cin * 1000, params


def work(case):
    k = case["kind"]
    if k in ("gemm", "gemm_bf16"):
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": 4 * (M * K + K * N + M * N), "flops": 2 * M * N * K}
    if k in ("conv", "conv_int8"):
        N, H, W, ci, co, ks, st = (case[n] for n in ("N", "H", "W", "Cin", "Cout", "ks", "stride"))
        o = _out(H, ks, st, ks // 2) * _out(W, ks, st, ks // 2)
        wb = 4 if k == "conv" else 1
        return {"bytes": 4 * N * (H * W * ci + o * co) + wb * ks * ks * ci * co,
                "flops": _conv_flops(N, H, W, ci, co, ks, st, k == "conv")}
    if k == "dw_pool":
        N, H, W, C, st = (case[n] for n in ("N", "H", "W", "C", "stride"))
        oh, ow = _out(H, 3, st, 1), _out(W, 3, st, 1)
        return {"bytes": 4 * N * C * (H * W + _out(oh, 3, 2, 1) * _out(ow, 3, 2, 1)),
                "flops": 18 * N * C * oh * ow}
    if k == "group_pool":
        N, H, W, G, ci, co = (case[n] for n in ("N", "H", "W", "groups", "cin", "cout"))
        return {"bytes": 4 * N * G * (H * W * ci + _out(H, 3, 2, 1) * _out(W, 3, 2, 1) * co),
                "flops": 18 * N * G * H * W * ci * co}
    fl, params = _model_work(case)
    return {"bytes": (1 if case["int8"] else 4) * params + 4 * 2048 * 1000
            + 4 * case["N"] * (3 * case["H"] ** 2 + 1000), "flops": fl}


def tolerance(case):
    k = case["kind"]
    if k in ("conv_int8", "dw_pool", "group_pool"):
        return "exact"           # every rounding of these paths is specified
    if k == "conv" and min(case["H"], case["W"]) >= 112 and case["ks"] == 3:
        return {"rel": 6e-6}     # F(4,3)'s transforms: 1.3e-6 from the 64-bit result
    # 32-bit sums, 2e-7 to 7e-7 from the 64-bit result; an int8 model differs in its fp32 head only
    return {"rel": 3e-6}


# ------------------------------------------------------------------ in 64 bits
def _windows(x, kh, kw, stride, pad, fill):
    """The taps of a sliding window over NHWC x, row by row."""
    N, H, W, C = x.shape
    oh, ow = _out(H, kh, stride, pad), _out(W, kw, stride, pad)
    p = x.new_full((N, H + 2 * pad, W + 2 * pad, C), fill)
    p[:, pad:pad + H, pad:pad + W] = x
    for i in range(kh):
        for j in range(kw):
            yield p[:, i:i + (oh - 1) * stride + 1:stride, j:j + (ow - 1) * stride + 1:stride]


def _conv64(x, w, ks, stride, pad):
    """x [N,H,W,Cin], w [ks*ks*Cin, Cout], both float64."""
    C, y = x.shape[3], 0
    for i, v in enumerate(_windows(x, ks, ks, stride, pad, 0.0)):
        y = y + (v.reshape(-1, C) @ w[i * C:(i + 1) * C].contiguous()).view(*v.shape[:3], -1)
    return y


def _pool64(x, pad=1):
    y = None
    for v in _windows(x, 3, 3, 2, pad, -math.inf):
        y = v if y is None else torch.maximum(y, v)
    return y


def _exact_int8(case, t):
    """The quantization is part of the definition (fp32, rounded as the route
    rounds); the products and the scaling are taken in 64 bits."""
    x, ks = t["x"], case["ks"]
    top = x.abs().max()
    v = x * (torch.tensor(127.0, device="cuda") / top)
    if ks == 3 and case["stride"] == 1 and min(case["H"], case["W"]) >= 3 and case["Cin"] >= 4:
        q = torch.trunc(v + torch.copysign(torch.tensor(0.5, device="cuda"), v))
    else:
        q = torch.round(v)
    q = q.clamp(-128, 127)
    y = _conv64(q.double(), t["w"].double(), ks, case["stride"], ks // 2)
    y = y * (top.double() / 127 * t["ws"].double()) + t["bias"].double()
    return y.relu() if case["act"] else y


def _exact_model(case, seed, x):
    """The records one by one; batch norms take their stored statistics."""
    _, _, _, recs = _records(case, seed)
    d = lambda a: torch.from_numpy(np.asarray(a)).to("cuda").double()  # noqa: E731
    cur, outs = x.double(), []
    for r in recs:
        if r[0] == "conv":
            cur = _conv64(cur, d(r[6]).view(-1, r[3]), r[1], r[4], r[5]) + d(r[7])
        elif r[0] == "bn":
            mean, var, gamma, beta = (d(a) for a in r[2:6])
            cur = (cur - mean) * (gamma / torch.sqrt(var + 1e-5)) + beta
        elif r[0] == "relu":
            cur = cur.relu()
        elif r[0] == "maxpool":
            cur = _pool64(cur, r[3])
        elif r[0] == "input":
            cur = outs[r[1]]
        elif r[0] == "add":
            cur = cur + outs[r[1]]
            cur = cur.relu() if r[2] else cur
        elif r[0] == "gap":
            cur = cur.mean((1, 2))
        elif r[0] == "fc":
            cur = cur.reshape(cur.shape[0], -1) @ d(r[3]) + d(r[4])
        outs.append(cur)
    return cur


def exact(case, seed):
    k, t = case["kind"], _inputs(case, seed)
    if k == "gemm":
        y = t["a"].double() @ t["b"].double()
        y = y + t["bias"].double() if case["bias"] else y
        return y.relu() if case["act"] else y
    if k == "gemm_bf16":
        # full 16 x 16 tiles round their operands to bf16, the ragged edge does not
        y = t["a"].double() @ t["b"].double()
        m, n = case["M"] // 16 * 16, case["N"] // 16 * 16
        y[:m, :n] = t["a"][:m].bfloat16().double() @ t["b"][:, :n].bfloat16().double()
        return y
    if k == "conv":
        y = _conv64(t["x"].double(), t["w"].double(), case["ks"], case["stride"], case["ks"] // 2)
        y = y + t["bias"].double()
        return y.relu() if case["act"] else y
    if k == "conv_int8":
        return _exact_int8(case, t)
    if k == "dw_pool":
        w, y = t["w"].double().reshape(-1, 9), t["bias"].double()
        for i, v in enumerate(_windows(t["x"].double(), 3, 3, case["stride"], 1, 0.0)):
            y = y + v * w[:, i]
        return _pool64(y.relu())
    if k == "group_pool":
        ci, x, w = case["cin"], t["x"].double(), t["w"].double()
        y = torch.cat([_conv64(x[..., g * ci:(g + 1) * ci].contiguous(), w[g], 3, 1, 1)
                       for g in range(case["groups"])], 3)
        return _pool64((y + t["bias"].double()).relu())
    if case["int8"]:
        return None   # a flip of one quantized value in an early layer moves all that follow
    return _exact_model(case, seed, t["x"])
