"""Every tile of k_gemms in each of its modes, and the switches that choose
between it and its alternatives, in child processes (tests/gpu_gemms_forced.py:
the switches are read once per process)."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _child(mode, **switches):
    env = {k: v for k, v in os.environ.items() if not k.startswith("ACFUN_")}
    r = subprocess.run([sys.executable, "-u", os.path.join(ROOT, "tests", "gpu_gemms_forced.py"), mode],
                       env=dict(env, ACFUN_TUNE_CACHE=os.devnull, **switches), capture_output=True,
                       text=True, timeout=120, cwd=ROOT)
    assert r.returncode == 0 and "forced ok" in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]
    return {ln.split()[1]: ln.split()[2] for ln in r.stdout.split("\n") if ln.startswith("ran ")}


@pytest.mark.parametrize("tile", ["1,1,4", "1,2,4", "1,4,4", "2,4,4", "2,4,2", "4,4,8"])
def test_every_tile(tile):
    _child("tiles", ACFUN_GEMMS=tile)


@pytest.mark.parametrize("switches,want", [
    ({}, dict(gemm="k_gemms", fc="k_gemms", gemm256="k_gemms", conv="k_gemms", conv3x3="k_gemms",
              tiny="k_gemm_f32", tiny1x1="k_gemm_f32", past="k_gemms")),
    ({"ACFUN_GEMMS": "0"}, dict(gemm="k_gemm32", fc="k_gemm_f32+k_splitk_reduce", gemm256="k_gemm32",
                                conv="k_gemm32", conv3x3="k_wino23+k_wino_filter_t")),
    # one tile per CU for the FC layer
    ({"ACFUN_FC_SPLITK": "0"}, dict(gemm="k_gemms", fc="k_gemm32", gemm256="k_gemms", conv="k_gemms",
                                    conv3x3="k_gemms")),
    # the switches of k_gemm32's tiles choose among those
    ({"ACFUN_G32P": "0"}, dict(gemm="k_gemm32", gemm256="k_gemm32", conv="k_gemm32")),
    ({"ACFUN_G32_NOKS": "1"}, dict(gemm="k_gemm32", gemm256="k_gemm32", conv="k_gemm32")),
    ({"ACFUN_G32_KMIN": "64"}, dict(gemm="k_gemm32", gemm256="k_gemm32", conv="k_gemm32")),
], ids=lambda v: "+".join(v) if isinstance(v, dict) else None)
def test_switches(switches, want):
    ran = _child("which", **switches)
    assert {k: ran[k] for k in want} == want
