"""bench.py divides a config's work by the duration of the kernel it names, and
takes its traffic from profiles/traffic_<kernel>_<config>.txt: config 1's kernel
is the one the library runs."""
import pytest

import bench
from acfun_amd import capi

pytestmark = pytest.mark.gpu


def test_config1_kernel(gpu):
    torch = pytest.importorskip("torch")
    a, b = torch.rand(1024, 1024, device="cuda"), torch.rand(1024, 1024, device="cuda")
    y = torch.empty_like(a)
    torch.cuda.synchronize()
    gpu.acfun_prof_enable(1)
    assert gpu.acfun_dev_gemm_epi(1024, 1024, 1024, a.data_ptr(), b.data_ptr(), y.data_ptr(), None, 0, None) == 0
    assert gpu.acfun_sync() == 0
    ran = {name for _, name in capi.prof_report()[0]}
    gpu.acfun_prof_enable(0)
    assert ran == {bench.CFG1_KERNEL}
    assert bench.read_traffic(bench.CFG1_KERNEL + "_cfg1") > 3 * 4 * 1024 * 1024
