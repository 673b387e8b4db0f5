"""The library's build rule: a kernel that spills vector registers fails it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
MAKEFILE = os.path.join(ROOT, "vegas_amd", "csrc", "Makefile")

KERNEL = """
#include <hip/hip_runtime.h>
__global__ __launch_bounds__(1024) void plain_kernel(float* p) { p[threadIdx.x] *= 2.0f; }
__global__ __launch_bounds__(1024) void many_live_kernel(float* p) {
    float v[%d];
#pragma unroll
    for (int i = 0; i < %d; ++i) v[i] = p[i * 1024 + threadIdx.x];
    __syncthreads();
#pragma unroll
    for (int i = 0; i < %d; ++i) p[i * 1024 + threadIdx.x] = v[i] * v[%d - 1 - i];
}
"""


@pytest.mark.skipif(not shutil.which(os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")), reason="no hipcc")
@pytest.mark.parametrize("live,spills", [(16, False), (200, True)])
def test_spilled_vector_registers_fail_the_build(tmp_path, live, spills):
    """1024 threads leave 128 vector registers each: 200 live values spill."""
    here = str(tmp_path) + "/"
    (tmp_path / "k.hip").write_text(KERNEL % ((live,) * 4))
    obj = here + "_build/k.o"
    r = subprocess.run(["make", "-f", MAKEFILE, "HERE=" + here, "ROOT=" + ROOT, "HDRS=", obj], capture_output=True,
                       text=True)
    assert (r.returncode != 0) == spills, r.stdout + r.stderr
    assert os.path.exists(obj) != spills
    if spills:
        assert "many_live_kernel" in r.stdout and "plain_kernel" not in r.stdout
