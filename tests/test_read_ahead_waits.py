"""A kernel that touches the weights behind it waits for its own loads, not for the touch: the assembly of a small row kernel, two loads of its own, one of
them in a branch as where a row ends, in front of the touch."""
import os
import re
import shutil
import subprocess

import pytest

from matmulfreellm_amd import build

SOURCE = """
#include "%s"
__global__ __launch_bounds__(512) void row_kernel(const float* x, const float* w, int K, MmfAhead ahead, float* out) {
    __shared__ float red[8];
    const int k = threadIdx.x;
    const float a = x[(long)blockIdx.x * K + k];
    float b = 0.0f;
    if (k < K - 512) b = w[512 + k];
    const uint32_t touched = mmf_touch(ahead, blockIdx.x * 8 + (threadIdx.x >> 6));
    const float m = mmf_wave_max(a + b);
    if ((threadIdx.x & 63) == 0) red[threadIdx.x >> 6] = m;
    __syncthreads();
    float most = red[0];
    for (int i = 1; i < 8; ++i) most = fmaxf(most, red[i]);
    out[(long)blockIdx.x * 512 + k] = a / most;
    mmf_touched(touched);
}
"""


@pytest.mark.skipif(not shutil.which(build._hipcc()), reason="no hipcc here: the library was built elsewhere")
def test_no_wait_for_the_touch_in_front_of_the_barrier(tmp_path):
    src, out = tmp_path / "row.hip", tmp_path / "row.s"
    src.write_text(SOURCE % os.path.join(build.CSRC, "mmf_common.h"))
    subprocess.run([build._hipcc(), *build.HIPCC_FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True, capture_output=True)
    lines = [line.split(";")[0].strip() for line in out.read_text().splitlines()]
    code = lines[next(i for i, line in enumerate(lines) if re.match(r"_Z10row_kernel\S*:", line)):]
    loads = [i for i, line in enumerate(code) if re.match(r"(global|buffer)_load", line)]
    barrier = next(i for i, line in enumerate(code) if line.startswith("s_barrier"))
    assert len(loads) == 3 and loads[-1] < barrier
    waits = [int(n) for line in code[:barrier] for n in re.findall(r"vmcnt\((\d+)\)", line)]
    assert waits and min(waits) >= 1, waits
    assert any("vmcnt(" in line for line in code[barrier:])                         # mmf_touched keeps the load
