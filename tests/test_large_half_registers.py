"""Registers of __tc::largeHalfProduct as the compiler reports them for gfx950: nothing goes to memory, in any order of the
operands, whether the number of reduction tiles is even or odd; operands that the direct copies cannot take are requested a
whole tile at a time."""
import os
import re
import subprocess

import pytest

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("m,n,k", [(4096, 4096, 384), (4096, 4096, 320), (2632, 3960, 1056)])
@pytest.mark.parametrize("a_transposed", [False, True])
@pytest.mark.parametrize("b_transposed", [False, True])
def test_no_register_is_spilled(tmp_path, a_transposed, b_transposed, m, n, k):
    a = ("K, M", "r_k, m", (k, m)) if a_transposed else ("M, K", "m, r_k", (m, k))
    b = ("N, K", "n, r_k", (n, k)) if b_transposed else ("K, N", "r_k, n", (k, n))
    source = f"def f(float16({a[0]}) A, float16({b[0]}) B) -> (O) {{ O(m, n) +=! float(A({a[1]})) * float(B({b[1]})) }}"
    text, _ = tc.map_only(source, "f", [ShapeOnly(a[2], "float16"), ShapeOnly(b[2], "float16")],
                          "naive;tile=256,256,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert "__tc::largeHalfProduct<" in text.split('extern "C"')[-1]
    path, assembly = tmp_path / "f.hip", tmp_path / "f.s"
    path.write_text(text)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-mllvm", "-amdgpu-kernarg-preload-count=16", "-include", "hip/hip_runtime.h", "-w", "-S",
                    "-o", str(assembly), str(path)], check=True)
    code = assembly.read_text()
    assert re.findall(r"\.vgpr_spill_count: +(\d+)", code) == ["0"] and re.findall(r"\.private_segment_fixed_size: +(\d+)", code) == ["0"]
    # copies through registers: the eight loads of a tile leave one after the other, nothing waits for memory in between
    run = longest = 0
    for line in code.splitlines():
        if "global_load_dwordx4" in line:
            run += 1
            longest = max(longest, run)
        elif "vmcnt" in line:
            run = 0
    assert longest >= 8
