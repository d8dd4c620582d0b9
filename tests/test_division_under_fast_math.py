"""Divisions by whole numbers known at compile time, compiled as TC_FAST_MATH has them compiled: the one multiplication that
the option makes of any division by a constant."""
import os
import re
import subprocess

import pytest

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("fast", [False, True])
def test_the_option_makes_it_one_multiplication(tmp_path, fast):
    text, _ = tc.map_only("def f(float(N) A) -> (O) { O(n) = A(n) / 3448 }", "f", [ShapeOnly((4096,))], "naive;tile=256;mapToThreads=256")
    assert "/ __tc::Whole<3448>()" in text
    source, assembly = tmp_path / "f.hip", tmp_path / "f.s"
    source.write_text(text)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-include", "hip/hip_runtime.h", "-w", "-S", "-o", str(assembly), str(source)] +
                   (["-ffast-math"] if fast else []), check=True)
    code = assembly.read_text()
    assert bool(re.search(r"v_div_fixup_f32|v_fma_f32|v_fmac_f32", code)) == (not fast)
    assert not fast or "0x39980e41" in code                 # the float next to 1 / 3448
