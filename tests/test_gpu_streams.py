"""Point-wise definitions whose dimensions merge into one stream, under options that address two or
three loops: every element written once, at extents around the lane groups and the block."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,tcname", [(np.float32, "float"), (np.float64, "double"), (np.int32, "int32"), (np.int8, "int8")])
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (1, 255), (2, 128), (257, 4), (7, 11, 13), (33, 31, 2, 5), (64, 63, 17)])
@pytest.mark.parametrize("options", ["naive", "pointwise"])
def test_merged_streams_write_every_element(shape, dtype, tcname, options):
    print(f"stream {shape} {tcname} {options}", flush=True)
    dims = ", ".join("NCHW"[i] for i in range(len(shape)))
    subs = ", ".join("nchw"[i] for i in range(len(shape)))
    src = f"def f({tcname}({dims}) A, {tcname}({dims}) B) -> (O) {{ O({subs}) = A({subs}) + B({subs}) }}"
    rng = np.random.Generator(np.random.Philox(sum(shape)))
    A, B = (rng.integers(-50, 51, size=shape).astype(dtype) for _ in range(2))
    ins = [torch.from_numpy(x).cuda() for x in (A, B)]
    ex = tc.compile(src, "f", ins, options)
    (O,) = tc.prepare_outputs(src, "f", ins)
    O.fill_(77)
    tc.run(ex, ins, [O])
    torch.cuda.synchronize()
    assert np.array_equal(O.cpu().numpy(), A + B)


@pytest.mark.parametrize("dtype,tcname", [(np.float32, "float"), (np.float16, "float16"), (np.float64, "double"), (np.int8, "int8")])
@pytest.mark.parametrize("shape", [(3, 5), (64, 1025), (512, 1000)])
@pytest.mark.parametrize("threads", ["256,8", "16,15", "64,64"])
def test_streams_under_nominal_blocks(shape, threads, dtype, tcname):
    print(f"stream {shape} {tcname} threads={threads}", flush=True)
    src = f"def f({tcname}(N, M) A, {tcname}(N, M) B) -> (O) {{ O(n, m) = A(n, m) + B(n, m) }}"
    rng = np.random.Generator(np.random.Philox(sum(shape)))
    A, B = (rng.integers(-50, 51, size=shape).astype(dtype) for _ in range(2))
    ins = [torch.from_numpy(x).cuda() for x in (A, B)]
    ex = tc.compile(src, "f", ins, f"naive;tile=32,32;mapToThreads={threads};mapToBlocks=256,256")
    (O,) = tc.prepare_outputs(src, "f", ins)
    O.fill_(77)
    tc.run(ex, ins, [O])
    torch.cuda.synchronize()
    assert np.array_equal(O.cpu().numpy(), A + B)
