"""Contiguous views that start off the boundaries of vectors: one element into an allocation, inputs
and results."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc
from tests import benchmark_tcs as B

pytestmark = pytest.mark.gpu

MATRIX = "mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"


def offset(array, elements):
    flat = torch.zeros(array.size + elements, dtype=torch.from_numpy(array).dtype, device="cuda")
    view = flat[elements:].view(array.shape)
    view.copy_(torch.from_numpy(array))
    return view


def ints(shape, seed, dtype):
    return np.random.Generator(np.random.Philox(seed)).integers(-4, 5, size=shape).astype(dtype)


@pytest.mark.parametrize("elements", [1, 3])
@pytest.mark.parametrize("half,tile", [(False, "64,64,32"), (False, "16,32,128"), (True, "64,64,32"), (True, "64,64,64")])
@pytest.mark.parametrize("m,k,n", [(128, 160, 128), (130, 131, 67)])
def test_products_of_offset_views(m, k, n, half, tile, elements):
    dtype = np.float16 if half else np.float32
    A, Bm = ints((m, k), 1, dtype), ints((k, n), 2, dtype)
    want = A.astype(np.float32) @ Bm.astype(np.float32)
    for src, entry, second in ((B.HALF_MATMUL, "half_matmul", Bm), (B.HALF_TMM, "half_tmm", Bm.T)) if half else (
            (B.MATMUL, "matmul", Bm), (B.TMM, "tmm", Bm.T)):
        print(f"{entry} {m}x{k}x{n} tile={tile} offset={elements}", flush=True)
        ins = [offset(A, elements), offset(np.ascontiguousarray(second), elements)]
        out = offset(np.full((m, n), np.nan, np.float32), elements)
        tc.run(tc.compile(src, entry, ins, f"naive;tile={tile};{MATRIX}"), ins, [out])
        torch.cuda.synchronize()
        assert np.array_equal(out.cpu().numpy(), want)


@pytest.mark.parametrize("dtype,tcname", [(np.float32, "float"), (np.float16, "float16"), (np.float64, "double"), (np.int8, "int8")])
@pytest.mark.parametrize("shape", [(3, 5), (64, 1025), (512, 1000)])
def test_streams_of_offset_views(shape, dtype, tcname):
    print(f"stream {shape} {tcname}", flush=True)
    src = f"def f({tcname}(N, M) A, {tcname}(N, M) B) -> (O) {{ O(n, m) = A(n, m) + B(n, m) }}"
    A, Bm = ints(shape, 3, dtype), ints(shape, 4, dtype)
    ins, out = [offset(A, 1), offset(Bm, 3)], offset(np.full(shape, 77, dtype), 1)
    tc.run(tc.compile(src, "f", ins, "naive"), ins, [out])
    torch.cuda.synchronize()
    assert np.array_equal(out.cpu().numpy(), A + Bm)
