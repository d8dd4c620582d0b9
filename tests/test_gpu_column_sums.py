"""Sums of the columns of a matrix under tiles that leave most of the device out (__tc::columnSums): columns and rows around
what a block and a turn take."""
import pytest
import torch

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

SOURCE = "def f(float(R, N) A) -> (O) { O(n) +=! A(r_r, n) }"
OPTIONS = "naive;tile=64;mapToThreads=64;mapToBlocks=256;unroll=32"


@pytest.mark.gpu
@pytest.mark.parametrize("rows,columns", [(64, 1), (64, 16), (65, 17), (127, 100), (128, 1024), (1000, 15), (1024, 4096), (1025, 33), (5000, 163)])
def test_column_sums(rows, columns):
    print(rows, columns, flush=True)
    g = torch.Generator(device="cuda").manual_seed(rows)
    whole = torch.randint(-100, 101, (rows, columns), generator=g, device="cuda").float()
    a = torch.randn(rows, columns, generator=g, device="cuda")
    executor = tc.compile(SOURCE, "f", [a], OPTIONS)
    assert "__tc::columnSums<" in executor.compiled_source.split('extern "C"')[-1]
    out = torch.full((columns,), float("nan"), device="cuda")
    tc.run(executor, [whole], [out])
    assert torch.equal(out, whole.sum(0))                       # (sums of whole numbers are exact)
    tc.run(executor, [a], [out])
    # one rounding a term, in whatever order
    assert ((out - a.double().sum(0)).abs() <= rows * 2.0 ** -24 * a.double().abs().sum(0)).all()
    a[rows - 1, columns - 1] = float("inf")                     # belongs to its column alone
    tc.run(executor, [a], [out])
    assert out[-1] == float("inf") and torch.isfinite(out[:-1]).all()


@pytest.mark.parametrize("source,rows,columns,options,taken", [
    (SOURCE, 63, 1024, OPTIONS, False),                                             # too few rows for the wavefronts
    (SOURCE, 1024, 100000, OPTIONS, False),                                         # columns enough
    (SOURCE, 1024, 1024, OPTIONS + ";matchLibraryCalls=1", False),
    (SOURCE, 1024, 1024, OPTIONS.replace("mapToThreads=64", "mapToThreads=64,4"), False),
    (SOURCE, 1024, 1024, OPTIONS.replace("mapToBlocks=256", "mapToBlocks=2"), False),   # fewer blocks than tiles
    (SOURCE.replace("A(r_r, n) }", "A(r_r, n) * A(r_r, n) }"), 1024, 1024, OPTIONS, False),
    (SOURCE.replace("+=!", "+="), 1024, 1024, OPTIONS, False),
    (SOURCE.replace("+=!", "max=!"), 1024, 1024, OPTIONS, False),
    (SOURCE, 1024, 1024, OPTIONS + ";maxSharedMemory=4095", False),                 # the partial sums take 4 KiB of LDS
    (SOURCE, 1024, 1024, OPTIONS + ";maxSharedMemory=4096", True),
    (SOURCE, 1024, 1024, OPTIONS, True),
    (SOURCE, 64, 8192, OPTIONS, True),
    (SOURCE, 64, 8256, OPTIONS, False),                                             # few rows beside columns on more than half of the compute units
    (SOURCE, 80, 8257, OPTIONS, True),
    (SOURCE, 200, 14336, OPTIONS, True),
    (SOURCE, 320, 14336, OPTIONS, False),                                           # lines read twice, from beyond the L2 caches
    (SOURCE, 512, 12288, OPTIONS, False),
    (SOURCE, 1024, 9216, OPTIONS, True),
    (SOURCE, 200, 15001, OPTIONS, True),
    (SOURCE, 200, 16001, OPTIONS, False),
])
def test_which_sums_are_taken(source, rows, columns, options, taken):
    text, _ = tc.map_only(source, "f", [ShapeOnly((rows, columns))], options)
    assert ("__tc::columnSums<" in text.split('extern "C"')[-1]) == taken
