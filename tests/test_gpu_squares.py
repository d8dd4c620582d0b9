"""Sums of squares, staged in LDS or read by the threads themselves: exact on small integers."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 4096), (64, 4100), (33, 2000), (128, 1000), (3, 70)])
@pytest.mark.parametrize("options", ["tile=1,0;mapToThreads=256;matchLibraryCalls=1", "tile=1,0;mapToThreads=64;matchLibraryCalls=1;vectorWidth=4",
                                     "tile=32,32;mapToThreads=32", "tile=1,0;mapToThreads=128;matchLibraryCalls=1;usePrivateMemory=1;unroll=64"])
def test_sums_of_squares_are_exact(shape, options):
    A = np.random.Generator(np.random.Philox(sum(shape))).integers(-4, 5, size=shape).astype(np.float32)
    I = torch.from_numpy(A).cuda()
    for src, want in (("def f(float(N, K) I) -> (s) { s(n) +=! I(n, k) * I(n, k) }", [(A * A).sum(1)]),
                      ("def f(float(N, K) I) -> (s) { s(k) +=! I(n, k) * I(n, k) }", [(A * A).sum(0)]),
                      ("def f(float(N, K) I) -> (t, s) { t(n) +=! I(n, k) s(n) +=! I(n, k) * I(n, k) }", [A.sum(1), (A * A).sum(1)])):
        print(f"squares {shape} {options} {src[24:]}", flush=True)
        ex = tc.compile(src, "f", [I], f"naive;outerScheduleFusionStrategy=Max;{options};mapToBlocks=4096;useSharedMemory=1")
        outs = tc.prepare_outputs(src, "f", [I])
        tc.run(ex, [I], outs)
        torch.cuda.synchronize()
        for o, w in zip(outs, want):
            assert np.array_equal(o.cpu().numpy(), w)
