"""Contractions whose epilogue reads operands per output row (a bias and a scale per filter), on the matrix cores: those
operands come from LDS where a wavefront has several tiles.  Small integers, every sum exact: results equal torch's."""
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu

CONVOLUTION = """
def convolution(float(N, C, H, W) I, float(M, C, KH, KW) W1, float(M) B, float(M) S) -> (O) {
    O(n, m, h, w) +=! I(n, r_c, h + r_kh, w + r_kw) * W1(m, r_c, r_kh, r_kw)
    O(n, m, h, w) = O(n, m, h, w) * S(m) + B(m)
}
"""


@pytest.mark.parametrize("n,c,m,h,w,kernel,tile,threads,blocks,extra", [
    (2, 30, 73, 16, 47, 1, "1,32,16,0,0", "64,8", "256,256,256", ""),                # many tiles a wavefront, last rows partial
    (2, 8, 40, 9, 9, 3, "1,32,7,0,8", "64,8", "256,256,256", "prefetchShared=1"),   # one reduction tile
    (2, 24, 40, 9, 9, 3, "1,32,7,0,8", "64,8", "256,256,256", "prefetchShared=1"),  # reduction tiles, pipelined
    (2, 24, 40, 9, 9, 3, "1,32,7,0,8", "64,8", "256,256,256", ""),                  # and not
    (2, 24, 40, 9, 9, 3, "1,32,7,0,8", "64,8", "256,256,256", "useSharedMemory=0"), # operands from memory: no other barrier
    (3, 24, 40, 9, 9, 3, "1,16,7,0,8", "64,8", "2,1,1", "prefetchShared=1"),        # blocks that loop over their tiles
    (3, 24, 40, 9, 9, 3, "1,32,7,0,0", "64,8", "2,1,1", "useSharedMemory=0"),
    (3, 24, 40, 9, 9, 3, "1,32,7,0,8", "64,8", "2,1,1", "useSharedMemory=0"),
    (2, 64, 24, 6, 6, 3, "1,24,2,0,8", "64,8", "256,256,256", "prefetchShared=1"),  # reduction shared by wavefronts
    (2, 5, 17, 8, 12, 3, "1,17,6,0,0", "64,4", "256,256,256", ""),                  # one row in the second row tile
    (2, 3, 96, 5, 5, 1, "1,96,5,0,0", "64,1", "256,256,256", ""),                   # more rows than threads: read where they lie
])
def test_operands_of_a_row(n, c, m, h, w, kernel, tile, threads, blocks, extra):
    g = torch.Generator(device="cuda").manual_seed(m + c)
    ints = lambda *shape: torch.randint(-3, 4, shape, generator=g, device="cuda").float()  # noqa: E731
    ins = [ints(n, c, h, w), ints(m, c, kernel, kernel), ints(m), ints(m)]
    options = f"naive;tile={tile};mapToThreads={threads};mapToBlocks={blocks};useMfma=1;useSharedMemory=1;{extra}"
    print(n, c, m, h, w, kernel, options, flush=True)
    ex = tc.compile(CONVOLUTION, "convolution", ins, options)
    assert ("__shared__ float rows0_1_[" in ex.compiled_source) == (threads != "64,1")
    outs = tc.prepare_outputs(CONVOLUTION, "convolution", ins)
    outs[0].fill_(float("nan"))
    tc.run(ex, ins, outs)
    want = torch.nn.functional.conv2d(ins[0].double().cpu(), ins[1].double().cpu())
    want = want * ins[3].double().cpu()[:, None, None] + ins[2].double().cpu()[:, None, None]
    assert torch.equal(outs[0].double().cpu(), want)
