"""Group convolutions on the matrix cores whose channels and windows do not divide into the four lane groups of a wavefront:
surplus steps of the padded quarters, every choice of the divided variable, reductions read in pieces.  Small integers,
every sum exact: results equal torch's."""
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu

GROUP_CONVOLUTION = """
def group_convolution(float(N,G,C,H,W) I, float(G,F,C,KH,KW) W1, float(G,F) B) -> (O) {
    O(n, g, f, h, w) +=! I(n, g, c, h + kh, w + kw) * W1(g, f, c, kh, kw)
    O(n, g, f, h, w) = O(n, g, f, h, w) + B(g, f)
}
"""


def run(n, g, c, f, h, w, kernel, extra="", infinite=False):
    gen = torch.Generator(device="cuda").manual_seed(c * 31 + kernel)
    ints = lambda *shape: torch.randint(-3, 4, shape, generator=gen, device="cuda").float()  # noqa: E731
    ins = [ints(n, g, c, h, w), ints(g, f, c, kernel, kernel), ints(g, f)]
    if infinite:
        ins[0] = ins[0].abs() + 1
        ins[1][0, 0, -1, -1, -1] = float("inf")
    rows, columns = h - kernel + 1, w - kernel + 1
    options = (f"naive;tile=1,1,{f},{rows},{columns};mapToThreads=64,4;mapToBlocks={n},{g};useMfma=1;useSharedMemory=1;"
               f"useReadOnlyCache=1;{extra}")
    print(n, g, c, f, h, w, kernel, extra, flush=True)
    ex = tc.compile(GROUP_CONVOLUTION, "group_convolution", ins, options)
    assert "matrix cores:" in ex.compiled_source
    outs = tc.prepare_outputs(GROUP_CONVOLUTION, "group_convolution", ins)
    outs[0].fill_(float("nan"))
    tc.run(ex, ins, outs)
    want = torch.nn.functional.conv2d(ins[0].double().cpu().reshape(n, g * c, h, w), ins[1].double().cpu().reshape(g * f, c, kernel, kernel),
                                      ins[2].double().cpu().reshape(-1), groups=g).reshape(n, g, f, rows, columns)
    return outs[0].double().cpu(), want


@pytest.mark.parametrize("c", [1, 2, 3, 4, 5, 6, 7, 9, 13, 18, 31])
@pytest.mark.parametrize("kernel", [1, 3, 5])
@pytest.mark.parametrize("f", [5, 17])      # one row of output tiles, whose operand stays in registers where it is short, and two
def test_any_number_of_channels(c, kernel, f):
    got, want = run(2, 3, c, f, 9, 12, kernel)
    assert torch.equal(got, want)


@pytest.mark.parametrize("c,kernel,extra", [
    (45, 5, ""),                            # 300 steps: more than are unrolled
    (13, 3, "useSharedMemory=0"),           # operands from memory
    (7, 5, "useSharedMemory=0"),
    (30, 1, ""), (2, 1, ""),
])
def test_long_and_unstaged_reductions(c, kernel, extra):
    got, want = run(2, 2, c, 6, 8, 11, kernel, extra)
    assert torch.equal(got, want)


@pytest.mark.parametrize("c,kernel", [(5, 3), (6, 5), (7, 3), (13, 5)])
def test_surplus_steps_multiply_zeros(c, kernel):
    """Surplus steps read an element that exists: an infinite weight there must not meet the zero of its partner."""
    got, want = run(2, 2, c, 6, 9, 9, kernel, infinite=True)
    assert torch.equal(got, want) and not bool(got.isnan().any()) and bool(got[:, 0, 1:].isfinite().all())


@pytest.mark.parametrize("m,k,n", [(40, 250, 72), (64, 35, 64), (33, 1030, 40)])
def test_untiled_products(m, k, n):
    gen = torch.Generator(device="cuda").manual_seed(k)
    A, B = (torch.randint(-3, 4, s, generator=gen, device="cuda").float() for s in ((m, k), (k, n)))
    src = "def mm(float(M, K) A, float(K, N) B) -> (O) { O(m, n) +=! A(m, r_k) * B(r_k, n) }"
    for options in ("tile=32,32;mapToThreads=64,4", "tile=32,32;mapToThreads=64,4;useSharedMemory=1", "tile=16,16;mapToThreads=64,8;useSharedMemory=1"):
        ex = tc.compile(src, "mm", [A, B], f"naive;{options};mapToBlocks=64,64;useMfma=1")
        out = tc.prepare_outputs(src, "mm", [A, B])
        tc.run(ex, [A, B], out)
        assert torch.equal(out[0], A @ B)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16])
@pytest.mark.parametrize("c,tile,waves", [(10, 5, 4), (14, 7, 4), (14, 7, 8), (28, 14, 8), (28, 14, 4), (15, 7, 4), (12, 6, 4)])
def test_quarters_of_tiled_reductions(dtype, c, tile, waves):
    """Rectangles of output tiles over reduction tiles of any number of channels, with and without whole points a quarter."""
    gen = torch.Generator(device="cuda").manual_seed(c)
    ins = [torch.randint(-3, 4, s, generator=gen, device="cuda").to(dtype) for s in ((3, c, 13, 19), (96, c, 3, 3))]
    name, load = ("float", "%s") if dtype == torch.float32 else ("float16", "float(%s)")
    src = (f"def conv({name}(N, C, H, W) I, {name}(M, C, KH, KW) W1) -> (O) "
           f"{{ O(n, m, h, w) +=! {load % 'I(n, r_c, h + r_kh, w + r_kw)'} * {load % 'W1(m, r_c, r_kh, r_kw)'} }}")
    print(dtype, c, tile, waves, flush=True)
    want = torch.nn.functional.conv2d(ins[0].double().cpu(), ins[1].double().cpu())
    for prefetch in (0, 1):
        ex = tc.compile(src, "conv", ins, f"naive;tile=1,64,5,0,{tile};mapToThreads=64,{waves};mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;"
                                          f"sharedDepth=7;prefetchShared={prefetch}")
        assert "matrix cores:" in ex.compiled_source
        out = torch.full((3, 96, 11, 17), float("nan"), device="cuda")
        tc.run(ex, ins, [out])
        assert torch.equal(out.double().cpu(), want)
