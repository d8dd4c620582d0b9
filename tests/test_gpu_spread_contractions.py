"""Contractions in registers whose tiles were made for other sizes: points of the innermost variable on a block axis of
their own, halved tiles, variables folded into the register tile, at remainders of every one of them."""
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu

STREAM = "naive;tile=1,8,2,0;mapToThreads=256;mapToBlocks=32,64;unroll=128;vectorWidth=4;useReadOnlyCache=1"
HEAD = "def f(float(N, C1, C2, H, W) A, float(N, C2, C3, H, W) B) -> (O) { O(n, c1, c3, h, w) %s A(n, c1, r_c2, h, w) %s B(n, r_c2, c3, h, w) %s }"


@pytest.mark.parametrize("changes", ["", "mapToThreads=64", "mapToBlocks=4,3", "mapToBlocks=7,7,7", "unroll=8", "vectorWidth=1"])
@pytest.mark.parametrize("sizes", [
    (1, 1, 2, 1, 7, 7), (1, 93, 3, 3, 25, 25), (4, 17, 8, 4, 47, 25), (2, 9, 5, 3, 16, 16), (3, 7, 2, 4, 33, 31), (1, 8, 3, 3, 1, 257), (2, 64, 16, 1, 40, 36),
])
@pytest.mark.parametrize("op,join,then", [("+=!", "*", ""), ("+=", "*", "O(n, c1, c3, h, w) = fmax(O(n, c1, c3, h, w), 0)"), ("max=!", "+", "")])
def test_against_float64(sizes, changes, op, join, then):
    n, c1, c2, c3, h, w = sizes
    generator = torch.Generator(device="cuda").manual_seed(n * 1000 + c1 + h)
    a = torch.randn((n, c1, c2, h, w), device="cuda", generator=generator)
    b = torch.randn((n, c2, c3, h, w), device="cuda", generator=generator)
    src = HEAD % (op, join, then)
    ex = tc.compile(src, "f", [a, b], tc.MappingOptions(f"{STREAM};{changes}"))
    outs = tc.prepare_outputs(src, "f", [a, b])
    outs[0].fill_(0.5)
    tc.run(ex, [a, b], outs)
    left, right = a.double()[:, :, :, None], b.double().permute(0, 2, 1, 3, 4)[:, None].permute(0, 1, 3, 2, 4, 5)
    if join == "*":
        terms = left * right
        expected = terms.sum(2)
        magnitude = terms.abs().sum(2) + 0.5
        if op == "+=":
            expected = (expected + 0.5).clamp(min=0)
        # c2 products and sums, each rounded once
        assert bool(((outs[0].double() - expected).abs() <= (c2 + 2) * 2.0 ** -24 * magnitude).all())
    else:
        # one rounded sum a term; rounding keeps the order
        assert torch.equal(outs[0], (left + right).amax(2).float())


@pytest.mark.parametrize("sizes,changes", [
    ((2, 8, 2, 4, 30, 56), "tile=1,8,4,0;mapToBlocks=32,64,8"),     # axes that a halved tile would have taken from the rows' pieces,
    ((3, 7, 5, 79, 14, 13), ""),                                     # from c3,
    ((3, 11, 4, 4, 6, 11), "tile=4,1,1,0;mapToBlocks=200,200"),      # and from c3 by way of c1
    ((2, 8, 2, 3, 31, 56), ""),                                      # c3 taken whole when c1 takes its axis
])
def test_axes_stay_with_their_variables(sizes, changes):
    test_against_float64(sizes, changes, "+=!", "*", "")
