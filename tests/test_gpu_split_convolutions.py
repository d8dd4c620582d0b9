"""Convolutions on the bf16 matrix instruction, each float in three parts (__tc::SplitConvolution): against the same sums in
64 bits at the edges of pixel tiles, filter tiles, channel chunks and windows, and for values the parts cannot hold."""
import os
import re
import subprocess

import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

HIPCC = "/opt/rocm/bin/hipcc"
DENSE = """
def f(float(N, C, H, W) I, float(M, C, KH, KW) W1, float(M) B) -> (O) {
    O(n, m, h, w) +=! I(n, r_c, h + r_kh, w + r_kw) * W1(m, r_c, r_kh, r_kw)
    O(n, m, h, w) = O(n, m, h, w) + B(m)
}
"""
GROUPS = """
def f(float(N, G, C, H, W) I, float(G, F, C, KH, KW) W1, float(G, F) B) -> (O) {
    O(n, g, f, h, w) +=! W1(g, f, r_c, r_kh, r_kw) * I(n, g, r_c, h + r_kh, w + r_kw)
    O(n, g, f, h, w) = B(g, f) + O(n, g, f, h, w)
}
"""
PLAIN = """
def f(float(N, G, C, H, W) I, float(G, F, C, KH, KW) W1) -> (O) {
    O(n, g, f, h, w) +=! I(n, g, r_c, h + r_kh, w + r_kw) * W1(g, f, r_c, r_kh, r_kw)
}
"""
SIZES = [
    # n, g, channels, filters, h, w, kernel
    (16, 1, 64, 64, 57, 57, (3, 3)),     # four chunks, a last band of 17 pixels
    (24, 1, 53, 41, 12, 7, (3, 3)),      # five pixels a row, 50 of them
    (28, 1, 93, 23, 9, 11, (3, 3)),      # a plane of 63 pixels
    (21, 1, 111, 119, 17, 17, (1, 1)),   # no window
    (28, 1, 65, 38, 43, 29, (3, 3)),     # one channel more than eight octets
    (9, 11, 6, 29, 19, 29, (3, 3)),      # a chunk that is not full, 13 filters in the last tile
    (4, 4, 7, 13, 28, 30, (5, 5)),       # 25 places: one slot of the last step
    (2, 8, 15, 4, 25, 28, (3, 3)),
    (3, 5, 17, 20, 22, 26, (5, 3)),      # a window that is no square
]


def options(kernel, sizes):
    n, g, c, f, h, w, _ = sizes
    rows, columns = h - kernel[0] + 1, w - kernel[1] + 1
    if g == 1:
        band = max(d for d in range(1, 17) if rows % d == 0)
        return (f"naive;tile=1,32,{band},0,8;mapToThreads=64,8;mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;"
                "useReadOnlyCache=1;sharedDepth=7;prefetchShared=1")
    return f"naive;tile=1,1,{f},{rows},{columns};mapToThreads=64,4;mapToBlocks={n},{g};useMfma=1;useSharedMemory=1;useReadOnlyCache=1"


def operands(sizes, make):
    n, g, c, f, h, w, (kh, kw) = sizes
    if g == 1:
        return [make(n, c, h, w), make(f, c, kh, kw), make(f)]
    return [make(n, g, c, h, w), make(g, f, c, kh, kw), make(g, f)]


def run(source, sizes, ins):
    text, _ = tc.map_only(source, "f", [ShapeOnly(tuple(t.shape)) for t in ins], options(sizes[6], sizes))
    assert "__tc::SplitConvolution<" in text
    device = [t.cuda() for t in ins]
    executor = tc.compile(source, "f", device, options(sizes[6], sizes))
    outs = tc.prepare_outputs(source, "f", device)
    outs[0].fill_(float("nan"))
    tc.run(executor, device, outs)
    return outs[0].cpu()


def reference(sizes, ins):
    n, g, c, f, h, w, (kh, kw) = sizes
    x, weights = ins[0].double().reshape(n, g * c, h, w), ins[1].double().reshape(g * f, c, kh, kw)
    bias = ins[2].double().reshape(-1) if len(ins) > 2 else None
    sums = torch.nn.functional.conv2d(x, weights, None, groups=g)
    magnitudes = torch.nn.functional.conv2d(x.abs(), weights.abs(), None, groups=g)
    if bias is not None:
        sums, magnitudes = sums + bias.view(1, -1, 1, 1), magnitudes + bias.abs().view(1, -1, 1, 1)
    return sums, magnitudes


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "x".join(map(str, s[:6])))
def test_sums(sizes):
    print(sizes, flush=True)
    source = DENSE if sizes[1] == 1 else GROUPS
    generator = torch.Generator().manual_seed(1)
    whole = operands(sizes, lambda *s: torch.randint(-8, 9, s, generator=generator).float())
    got = run(source, sizes, whole)
    assert torch.equal(got.reshape(-1).double(), reference(sizes, whole)[0].reshape(-1))   # (sums of whole numbers are exact)
    ins = operands(sizes, lambda *s: torch.randn(s, generator=generator))
    got = run(source, sizes, ins).double()
    want, magnitudes = reference(sizes, ins)
    # one rounding of 2^-24 a term and the bias, in whatever order, and up to 2^-24 of every product for the parts left out
    terms = sizes[2] * sizes[6][0] * sizes[6][1]
    assert ((got.reshape(want.shape) - want).abs() <= (terms + 2) * 2.0 ** -24 * magnitudes).all()
    # Roundings do not add up like that: 0.5e-7 to 1.7e-7 here.  Without any one of the six products of parts it is 2.4e-6 or more.
    assert (got.reshape(want.shape) - want).norm() <= 1e-6 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "x".join(map(str, s[:6])))
def test_every_product_of_parts(sizes):
    """Sums of 24 bits, which are exact only with all six products of parts: values 1 + y 2^-9 + z 2^-18 (y, z of -1, 0, 1) in a few channels and places."""
    source = DENSE if sizes[1] == 1 else GROUPS
    generator = torch.Generator().manual_seed(sizes[2])
    signs = lambda *s: torch.randint(-1, 2, s, generator=generator).float()  # noqa: E731
    x, weights, bias = operands(sizes, signs)
    places = torch.zeros(weights[0].numel() if sizes[1] == 1 else weights[0, 0].numel())
    places[torch.randperm(places.numel(), generator=generator)[:24]] = 1.0
    weights, bias = weights * places.view(weights.shape[-3:]), 0 * bias
    middle = lambda t: t * (1 + signs(*t.shape) * 2.0 ** -9)  # noqa: E731
    low = lambda t: t * (1 + signs(*t.shape) * 2.0 ** -9 + signs(*t.shape) * 2.0 ** -18)  # noqa: E731
    for ins in ([low(x), weights, bias], [x, low(weights), bias], [middle(x), middle(weights), bias]):
        assert torch.equal(run(source, sizes, ins).reshape(-1).double(), reference(sizes, ins)[0].reshape(-1))


@pytest.mark.gpu
def test_without_a_bias():
    sizes = next(s for s in SIZES if s[:3] == (9, 11, 6))
    ins = operands(sizes, lambda *s: torch.randint(-8, 9, s).float())[:2]
    assert torch.equal(run(PLAIN, sizes, ins).reshape(-1).double(), reference(sizes, ins)[0].reshape(-1))


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["infinity", "nan", "rounds to infinity", "small", "denormal", "large sums"])
def test_values_the_parts_cannot_hold(case):
    sizes = next(s for s in SIZES if s[:3] == (2, 8, 15))
    generator = torch.Generator().manual_seed(2)
    x, weights, bias = operands(sizes, lambda *s: torch.randn(s, generator=generator))
    flat = x.view(-1)
    if case == "infinity":
        flat[[5, 4711, -1]] = torch.tensor([np.inf, -np.inf, np.inf])
    elif case == "nan":
        flat[[5, 4711]] = np.nan
    elif case == "rounds to infinity":
        flat[::1001] = 3.4e38                   # its nearest bf16 is infinite
        weights *= 2.0 ** -20
    elif case == "small":
        flat[:] *= 2.0 ** -110                  # their low parts would be denormal
        bias[:] = 0
    elif case == "denormal":
        flat[: flat.numel() // 2] *= 2.0 ** -130
        bias[:] = 0
    else:
        flat[:] *= 2.0 ** 100
        weights *= 2.0 ** 30                    # sums beyond the largest float
    got = run(GROUPS, sizes, [x, weights, bias]).double()
    want, magnitudes = reference(sizes, [x, weights, bias])
    got, want = got.reshape(-1), want.float().double().reshape(-1)   # (the float nearest to the sum: infinite beyond the largest)
    finite = torch.isfinite(want) & (magnitudes.reshape(-1) < 3.4e38)
    terms = sizes[2] * 9
    # (a denormal sum is a whole number of 2^-149)
    assert ((got - want).abs()[finite] <= (terms + 2) * (2.0 ** -24 * magnitudes.reshape(-1)[finite] + 2.0 ** -149)).all()
    if case in ("infinity", "nan"):
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(torch.isinf(got), torch.isinf(want))
        assert torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["denormal image", "denormal rows", "denormal filters", "denormal terms", "zero image"])
def test_small_values_beside_others(case):
    """Values below what the parts hold, beside ordinary ones and times large ones."""
    sizes = next(s for s in SIZES if s[:3] == (2, 8, 15))
    generator = torch.Generator().manual_seed(3)
    x, weights, bias = operands(sizes, lambda *s: torch.randn(s, generator=generator))
    bias[:] = 0
    if case == "denormal image":
        x[0] *= 2.0 ** -140
        weights *= 2.0 ** 29
    elif case == "denormal rows":
        x[:, :, :, 3:9] *= 2.0 ** -140
        weights *= 2.0 ** 29
    elif case == "denormal filters":
        weights[:, 1] *= 2.0 ** -139
        x *= 2.0 ** 28
    elif case == "denormal terms":                # ordinary weights meet zeros: the sum is one of the others
        weights[:, :, :5] *= 2.0 ** -140
        x[:, :, 5:] = 0
        x *= 2.0 ** 28
    else:
        x[1] = 0
    got = run(GROUPS, sizes, [x, weights, bias]).double()
    want, magnitudes = reference(sizes, [x, weights, bias])
    got = got.reshape(want.shape)
    terms = sizes[2] * 9
    # (a denormal sum is a whole number of 2^-149)
    assert ((got - want).abs() <= (terms + 2) * (2.0 ** -24 * magnitudes + 2.0 ** -149)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", SIZES, ids=lambda s: "x".join(map(str, s[:6])))
def test_sums_of_floats_themselves(sizes):
    """Blocks that compute again: infinities and NaNs at the corners of an image reach the windows they are in and no other, whatever the weights of
    steps and channels that do not exist, and denormal images keep their sums."""
    source = DENSE if sizes[1] == 1 else GROUPS
    generator = torch.Generator().manual_seed(4)
    x, weights, bias = operands(sizes, lambda *s: torch.randn(s, generator=generator))
    terms = sizes[2] * sizes[6][0] * sizes[6][1]
    corners = x.clone()
    flat = corners.view(sizes[0] * sizes[1], sizes[2], sizes[4], sizes[5])
    flat[0, 0, 0, 0], flat[0, -1, -1, -1], flat[-1, -1, 0, -1], flat[-1, 0, -1, 0] = np.inf, -np.inf, np.nan, np.inf
    for ins in ([corners, weights, bias], [x * 2.0 ** -125, weights, 0 * bias]):
        got = run(source, sizes, ins).double()
        want, magnitudes = reference(sizes, ins)
        got = got.reshape(want.shape)
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
        finite = torch.isfinite(want)
        # (a denormal sum is a whole number of 2^-149)
        assert ((got - want).abs()[finite] <= (terms + 2) * (2.0 ** -24 * magnitudes[finite] + 2.0 ** -149)).all()


@pytest.mark.gpu
def test_time_of_sums_of_floats_themselves():
    """A block that computes again uses the matrix cores too: one infinity makes a convolution take some 2.1 times as long (without them 62 times)."""
    sizes = SIZES[0]
    ins = [t.cuda() for t in operands(sizes, lambda *s: torch.randn(s))]
    executor = tc.compile(DENSE, "f", ins, options(sizes[6], sizes))
    outs = tc.prepare_outputs(DENSE, "f", ins)
    times = []
    for value in (1.0, float("inf")):
        ins[0][3, 5, 7, 9] = value
        tc.run(executor, ins, outs)
        times.append(min(tc.profile_repeated(executor, ins, outs, 20) for _ in range(5)))
    assert times[1] < 8 * times[0]


# (in 80 drawn dense convolutions taken with less of a margin these took up to 1.3 times as long as in the general pipeline)
@pytest.mark.parametrize("sizes,taken", [((27, 1, 8, 28, 46, 59, (3, 3)), False), ((30, 1, 10, 73, 39, 47, (3, 3)), False), ((12, 1, 60, 60, 43, 22, (1, 1)), False),
                                         ((16, 1, 96, 110, 35, 9, (3, 3)), False), ((16, 1, 64, 64, 57, 57, (3, 3)), True), ((2, 8, 15, 4, 25, 28, (3, 3)), True)])
def test_which_convolutions_are_taken(sizes, taken):
    ins = operands(sizes, lambda *s: ShapeOnly(s))
    text, _ = tc.map_only(DENSE if sizes[1] == 1 else GROUPS, "f", ins, options(sizes[6], sizes))
    assert ("__tc::SplitConvolution<" in text.split('extern "C"')[-1]) == taken


@pytest.mark.parametrize("sizes", [(16, 1, 79, 117, 23, 41, (3, 3)), (23, 1, 126, 64, 83, 19, (3, 3)), (9, 16, 54, 50, 64, 10, (3, 3)), (8, 1, 120, 73, 61, 35, (3, 3))],
                         ids=lambda s: "x".join(map(str, s[:6])))
def test_all_of_the_shared_memory(sizes):
    """Blocks whose parts take all but 16 to 256 bytes of a compute unit's LDS: what else the kernel declares has to fit there too."""
    source, ins = DENSE if sizes[1] == 1 else GROUPS, operands(sizes, lambda *s: ShapeOnly(s))
    assert tc.compile(source, "f", ins, options(sizes[6], sizes)).lds_bytes() <= 160 * 1024


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="no hipcc")
@pytest.mark.parametrize("kernel", ["convolution", "product"])
def test_no_other_shared_memory_than_the_options_see(tmp_path, kernel):
    if kernel == "convolution":
        sizes = SIZES[0]
        source, ins, opts = DENSE, operands(sizes, lambda *s: ShapeOnly(s)), options(sizes[6], sizes)
    else:
        source, ins = "def f(float(M, K) A, float(K, N) B) -> (O) { O(m, n) +=! A(m, r_k) * B(r_k, n) }", [ShapeOnly((1000, 1000))] * 2
        opts = "naive;tile=64,64,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"
    text, _ = tc.map_only(source, "f", ins, opts)
    declared = int(re.search(r"char (?:window|sums)_\[(\d+)\]", text).group(1))
    path, assembly = tmp_path / "f.hip", tmp_path / "f.s"
    path.write_text(text)
    subprocess.run([HIPCC, "-x", "hip", "--offload-arch=gfx950", "--offload-device-only", "-O3", "-std=c++17", "-Xclang", "-target-feature",
                    "-Xclang", "-packed-fp32-ops", "-include", "hip/hip_runtime.h", "-w", "-S", "-o", str(assembly), str(path)], check=True)
    assert int(re.search(r"amdhsa_group_segment_fixed_size (\d+)", assembly.read_text()).group(1)) == declared


@pytest.mark.parametrize("height,taken", [(1 << 18, True), (1 << 18 | 1 << 11, False)])
def test_offsets_of_channels_that_do_not_exist(height, taken):
    """Eight channels to a chunk: with five of them the offsets of the others stay below 2^31 bytes too."""
    sizes = (1, 1, 5, 7, height, 255, (5, 5))
    ins = operands(sizes, lambda *s: ShapeOnly(s))
    text, _ = tc.map_only(DENSE, "f", ins, "naive;tile=1,16,1,16;mapToThreads=64,8;mapToBlocks=1000000,1000000,1000000;useMfma=1;useSharedMemory=1;useReadOnlyCache=1")
    assert ("__tc::SplitConvolution<" in text.split('extern "C"')[-1]) == taken
