"""Divisions of floats by whole numbers known when a definition is compiled (sizes, mostly): the same bits as the division,
for every kind of dividend, except that quotients below the smallest normal number may go to the other of two floats that
lie equally near."""
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("divisor,by_reciprocal", [
    ("3", True), ("7", True), ("10", True), ("1000", True), ("4194303", True), ("(N / N * 36864)", False), ("1.5", False),
    ("1", False), ("2", False), ("1024", False), ("4194305", False), ("(9 * 11)", True), ("99.0", True),
])
def test_quotients_are_those_of_the_division(divisor, by_reciprocal):
    bits = torch.randint(-2**31, 2**31 - 1, (1 << 20,), device="cuda", dtype=torch.int64, generator=torch.Generator(device="cuda").manual_seed(3))
    x = bits.int().view(torch.float32)
    x[:12] = torch.tensor([0.0, -0.0, float("inf"), -float("inf"), float("nan"), 1e-45, -1e-45, 3e-45, 3.4028235e38, -3.4028235e38, 1.1754944e-38, 1.0])
    src = f"def quotient(float(N) A) -> (O) {{ O(n) = A(n) / {divisor} }}"
    ex = tc.compile(src, "quotient", [x], "naive;tile=256;mapToThreads=256;mapToBlocks=65536")
    assert ("/ __tc::Whole<" in ex.compiled_source.split('extern "C"')[-1]) == by_reciprocal
    out = tc.prepare_outputs(src, "quotient", [x])
    tc.run(ex, [x], out)
    c = eval(divisor, {}, {"N": 1})
    got, want = out[0].cpu(), x.cpu() / c
    nan = want.isnan()
    assert torch.equal(got.isnan(), nan)
    same = (got.view(torch.int32) == want.view(torch.int32)) | nan
    exact = x.cpu().double() / c
    tie = (want.abs() < 2.0 ** -126) & ((got.double() - exact).abs() == (want.double() - exact).abs())
    assert bool((same | tie).all())


def test_sizes_divide_by_their_reciprocal():
    src = "def mean(float(M, N) X) -> (mean) { mean(m) +=! X(m, r_n) / N }"
    X = torch.randn(64, 3448, device="cuda")
    ex = tc.compile(src, "mean", [X], "naive;tile=1;mapToThreads=256;mapToBlocks=64;matchLibraryCalls=1")
    assert "/ __tc::Whole<3448>()" in ex.compiled_source
    out = tc.prepare_outputs(src, "mean", [X])
    tc.run(ex, [X], out)
    # (a float sum of n terms is within n * 2^-24 of the sum of their magnitudes)
    assert bool(((out[0].double() - X.double().mean(1)).abs() <= 3448 * 2.0 ** -24 * X.double().abs().mean(1)).all())
