"""Products of float16 matrices in blocks of 256 x 256 outputs (__tc::largeHalfProduct): every order of the two
operands, last blocks and reduction tiles that are partial, odd and even numbers of reduction tiles, operands that
start off vector boundaries.  Small integers: every sum is exact, so results equal the float32 product in every bit."""
import pytest
import torch

import tensorcomprehensions_amd as tc

pytestmark = pytest.mark.gpu

# (given tiles of the same size: the mapper takes the large blocks wherever they are allowed)
OPTIONS = "naive;tile=256,256,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"


def source(a_transposed, b_transposed):
    a = ("K, M", "r_k, m") if a_transposed else ("M, K", "m, r_k")
    b = ("N, K", "n, r_k") if b_transposed else ("K, N", "r_k, n")
    return (f"def product(float16({a[0]}) A, float16({b[0]}) B) -> (O) "
            f"{{ O(m, n) +=! float(A({a[1]})) * float(B({b[1]})) }}")


def ints(shape, seed, offset=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    n = shape[0] * shape[1]
    return torch.randint(-4, 5, (n + offset,), generator=g, device="cuda").half()[offset:].view(shape)


@pytest.mark.parametrize("a_transposed", [False, True])
@pytest.mark.parametrize("b_transposed", [False, True])
@pytest.mark.parametrize("m,n,k,offsets", [
    (512, 512, 256, (0, 0)),        # whole blocks, four reduction tiles
    (256, 768, 320, (0, 0)),        # five
    (264, 248, 264, (0, 0)),        # one row of vectors more and less than a block, eight points in the last tile
    (504, 520, 312, (0, 0)),        # 56 points in it
    (2304, 2312, 328, (0, 0)),      # more than one stripe of block columns, blocks that do not divide by eight
    (520, 512, 392, (8, 0)),        # a view that starts on a vector
    (512, 264, 264, (1, 0)),        # and views that start inside one
    (264, 512, 320, (0, 3)),
    (504, 504, 328, (2, 1)),
])
def test_products_are_exact(a_transposed, b_transposed, m, n, k, offsets):
    A = ints((k, m) if a_transposed else (m, k), 1, offsets[0])
    B = ints((n, k) if b_transposed else (k, n), 2, offsets[1])
    print(f"{m}x{n}x{k} {a_transposed} {b_transposed} {offsets}", flush=True)
    ex = tc.compile(source(a_transposed, b_transposed), "product", [A, B], OPTIONS)
    assert "__tc::largeHalfProduct<" in ex.compiled_source.split('extern "C"')[-1]
    out = torch.full((m, n), float("nan"), device="cuda")
    tc.run(ex, [A, B], [out])
    want = (A.float().t() if a_transposed else A.float()) @ (B.float().t() if b_transposed else B.float())
    assert torch.equal(out, want)


@pytest.mark.parametrize("offsets", [(0, 0), (1, 3)])
@pytest.mark.parametrize("k", [257, 259, 260, 321])
def test_last_reduction_tiles_of_a_few_rows(k, offsets):
    """The reduction outermost in both operands may have any number of points: pieces of the last tile without a row."""
    A, B = ints((k, 264), 8, offsets[0]), ints((k, 256), 9, offsets[1])
    print(k, offsets, flush=True)
    ex = tc.compile(source(True, False), "product", [A, B], OPTIONS)
    assert "__tc::largeHalfProduct<" in ex.compiled_source.split('extern "C"')[-1]
    out = tc.prepare_outputs(source(True, False), "product", [A, B])
    tc.run(ex, [A, B], out)
    assert torch.equal(out[0], A.float().t() @ B.float())


@pytest.mark.parametrize("m,n,k", [(257, 511, 264), (510, 259, 320)])
def test_outputs_of_any_size(m, n, k):
    """Rows and columns need be no multiples of anything where the reduction is innermost in both operands."""
    A, B = ints((m, k), 3), ints((n, k), 4)
    ex = tc.compile(source(False, True), "product", [A, B], OPTIONS)
    assert "__tc::largeHalfProduct<" in ex.compiled_source.split('extern "C"')[-1]
    guarded = torch.full((m + 2, n), float("nan"), device="cuda")   # what lies behind the result stays
    out = guarded[:m]
    tc.run(ex, [A, B], [out])
    assert torch.equal(out, A.float() @ B.float().t()) and bool(guarded[m:].isnan().all())


def test_surplus_points_meet_zeros():
    """Points past the end of the reduction belong to the next row: infinities there stay out of the sums."""
    A, B = ints((256, 264), 5), ints((256, 264), 6)
    A[1::2], B[1::2] = float("inf"), float("inf")
    ex = tc.compile(source(False, True), "product", [A, B], OPTIONS)
    out = tc.prepare_outputs(source(False, True), "product", [A, B])
    tc.run(ex, [A, B], out)
    assert torch.equal(out[0][::2, ::2], A[::2].float() @ B[::2].float().t())


def test_errors_on_deviates_are_those_of_float_sums():
    """A sum of k products in float, in any order of its partial sums, is within k * 2^-24 of the sum of their
    magnitudes (first order); deviates come nowhere near it."""
    g = torch.Generator(device="cuda").manual_seed(7)
    A, B = (torch.randn((512, 1024), generator=g, device="cuda").half() for _ in range(2))
    ex = tc.compile(source(False, True), "product", [A, B], OPTIONS)
    out = tc.prepare_outputs(source(False, True), "product", [A, B])
    tc.run(ex, [A, B], out)
    exact = A.double().cpu() @ B.double().cpu().t()
    bound = 1024 * 2.0 ** -24 * (A.double().abs().cpu() @ B.double().abs().cpu().t())
    assert bool(((out[0].double().cpu() - exact).abs() <= bound).all())
