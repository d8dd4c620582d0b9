"""Products of float matrices whose wavefronts divide the reduction, each float in three bf16 parts (__tc::SlicedProduct): every order
of the two operands against the same sums in 64 bits, at sizes around the tiles and steps, and for values the parts cannot hold."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly


def source(a_inner, b_inner, bias=False):
    a = ("M, K", "m, r_k") if a_inner else ("K, M", "r_k, m")
    b = ("N, K", "n, r_k") if b_inner else ("K, N", "r_k, n")
    return (f"def f(float({a[0]}) A, float({b[0]}) B{', float(N) C' if bias else ''}) -> (O) {{ O(m, n) +=! A({a[1]}) * B({b[1]})"
            + (" O(m, n) = O(m, n) + C(n) }" if bias else " }"))


def options(m, n):
    tile = "16,32,128" if m * n <= 1 << 18 else "64,64,32" if m * n <= 1 << 21 else "128,128,16"
    return f"naive;tile={tile};mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"


def run(m, n, k, a_inner, b_inner, a, b, bias=None):
    text = source(a_inner, b_inner, bias is not None)
    ins = [(a if a_inner else a.t()).contiguous().cuda(), (b if b_inner else b.t()).contiguous().cuda()] + ([] if bias is None else [bias.cuda()])
    executor = tc.compile(text, "f", ins, options(m, n))
    assert "__tc::SlicedProduct<" in executor.compiled_source.split('extern "C"')[-1]
    out = torch.full((m, n), float("nan"), device="cuda")
    tc.run(executor, ins, [out])
    return out.cpu()


# whether the reduction is innermost in the first operand, in the second one, and whether a bias is added
ORDERS = {"mk,kn": (True, False, False), "mk,nk": (True, True, True), "km,kn": (False, False, False), "km,nk": (False, True, True)}
SIZES = [  # sizes, orders of the operands in which they are taken, tiles of a wavefront, wavefronts and slices
    (1000, 1000, 1000, "mk,kn mk,nk km,kn km,nk", "4, 4, 1, 1, 8"),  # 64 x 64 outputs a block, the last step of eight points
    (691, 792, 1840, "mk,kn mk,nk km,kn km,nk", "4, 4, 1, 1, 8"),
    (254, 292, 1500, "mk,kn km,kn", "1, 2, 1, 1, 8"),                # 16 x 32
    (655, 1031, 545, "mk,kn km,kn km,nk", "4, 4, 1, 1, 8"),          # one point in the last step, an odd number of columns
    (45, 2516, 2699, "mk,kn km,kn km,nk", "1, 2, 1, 1, 8"),          # fewer rows than a tile of 48 has
    (986, 71, 1987, "mk,kn km,kn", "1, 2, 1, 1, 8"),
    (497, 681, 1530, "mk,kn km,kn km,nk", "4, 2, 1, 1, 8"),          # 64 x 32
    (617, 467, 6106, "mk,nk", "4, 2, 1, 1, 8"),
    (2048, 2048, 160, "km,kn", "4, 4, 2, 2, 2"),                     # an odd number of steps for two slices
    (2062, 1895, 768, "mk,kn mk,nk km,kn km,nk", "4, 4, 2, 2, 2"),   # 128 x 128, four rectangles of wavefronts
    (451, 349, 996, "km,nk", "2, 2, 1, 1, 8"),
    (1171, 37, 2759, "km,nk", "1, 1, 1, 1, 8"),                      # fewer outputs to a slice than a wavefront has lanes
    (907, 2194, 798, "km,nk", "2, 4, 1, 1, 4"),
    (1401, 1122, 366, "km,nk", "4, 2, 1, 2, 4"),                     # two rectangles side by side
]
TAKEN = [(*size[:3], order) for size in SIZES for order in size[3].split()]


def mapped(m, n, k, order):
    a_inner, b_inner, bias = ORDERS[order]
    shapes = [(m, k) if a_inner else (k, m), (n, k) if b_inner else (k, n)] + ([(n,)] if bias else [])
    text, _ = tc.map_only(source(a_inner, b_inner, bias), "f", [ShapeOnly(s) for s in shapes], options(m, n))
    return text.split('extern "C"')[-1]


@pytest.mark.parametrize("m,n,k,orders,tiles", SIZES)
def test_shapes_of_the_sizes_below(m, n, k, orders, tiles):
    for order in orders.split():
        assert f"{m}, {n}, {k}, {tiles}>" in mapped(m, n, k, order)


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,order", TAKEN)
def test_sums(m, n, k, order):
    print(m, n, k, order, flush=True)
    a_inner, b_inner, bias = ORDERS[order]
    generator = torch.Generator().manual_seed(m)
    ints = lambda *s: torch.randint(-8, 9, s, generator=generator).float()  # noqa: E731
    a, b, c = ints(m, k), ints(n, k), ints(n)
    got = run(m, n, k, a_inner, b_inner, a, b, c if bias else None)
    want = a.double() @ b.double().t()
    assert torch.equal(got.double(), want + c if bias else want)     # (sums of whole numbers are exact)
    a, b, c = (torch.randn(s, generator=generator) for s in ((m, k), (n, k), (n,)))
    got = run(m, n, k, a_inner, b_inner, a, b, c if bias else None).double()
    want, magnitudes = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    if bias:
        want, magnitudes = want + c, magnitudes + c.abs()
    # one rounding of 2^-24 a term and the bias, in whatever order, and up to 2^-24 of every product for the parts left out
    assert ((got - want).abs() <= (k + 2) * 2.0 ** -24 * magnitudes).all()
    # Roundings do not add up like that: 0.7e-7 to 2.9e-7 here.  Without any one of the six products of parts it is 2.4e-6 or more.
    assert (got - want).norm() <= 1e-6 * want.norm()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,order", TAKEN)
def test_every_product_of_parts(m, n, k, order):
    """Sums of 24 bits, which are exact only with all six products of parts: values 1 + y 2^-9 + z 2^-18 (y, z of -1, 0, 1) in 24 points a row."""
    a_inner, b_inner, bias = ORDERS[order]
    generator = torch.Generator().manual_seed(k)

    def values(rows, low):
        x, y, z = (torch.randint(-1, 2, (rows, k), generator=generator).float() for _ in range(3))
        return x * (1 + y * 2.0 ** -9 + (z * 2.0 ** -18 if low else 0))

    points = torch.zeros(k)
    points[torch.randperm(k, generator=generator)[:24]] = 1.0
    for low_a, low_b, middle in ((True, False, False), (False, True, False), (False, False, True)):
        a = values(m, low_a) * points if low_a or middle else torch.randint(-1, 2, (m, k), generator=generator) * points
        b = values(n, low_b) if low_b or middle else torch.randint(-1, 2, (n, k), generator=generator).float()
        got = run(m, n, k, a_inner, b_inner, a, b, torch.zeros(n) if bias else None)
        assert torch.equal(got.double(), a.double() @ b.double().t())


@pytest.mark.gpu
@pytest.mark.parametrize("case", ["infinity", "nan", "rounds to infinity", "small", "small rows", "denormal", "large", "large sums", "zero rows"])
def test_values_the_parts_cannot_hold(case):
    m, n, k = 254, 292, 1500
    generator = torch.Generator().manual_seed(2)
    a, b = torch.randn(m, k, generator=generator), torch.randn(n, k, generator=generator)
    if case == "infinity":
        a.view(-1)[[5, 47110, -1]] = torch.tensor([np.inf, -np.inf, np.inf])
    elif case == "nan":
        a.view(-1)[[5, 47110]] = np.nan
    elif case == "rounds to infinity":
        a.view(-1)[::10001] = 3.4e38              # its nearest bf16 is infinite
        b *= 2.0 ** -20
    elif case == "small":
        a *= 2.0 ** -110                          # what is below 2^-134 of them is lost
    elif case == "small rows":
        a[::7] *= 2.0 ** -120
    elif case == "denormal":
        a *= 2.0 ** -140
    elif case == "large":
        a[3] *= 2.0 ** -110                       # beside values that lift its low parts out of the denormal numbers
        b *= 2.0 ** 90
    elif case == "large sums":
        a *= 2.0 ** 100
        b *= 2.0 ** 30                            # beyond the largest float
    else:
        a[::3] = 0
    got = run(m, n, k, True, False, a, b).double()
    want, magnitudes = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    finite = torch.isfinite(want) & (magnitudes < 3.4e38)
    # (a denormal sum is a whole number of 2^-149)
    assert ((got - want).abs()[finite] <= (k + 2) * (2.0 ** -24 * magnitudes[finite] + 2.0 ** -149)).all()
    if case in ("infinity", "nan"):
        assert torch.equal(torch.isnan(got), torch.isnan(want))
        assert torch.equal(got[torch.isinf(want)], want[torch.isinf(want)]) and torch.equal(torch.isinf(got), torch.isinf(want))
    if case == "zero rows":
        assert (got[::3] == 0).all()


@pytest.mark.parametrize("m,n,k,a_inner,b_inner,taken", [
    (1250, 208, 1015, True, False, True),
    # two rounds of full tiles over few points, which the general pipeline does in 10 us, this form in 14
    (1250, 1015, 208, True, False, False),
    (4072, 261, 219, True, False, False),
    (1064, 1261, 162, False, False, False),
    (1108, 1394, 564, True, True, False),
])
def test_which_products_are_taken(m, n, k, a_inner, b_inner, taken):
    shapes = [(m, k) if a_inner else (k, m), (n, k) if b_inner else (k, n)]
    text, _ = tc.map_only(source(a_inner, b_inner), "f", [ShapeOnly(s) for s in shapes], options(m, n))
    assert ("__tc::SlicedProduct<" in text.split('extern "C"')[-1]) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,tiles", [(1000, 1000, 1000, "4, 4, 1, 1, 8"), (254, 292, 1500, "1, 2, 1, 1, 8")])
@pytest.mark.parametrize("case", ["denormal rows", "denormal columns", "denormal terms", "denormal rows, small sums", "zero rows", "large, zero rows"])
def test_small_values_beside_others(m, n, k, tiles, case):
    """Values below what the parts hold, beside ordinary ones and times large ones, where a lane sees several rows."""
    generator = torch.Generator().manual_seed(3)
    a, b = torch.randn(m, k, generator=generator), torch.randn(n, k, generator=generator)
    if case == "denormal rows":
        a[::7] *= 2.0 ** -140
        b *= 2.0 ** 28
    elif case == "denormal columns":
        b[::5] *= 2.0 ** -139
        a *= 2.0 ** 29
    elif case == "denormal terms":                # ordinary values meet zeros: the sum is one of the others
        a[3, 1::2] *= 2.0 ** -140
        b[17, ::2] = 0
        b[17] *= 2.0 ** 30
    elif case == "denormal rows, small sums":
        a[::7] *= 2.0 ** -137
        b *= 2.0 ** -5
    elif case == "zero rows":
        a[::3] = 0
    else:
        a[::3] = 0
        a[1] *= 2.0 ** 60
    text, _ = tc.map_only(source(True, False), "f", [ShapeOnly((m, k)), ShapeOnly((k, n))], options(m, n))
    assert f"{m}, {n}, {k}, {tiles}>" in text
    got = run(m, n, k, True, False, a, b).double()
    want, magnitudes = a.double() @ b.double().t(), a.double().abs() @ b.double().abs().t()
    # (a denormal sum is a whole number of 2^-149)
    assert ((got - want).abs() <= (k + 2) * (2.0 ** -24 * magnitudes + 2.0 ** -149)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("m,n,k,order", [t for t in TAKEN if t[:3] in [(1000, 1000, 1000), (254, 292, 1500), (655, 1031, 545), (2062, 1895, 768)]])
def test_sums_of_floats_themselves(m, n, k, order):
    """Blocks that compute again, with every order of the operands: an infinity and a NaN reach their row and column alone, also where the last step
    has fewer points, and denormal operands keep their sums."""
    a_inner, b_inner, bias = ORDERS[order]
    generator = torch.Generator().manual_seed(4)
    a, b, c = (torch.randn(s, generator=generator) for s in ((m, k), (n, k), (n,)))
    for scale in (1.0, 2.0 ** -125):
        x, y = a * scale, b.clone()
        if scale == 1.0:
            x[0, k - 1], x[m - 1, 0], y[n - 1, k - 1] = np.inf, -np.inf, np.nan
        got = run(m, n, k, a_inner, b_inner, x, y, c if bias and scale == 1.0 else 0 * c if bias else None).double()
        x, y = x.double(), y.double()
        want, magnitudes = x @ y.t(), x.abs() @ y.abs().t()
        if bias and scale == 1.0:
            want, magnitudes = want + c, magnitudes + c.abs()
        assert torch.equal(torch.isnan(got), torch.isnan(want)) and torch.equal(got[torch.isinf(want)], want[torch.isinf(want)])
        finite = torch.isfinite(want)
        # (a denormal sum is a whole number of 2^-149)
        assert ((got - want).abs()[finite] <= (k + 2) * (2.0 ** -24 * magnitudes[finite] + 2.0 ** -149)).all()


@pytest.mark.gpu
def test_time_of_sums_of_floats_themselves():
    """A block that computes again uses the matrix cores too: one infinity makes a product take some 2.4 times as long (without them 50 times)."""
    m = n = k = 1000
    a, b = torch.randn(m, k, device="cuda"), torch.randn(k, n, device="cuda")
    executor = tc.compile(source(True, False), "f", [a, b], options(m, n))
    out = torch.empty(m, n, device="cuda")
    times = []
    for value in (1.0, float("inf")):
        a[5, 7] = value
        tc.run(executor, [a, b], [out])
        times.append(min(tc.profile_repeated(executor, [a, b], [out], 20) for _ in range(5)))
    assert times[1] < 8 * times[0]
