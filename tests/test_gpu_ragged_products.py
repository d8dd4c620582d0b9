"""Matrix products and convolutions whose sides are no multiples of the tiles: reduction tiles that
end past the reduction, rows that end in mid-vector, tensors that end in mid-vector, rectangles of
output tiles that overhang the block tile.  Integer-valued data: bit-exact against numpy, the oracle
for the convolution."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc
from oracle import tc_oracle
from tests import benchmark_tcs as B

pytestmark = pytest.mark.gpu

TAIL = "mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"
TILES = ["16,32,128", "64,64,32", "128,128,16"]
HALF_TILES = ["64,64,32", "128,128,64", "128,256,32"]
# m, k, n: one past and one short of tiles and vectors, odd everywhere, a single short reduction tile
SIZES = [(64, 33, 64), (65, 36, 67), (130, 70, 129), (127, 131, 255), (200, 1000, 72), (17, 261, 5), (96, 130, 300)]


def ints(shape, seed, dtype=np.float32):
    return np.random.Generator(np.random.Philox(seed)).integers(-4, 5, size=shape).astype(dtype)


def run(src, entry, arrays, options):
    ins = [torch.from_numpy(a).cuda() for a in arrays]
    ex = tc.compile(src, entry, ins, options)
    outs = tc.prepare_outputs(src, entry, ins)
    outs[0].fill_(float("nan"))
    tc.run(ex, ins, outs)
    torch.cuda.synchronize()
    return outs[0].cpu().numpy()


@pytest.mark.parametrize("m,k,n", SIZES)
@pytest.mark.parametrize("half", [False, True])
def test_ragged_products_are_exact(m, k, n, half):
    dtype = np.float16 if half else np.float32
    A, Bm = ints((m, k), m + k, dtype), ints((k, n), k + n, dtype)
    want = A.astype(np.float32) @ Bm.astype(np.float32)
    for tile in HALF_TILES if half else TILES:
        for waves in (4, 8):
            print(f"product {m}x{k}x{n} half={half} tile={tile} waves={waves}", flush=True)
            options = f"naive;tile={tile};mapToThreads=64,{waves};{TAIL}"
            if half:
                got = run(B.HALF_MATMUL, "half_matmul", [A, Bm], options)
                got_t = run(B.HALF_TMM, "half_tmm", [A, np.ascontiguousarray(Bm.T)], options)
            else:
                got = run(B.MATMUL, "matmul", [A, Bm], options)
                got_t = run(B.TMM, "tmm", [A, np.ascontiguousarray(Bm.T)], options)
            assert np.array_equal(got, want) and np.array_equal(got_t, want), (tile, waves)


@pytest.mark.parametrize("half", [False, True])
def test_surplus_reduction_points_contribute_nothing_even_next_to_infinities(half):
    """The vector that ends a row reads on into the next row: an infinity there belongs to that row
    of the product alone."""
    dtype = np.float16 if half else np.float32
    A, Bm = ints((70, 37), 1, dtype), ints((37, 66), 2, dtype)
    A[5, 0] = Bm[0, 7] = np.inf
    A[6:8, 1:4] = 0.0
    with np.errstate(invalid="ignore"):
        want = A.astype(np.float32) @ Bm.astype(np.float32)
    src, entry = (B.HALF_MATMUL, "half_matmul") if half else (B.MATMUL, "matmul")
    got = run(src, entry, [A, Bm], f"naive;tile=64,64,32;mapToThreads=64,8;{TAIL}")
    assert np.array_equal(got, want, equal_nan=True)


@pytest.mark.parametrize("n,c,m,h,w,kernel,tile", [
    (2, 13, 37, 11, 15, 3, "1,32,9,0,8"), (2, 20, 33, 9, 7, 1, "1,32,3,0,8"), (1, 9, 16, 8, 18, 3, "1,16,3,0,4"),
])
def test_convolutions_over_channels_in_partial_tiles(n, c, m, h, w, kernel, tile):
    print(f"convolution {n}x{c}x{h}x{w} m={m} kernel={kernel} tile={tile}", flush=True)
    arrays = [ints((n, c, h, w), 3), ints((m, c, kernel, kernel), 4), ints((m,), 5)]
    got = run(B.CONVOLUTION, "convolution", arrays,
              f"naive;tile={tile};mapToThreads=64,8;mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;sharedDepth=7;prefetchShared=1")
    (want,) = tc_oracle.run(B.CONVOLUTION, "convolution", arrays)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,k,n", [(101, 128, 101), (130, 70, 129), (66, 33, 300), (67, 64, 5), (64, 96, 128)])
@pytest.mark.parametrize("first,second", [("m, r_k", "r_k, {n} - n"), ("{m} - m, r_k", "r_k, n"), ("r_k, {m} - m", "{n} - n, r_k")])
def test_reversed_subscripts_over_partial_tiles(m, k, n, first, second, half):
    """The copy of the last tile begins in front of the tensor."""
    dtype, ty, load = (np.float16, "float16", "float(%s)") if half else (np.float32, "float", "%s")
    A, Bm = ints((m, k), m + k, dtype), ints((k, n), k + n, dtype)
    want = A.astype(np.float32) @ Bm.astype(np.float32)
    stored = [A, Bm]
    if first.startswith("r_k"):
        stored = [A.T, Bm.T]
    dims = [[d.strip() for d in subs.split(",")] for subs in (first, second)]
    for i, side in enumerate(dims):
        for axis, sub in enumerate(side):
            if sub.startswith("{"):
                stored[i] = np.flip(stored[i], axis)
    stored = [np.ascontiguousarray(a) for a in stored]
    subs = [s.format(m=m - 1, n=n - 1) for s in (first, second)]
    src = (f"def f({ty}(P, Q) A, {ty}(R, S) B) -> (O) {{ O(m, n) +=! {load % f'A({subs[0]})'} * {load % f'B({subs[1]})'}"
           f" where m in 0:{m}, n in 0:{n}, r_k in 0:{k} }}")
    for tile in ("64,64,32", "16,32,64"):
        print(f"reversed {m}x{k}x{n} half={half} A({subs[0]}) B({subs[1]}) tile={tile}", flush=True)
        assert np.array_equal(run(src, "f", stored, f"naive;tile={tile};mapToThreads=64,8;{TAIL}"), want)


@pytest.mark.parametrize("extra", ["", "useSharedMemory=1", "useSharedMemory=1;prefetchShared=1;maxSharedMemory=9000", "useSharedMemory=1;sharedDepth=1",
                                   "useSharedMemory=1;prefetchShared=1"])
@pytest.mark.parametrize("m,k,n", [(70, 100, 66), (33, 250, 130), (130, 72, 65)])
def test_reductions_in_tiles_and_in_one_piece(m, k, n, extra):
    """Both sides of the rule that keeps a partial reduction tile or drops it, operands staged or not."""
    A, Bm = ints((m, k), m + k), ints((k, n), k + n)
    want = A @ Bm
    for tile, waves in (("64,64,32", 8), ("32,32,32", 8), ("16,32,64", 4)):
        options = f"naive;tile={tile};mapToThreads=64,{waves};mapToBlocks=256,256;useMfma=1;{extra}"
        print(f"product {m}x{k}x{n} {options}", flush=True)
        assert np.array_equal(run(B.MATMUL, "matmul", [A, Bm], options), want)
        assert np.array_equal(run(B.TMM, "tmm", [A, np.ascontiguousarray(Bm.T)], options), want)


@pytest.mark.parametrize("n,c,m,side,kernel,tile,waves", [
    (2, 13, 32, 30, 3, "1,16,7,0,8", 8), (2, 16, 32, 30, 3, "1,16,7,0,8", 4), (2, 12, 20, 18, 3, "1,32,7,0,8", 4), (3, 24, 16, 16, 1, "1,16,14,0,16", 8),
])
def test_convolutions_of_one_row_of_output_tiles(n, c, m, side, kernel, tile, waves):
    """Thirteen or fourteen output tiles on four or eight wavefronts."""
    arrays = [ints((n, c, side, side), 3), ints((m, c, kernel, kernel), 4), ints((m,), 5)]
    got = run(B.CONVOLUTION, "convolution", arrays,
              f"naive;tile={tile};mapToThreads=64,{waves};mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;sharedDepth=7;prefetchShared=1")
    (want,) = tc_oracle.run(B.CONVOLUTION, "convolution", arrays)
    assert np.array_equal(got, want)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,k,n", [(300, 1000, 260), (130, 513, 200), (96, 160, 128), (257, 2048, 129)])
def test_errors_on_deviates_stay_within_those_of_float_sums(m, k, n, half):
    """Products are exact in float (halves) or rounded once, and k of them are added in float: every
    element within (k + 1) u sum |a b|, u = 2^-24, and the norm of the errors within sqrt(k) u of the
    result's, about twice what rounding k sums at random leaves."""
    rng = np.random.Generator(np.random.Philox(k))
    dtype = np.float16 if half else np.float32
    A, Bm = rng.standard_normal((m, k)).astype(dtype), rng.standard_normal((k, n)).astype(dtype)
    want = A.astype(np.float64) @ Bm.astype(np.float64)
    bound = (k + 1) * 2.0 ** -24 * (np.abs(A.astype(np.float64)) @ np.abs(Bm.astype(np.float64)))
    for tile in (HALF_TILES if half else TILES):
        options = f"naive;tile={tile};mapToThreads=64,8;{TAIL}"
        print(f"deviates {m}x{k}x{n} half={half} tile={tile}", flush=True)
        got = run(B.HALF_MATMUL if half else B.MATMUL, "half_matmul" if half else "matmul", [A, Bm], options).astype(np.float64)
        assert (np.abs(got - want) <= bound).all()
        assert np.linalg.norm(got - want) <= np.sqrt(k) * 2.0 ** -24 * np.linalg.norm(want)


@pytest.mark.parametrize("waves", [4, 8])
@pytest.mark.parametrize("m,k,n", [(881, 130, 2389), (1479, 221, 1728), (1730, 171, 1478), (764, 258, 3237), (1500, 160, 1700), (2040, 128, 1100), (150, 200, 140), (2100, 130, 2100)])
def test_products_with_fitted_sides(m, k, n, waves):
    """Blocks of 80 to 144 rows or columns (128 given), where those of the given tiles leave compute units idle."""
    print(f"product {m}x{k}x{n} waves={waves}", flush=True)
    A, Bm = ints((m, k), m + k, np.float32), ints((k, n), k + n, np.float32)
    want = A @ Bm
    options = f"naive;tile=128,128,16;mapToThreads=64,{waves};{TAIL}"
    assert np.array_equal(run(B.MATMUL, "matmul", [A, Bm], options), want)
    assert np.array_equal(run(B.TMM, "tmm", [A, np.ascontiguousarray(Bm.T)], options), want)


@pytest.mark.parametrize("m,k,n", [(1100, 264, 1100), (1050, 300, 1080), (1150, 256, 1200)])
def test_products_with_longer_sides(m, k, n):
    A, Bm = ints((m, k), m + k, np.float32), ints((k, n), k + n, np.float32)
    options = f"naive;tile=64,64,32;mapToThreads=64,8;{TAIL}"
    assert np.array_equal(run(B.MATMUL, "matmul", [A, Bm], options), A @ Bm)
    assert np.array_equal(run(B.TMM, "tmm", [A, np.ascontiguousarray(Bm.T)], options), A @ Bm)


@pytest.mark.parametrize("m,k,n", [(116, 2960, 204), (108, 1643, 127), (17, 1100, 33), (16, 1024, 32), (64, 2048, 897)])
def test_few_blocks_over_long_reductions(m, k, n):
    """Blocks of 16 x 16 outputs (16 x 32 given), eight wavefronts sharing the reduction."""
    A, Bm = ints((m, k), m + k, np.float32), ints((k, n), k + n, np.float32)
    options = f"naive;tile=16,32,128;mapToThreads=64,8;{TAIL}"
    assert np.array_equal(run(B.MATMUL, "matmul", [A, Bm], options), A @ Bm)
    assert np.array_equal(run(B.TMM, "tmm", [A, np.ascontiguousarray(Bm.T)], options), A @ Bm)


@pytest.mark.parametrize("dtype", ["float", "float16"])
@pytest.mark.parametrize("m,k,n,options", [
    (45, 70, 37, "tile=32,32,16;mapToThreads=64,4"),            # rectangles of tiles, the last reduction tile partial
    (45, 70, 37, "tile=16,32,16;mapToThreads=64,4"),            # tile by tile
    (130, 93, 75, "tile=64,32,0;mapToThreads=64,4"),            # the whole reduction, 24 steps of a quarter
    (33, 61, 40, "tile=16,16,0;mapToThreads=64,2"),
    (50, 131, 33, "tile=32,16,64;mapToThreads=64,2"),           # runs of more steps
    (50, 300, 33, "tile=32,16,0;mapToThreads=64,4"),
])
def test_steps_past_the_reduction_with_operands_from_memory(dtype, m, k, n, options):
    """Without shared memory: steps that do not exist read an element that does, and count as zeros on both sides (an infinity
    there makes no NaN)."""
    g = torch.Generator(device="cuda").manual_seed(k)
    A, B = (torch.randint(1, 4, s, generator=g, device="cuda").to(torch.float16 if dtype == "float16" else torch.float32) for s in ((m, k), (k, n)))
    A[3, k - 1] = float("inf")
    load = "%s" if dtype == "float" else "float(%s)"
    src = f"def f({dtype}(M, K) A, {dtype}(K, N) B) -> (O) {{ O(m, n) +=! {load % 'A(m, r_k)'} * {load % 'B(r_k, n)'} }}"
    ex = tc.compile(src, "f", [A, B], f"naive;{options};mapToBlocks=64,64;useMfma=1;useSharedMemory=0")
    assert "matrix cores:" in ex.compiled_source
    out = torch.full((m, n), float("nan"), device="cuda")
    tc.run(ex, [A, B], [out])
    want = (A[:, :, None].double() * B[None].double()).sum(1)
    assert torch.equal(out.double(), want)
