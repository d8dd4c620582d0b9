"""Products of float16 operands at the edges of what the wide matrix instruction, the vector and the
transposing reads of the copies take: reduction tiles that are deepened to 64 points or not, whole
and partial last tiles, rows of whole vectors and ragged ones, block tiles that overhang.  Small
integers: every sum is exact, so results equal numpy's in every bit."""
import numpy as np
import pytest
import torch

import tensorcomprehensions_amd as tc
from tests import benchmark_tcs as B

pytestmark = pytest.mark.gpu

# A(k, m): rows along the output variable in the first operand as well
TRANSPOSED_A = "def half_tam(float16(K, M) A, float16(K, N) B) -> (C) { C(m, n) +=! float(A(r_k, m)) * float(B(r_k, n)) }"
# operands that start inside their tensors: subscripts of one variable and a constant, or its mirror image
SHIFTED = ("def half_shift(float16(M, KP) A, float16(KQ, N) B) -> (C) { C(m, n) +=! float(A(%s)) * float(B(%s))"
           " where r_k in 0:%d, m in 0:%d, n in 0:%d }")

def ints(shape, seed):
    return np.random.Generator(np.random.Philox(seed)).integers(-4, 5, size=shape).astype(np.float16)


def run(src, entry, arrays, options):
    ins = [torch.from_numpy(a).cuda() for a in arrays]
    ex = tc.compile(src, entry, ins, options)
    outs = tc.prepare_outputs(src, entry, ins)
    outs[0].fill_(float("nan"))
    tc.run(ex, ins, outs)
    torch.cuda.synchronize()
    return outs[0].cpu().numpy(), ex.compiled_source


@pytest.mark.parametrize("m,k,n,tile,waves,wide", [
    (128, 128, 128, "64,64,32", 8, True),       # two deepened tiles
    (128, 127, 128, "64,64,32", 8, False),      # one short of two: as given
    (128, 160, 256, "64,64,32", 4, True),       # deepened, last tile half full
    (128, 160, 256, "64,64,16", 4, False),      # shallower tiles stay
    (130, 200, 132, "64,64,32", 8, True),       # whole vectors of eight, partial tiles on every side
    (65, 203, 97, "64,64,64", 8, True),         # rows of any length
    (144, 192, 192, "48,96,64", 6, True),       # rectangles of one tile by three
    (32, 192, 224, "32,112,64", 4, True),       # 14 output tiles in 16 places: rectangles that overhang
    (224, 192, 32, "112,32,64", 4, True),
    (256, 192, 512, "128,256,32", 8, True),
    (64, 96, 64, "64,64,24", 8, False),         # 24 does not divide 64
    (64, 320, 64, "32,32,32", 8, False),        # fewer output tiles than wavefronts
    (144, 160, 160, "48,80,32", 4, False),      # no rectangles: the given tile, one output tile at a time
])
def test_products_are_exact(m, k, n, tile, waves, wide):
    A, Bm = ints((m, k), m + k), ints((k, n), k + n)
    want = A.astype(np.float32) @ Bm.astype(np.float32)
    options = f"naive;tile={tile};mapToThreads=64,{waves};mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"
    for src, entry, arrays in ((B.HALF_MATMUL, "half_matmul", [A, Bm]),
                               (B.HALF_TMM, "half_tmm", [A, np.ascontiguousarray(Bm.T)]),
                               (TRANSPOSED_A, "half_tam", [np.ascontiguousarray(A.T), Bm])):
        print(f"{entry} {m}x{k}x{n} tile={tile} waves={waves}", flush=True)
        got, text = run(src, entry, arrays, options)
        assert np.array_equal(got, want), entry
        assert ("const __tc::halfx8 av_" in text) == wide, entry
        if wide:
            assert ("__tc::readTransposed(&" in text) == (entry != "half_tmm")


@pytest.mark.parametrize("a,b,m,k,n,vectors", [
    ("m, r_k + 3", "r_k, n", 64, 128, 64, True),
    ("m, r_k", "r_k + 1, n + 2", 64, 128, 64, True),
    ("m + 1, r_k + 3", "r_k + 3, n + 5", 65, 131, 67, True),    # rows that end in mid-vector
    ("m + 2, r_k", "r_k, 66 - n", 66, 130, 67, False),          # a mirrored subscript keeps the general reads
    ("65 - m, r_k + 1", "r_k + 1, 98 - n", 66, 160, 99, False),
])
def test_offsets_move_the_copies_and_not_their_reads(a, b, m, k, n, vectors):
    A, Bm = ints((m + 2, k + 3), 1), ints((k + 3, n + 5), 2)
    index = {"m": np.arange(m), "r_k": np.arange(k), "n": np.arange(n)}
    rows = [[eval(sub, {}, index) for sub in subs.split(",")] for subs in (a, b)]  # the subscripts, on all points
    want = A[np.ix_(*rows[0])].astype(np.float32) @ Bm[np.ix_(*rows[1])].astype(np.float32)
    got, text = run(SHIFTED % (a, b, k, m, n), "half_shift", [A, Bm],
                    "naive;tile=64,64,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert np.array_equal(got, want)
    assert ("__tc::readTransposed(&lds0_B[" in text) == vectors


def test_a_tensor_that_is_both_operands():
    A = ints((192, 320), 5)
    got, _ = run("def half_gram(float16(M, K) A) -> (C) { C(m, n) +=! float(A(m, r_k)) * float(A(n, r_k)) }", "half_gram", [A],
                 "naive;tile=64,64,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert np.array_equal(got, A.astype(np.float32) @ A.T.astype(np.float32))


def test_lds_limit_of_the_options_keeps_the_given_tile():
    """128 x 256 tiles of 64 points twice are 108 KB: under a limit of 64 KB the tile stays 32 deep."""
    A, Bm = ints((128, 256), 3), ints((256, 256), 4)
    got, text = run(B.HALF_MATMUL, "half_matmul", [A, Bm],
                    "naive;tile=128,256,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1;maxSharedMemory=65536")
    assert np.array_equal(got, A.astype(np.float32) @ Bm.astype(np.float32))
    assert "const __tc::halfx8 av_" not in text


@pytest.mark.parametrize("m,k,n,tile,blocks", [(126, 81, 44, "16,16,13", "3,256"), (70, 81, 50, "16,16", "2,2"), (191, 105, 34, "4,4,2", "1,256")])
def test_odd_rows_of_tiles_requested_ahead(m, k, n, tile, blocks):
    """Blocks that walk several tiles and request the next one's operands ahead, rows of an odd number of halves: vectors across
    the end of a tensor are shifted by the place of the tile they belong to."""
    g = torch.Generator(device="cuda").manual_seed(k)
    A, B = (torch.randint(-3, 4, s, generator=g, device="cuda").half() for s in ((m, k), (k, n)))
    src = "def f(float16(M, K) A, float16(K, N) B) -> (O) { O(m, n) +=! float(A(m, r_k)) * float(B(r_k, n)) }"
    ex = tc.compile(src, "f", [A, B], f"naive;tile={tile};mapToThreads=64,4;mapToBlocks={blocks};useMfma=1;useSharedMemory=1;prefetchShared=1")
    out = torch.full((m, n), float("nan"), device="cuda")
    tc.run(ex, [A, B], [out])
    assert torch.equal(out, A.float() @ B.float())
