"""Rules by which the mapper chooses a kernel's form, on the generated source (no GPU)."""
import re

import pytest

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly
from tests.scaffolding import scaffold_query


def mapped(src, entry, shapes, options):
    return tc.map_only(src, entry, [ShapeOnly(s) for s in shapes], options)


@pytest.mark.parametrize("term,staged", [("I(n, k) * I(n, k)", False), ("I(n, k) * I(n, k + 1) * I(n, k + 2)", True)])
def test_loads_of_one_element_are_one_access(term, staged):
    """An element a thread names twice is read once: no reuse that would pay for a copy in LDS; three
    neighbouring elements are reuse between threads."""
    src = "def f(float(N, K) I) -> (s) { s(n) +=! %s where k in 0:4096 }" % term
    text, _ = mapped(src, "f", [(64, 4100)], "naive;tile=1,0;mapToThreads=256;mapToBlocks=64;matchLibraryCalls=1;useSharedMemory=1")
    assert ("lds0_I" in text) == staged


MATRIX = "mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1"


@pytest.mark.parametrize("dtype", ["float", "float16"])
@pytest.mark.parametrize("columns,vectors", [("n", True), ("100 - n", False)])
def test_no_vector_of_a_copy_begins_in_front_of_its_tensor(dtype, columns, vectors):
    """100 - n over tiles of 64 points: the second tile's copy starts 27 elements in front of the
    row, and a vector of four would hold element 0 of the tensor as its last."""
    load = "%s" if dtype == "float" else "float(%s)"
    src = f"def f({dtype}(M, K) A, {dtype}(K, N) B) -> (O) {{ O(m, n) +=! {load % 'A(m, r_k)'} * {load % f'B(r_k, {columns})'} where n in 0:101 }}"
    name = "float32" if dtype == "float" else "float16"
    text, _ = tc.map_only(src, "f", [ShapeOnly((96, 128), name), ShapeOnly((128, 101), name)], f"naive;tile=64,64,32;{MATRIX}")
    loads = re.findall(r"pk\d*_B_\[it_\] = (?:__tc::loadBounded|\*|pB\[).*", text)
    assert loads and all(("x4" in line) == vectors for line in loads)
    if not vectors:
        assert all("__tc::tmax(0, " in line or "(unsigned)g1_ < 101u" in line for line in loads)


@pytest.mark.parametrize("threads,used", [("256,8", 1024), ("64,64", 1024), ("32,32,8", 1024), ("1024,1024", 1024), ("16,15", 240), ("4294967296,4294967296", 1024)])
def test_streams_take_any_nominal_block(threads, used):
    """Thread sizes for loops that merging removed are nominal: their product may pass the device's
    limit (and 64 bits)."""
    src = "def f(float(N, M) A, float(N, M) B) -> (O) { O(n, m) = A(n, m) + B(n, m) }"
    for blocks in ("256,256", "4294967296,4294967296"):
        _, launches = tc.map_only(src, "f", [ShapeOnly((512, 1000))] * 2, f"naive;tile=32,32;mapToThreads={threads};mapToBlocks={blocks}")
        (grid, block), = launches
        assert block == (used, 1, 1) and grid == (-(-512 * 1000 // (4 * used)), 1, 1)


@pytest.mark.parametrize("dtype,name,through", [("float", "float32", True), ("int32", "int32", True), ("float16", "float16", False),
                                                ("double", "float64", False), ("int8", "int8", False)])
def test_only_words_of_a_stream_are_written_through(dtype, name, through):
    src = f"def f({dtype}(N, M) A, {dtype}(N, M) B) -> (O) {{ O(n, m) = A(n, m) + B(n, m) }}"
    text, _ = tc.map_only(src, "f", [ShapeOnly((512, 1000), name)] * 2, "naive")
    assert ("__tc::storeThrough(rsO_" in text) == through
    text, _ = tc.map_only(src, "f", [ShapeOnly((512, 1000), name)] * 2, "naive;useReadOnlyCache=1")
    assert "__tc::storeThrough(rsO_" in text                    # as the options say


PRODUCT = "def f(float(M, K) A, float(N, K) B) -> (O) { O(m, n) +=! A(m, r_k) * B(n, r_k) }"


@pytest.mark.parametrize("extra,tiled", [
    ("useSharedMemory=1;prefetchShared=1", True), ("prefetchShared=1", False), ("useSharedMemory=1;prefetchShared=1;maxSharedMemory=9000", False),
    ("useSharedMemory=1;prefetchShared=1;sharedDepth=1", False),
])
def test_partial_reduction_tiles_need_copies_of_both_operands(extra, tiled):
    text, _ = tc.map_only(PRODUCT, "f", [ShapeOnly((512, 1000)), ShapeOnly((512, 1000))],
                          f"naive;tile=64,64,32;mapToThreads=64,8;mapToBlocks=256,256;useMfma=1;{extra}")
    assert ("for (int t_r_k" in text) == tiled and "kok_ ?" not in text


def test_a_copy_smaller_than_the_block_leaves_the_reduction_whole():
    """16 filters of 16 channels are fewer elements than threads and are not staged."""
    src = "def f(float(N, C, H, W) I, float(M, C, KH, KW) W1) -> (O) { O(n, m, h, w) +=! I(n, r_c, h + r_kh, w + r_kw) * W1(m, r_c, r_kh, r_kw) }"
    for threads, tiled in (("64,8", False), ("64,4", True)):
        text, _ = tc.map_only(src, "f", [ShapeOnly((32, 114, 16, 16)), ShapeOnly((64, 114, 1, 1))],
                              f"naive;tile=1,16,8,0,16;mapToThreads={threads};mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
        assert ("for (int t_r_c" in text) == tiled


HALF_PRODUCT = "def f(float16(M, K) A, float16(N, K) B) -> (O) { O(m, n) +=! float(A(m, r_k)) * float(B(n, r_k)) }"


@pytest.mark.parametrize("k,threads,vector,shifted", [
    (128, "64,8", 8, False),        # whole tiles
    (160, "64,8", 8, False),        # the last tile half empty: whole vectors all the same
    (164, "64,8", 4, False),        # rows of whole vectors of four
    (163, "64,8", 4, True),         # vectors across the end of the tensor
    (128, "64,16", 4, False),       # vectors of eight for half of the threads
])
def test_copies_of_halves(k, threads, vector, shifted):
    text, _ = tc.map_only(HALF_PRODUCT, "f", [ShapeOnly((128, k), "float16"), ShapeOnly((128, k), "float16")],
                          f"naive;tile=64,64,64;mapToThreads={threads};mapToBlocks=256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert set(re.findall(r"pk\d*_[AB]_\[it_\] = \*\(const __tc::halfx(\d)u\*\)", text)) == {str(vector)}
    assert ("= __tc::shiftDown(" in text) == shifted


def depths(text):
    return {int(d) for d in re.findall(r"t_r_k[^;]*\* (\d+)\)", text)}


@pytest.mark.parametrize("tile,k,depth", [("128,128,32", 127, 32), ("128,128,32", 128, 64), ("128,128,32", 224, 32), ("128,128,32", 288, 64),
                                          ("128,256,32", 160, 32), ("64,64,32", 160, 64), ("64,64,16", 128, 16), ("128,128,24", 240, 24)])
def test_tiles_of_halves_that_are_deepened(tile, k, depth):
    """To 64 points, from two tiles on, in large blocks up to an eighth of surplus points."""
    text, _ = tc.map_only(HALF_PRODUCT, "f", [ShapeOnly((512, k), "float16")] * 2, f"naive;tile={tile};{MATRIX}")
    assert depths(text) == {depth}


def test_a_deepened_tile_is_given_up_where_its_copies_fit_only_once():
    """Copies read through the transposing read have wider pitches than the rule counts on."""
    src = "def f(float16(K, M) A, float16(K, N) B) -> (O) { O(m, n) +=! float(A(r_k, m)) * float(B(r_k, n)) }"
    for limit, depth in ((38000, 32), (42000, 64)):
        text, _ = tc.map_only(src, "f", [ShapeOnly((256, 512), "float16")] * 2, f"naive;tile=64,64,32;{MATRIX};maxSharedMemory={limit}")
        assert depths(text) == {depth}
        assert text.count("lds0_A[") and f"lds0_A[{2 * depth * 80}]" in text  # two copies


@pytest.mark.parametrize("m,n,k,tile,threads,tail,tiled", [
    (512, 512, 200, "64,64,32", "64,8", ";prefetchShared=1", True),     # an eighth of surplus points under the pipeline
    (512, 512, 100, "64,64,32", "64,8", ";prefetchShared=1", False),    # more than a fifth
    (512, 512, 72, "64,64,32", "64,8", ";prefetchShared=1", False),     # three tiles
    (512, 512, 200, "64,64,32", "64,8", "", False),                     # no overlap to gain
    (512, 512, 1000, "64,64,32", "64,8", "", True),                     # whole, the copies do not fit
    (512, 512, 130, "64,64,32", "64,8", ";prefetchShared=1", True),     # whole, the steps are masked
    (512, 512, 33, "64,64,32", "64,8", ";prefetchShared=1", False),     # and half of them would be surplus
    (512, 512, 1000, "32,32,32", "64,8", ";prefetchShared=1", False),   # wavefronts that only a whole reduction keeps busy
    (512, 512, 1000, "32,32,32", "64,4", ";prefetchShared=1", True),
    (512, 512, 400, "16,32,128", "64,8", ";prefetchShared=1", True),    # a tile's reduction shared by four wavefronts
    (512, 512, 300, "16,32,128", "64,8", ";prefetchShared=1", False),
    (512, 512, 250, "64,64,32", "64,8", ";maxSharedMemory=9000", True), # masked either way
])
def test_partial_reduction_tiles(m, n, k, tile, threads, tail, tiled):
    text, _ = tc.map_only(PRODUCT, "f", [ShapeOnly((m, k)), ShapeOnly((n, k))],
                          f"naive;tile={tile};mapToThreads={threads};mapToBlocks=256,256;useMfma=1;useSharedMemory=1{tail}")
    assert ("for (int t_r_k" in text) == tiled


@pytest.mark.parametrize("k", [33, 70, 100, 160])
def test_partial_reduction_tiles_of_halves_stay(k):
    text, _ = tc.map_only(HALF_PRODUCT, "f", [ShapeOnly((512, k), "float16")] * 2, f"naive;tile=64,64,32;{MATRIX}")
    assert "for (int t_r_k" in text


@pytest.mark.parametrize("src,shape,options,staged", [
    ("def f(float(N, K) I) -> (s) { s(n) +=! I(n, k) * I(n, k) }", (64, 4096), "tile=1,0;mapToThreads=256;matchLibraryCalls=1", False),
    ("def f(float(N, K) I) -> (s) { s(n) +=! I(n, k) * I(n, k) }", (64, 4100), "tile=1,0;mapToThreads=256;matchLibraryCalls=1", True),
    ("def f(float(N, K) I) -> (s) { s(n) +=! I(n, k) * I(n, k) }", (64, 2000), "tile=1,0;mapToThreads=256;matchLibraryCalls=1;vectorWidth=4", True),
    ("def f(float(N, K) I) -> (s) { s(k) +=! I(n, k) * I(n, k) }", (128, 1000), "tile=32,32;mapToThreads=32", True),
    # (the sum before it leaves the elements in registers)
    ("def f(float(N, K) I) -> (t, s) { t(n) +=! I(n, k) s(n) +=! I(n, k) * I(n, k) }", (64, 4100),
     "outerScheduleFusionStrategy=Max;tile=1,0;mapToThreads=256;matchLibraryCalls=1;usePrivateMemory=1;unroll=64", False),
])
def test_squares_are_staged_where_the_copies_read_better(src, shape, options, staged):
    text, _ = mapped(src, "f", [shape], f"naive;{options};mapToBlocks=4096;useSharedMemory=1")
    assert bool(re.search(r"lds\d_I", text)) == staged


BANDS = "naive;tile=1,32,11,0,8;mapToThreads=64,8;useMfma=1;useSharedMemory=1;sharedDepth=7;prefetchShared=1"


@pytest.mark.parametrize("units,sizes,blocks,grid", [
    (256, "16x64x57x57", "256,256,256", "16x8x2"),      # 160 blocks of 11 rows leave units idle: 256 of 7
    (128, "16x64x57x57", "256,256,256", "16x5x2"),      # more blocks than units
    (256, "1x64x57x57", "256,256,256", "2x55x1"),
    (32, "1x64x57x57", "256,256,256", "2x14x1"),
    (256, "1x64x57x57", "2,5", "2x5x1"),                # as many blocks as the given tiles make: they stay
    (256, "32x64x30x30", "256,256,256", "32x3x2"),      # no smaller tile that is a quarter faster
    (256, "1x64x57x57", "64,64", "2x55x1"),
])
def test_convolutions_get_tiles_that_fill_the_device(units, sizes, blocks, grid):
    assert scaffold_query("convolution_grid", f"{units}|{sizes}|{BANDS};mapToBlocks={blocks}") == grid


def test_tiles_that_stay_as_given():
    for options in (BANDS.replace(";prefetchShared=1", ""), BANDS.replace("useSharedMemory=1;", ""), BANDS.replace(",0,8", ",0,0"),
                    BANDS.replace("1,32,11", "1,16,1")):    # fewer output tiles than wavefronts
        rows = 55 if "1,16,1" in options else 5
        got = scaffold_query("convolution_grid", f"256|1x64x57x57|{options};mapToBlocks=256,256,256")
        assert f"{rows}" in got.split("x")


@pytest.mark.parametrize("width,tile,waves,blocked", [
    (30, "1,16,7,0,8", 8, False),       # 13 tiles in one row as 16 places
    (30, "1,16,7,0,8", 4, False),
    (18, "1,16,14,0,8", 4, True),       # 14 as 16 in rows of four
    (18, "1,16,14,0,8", 8, False),      # in rows of two
    (34, "1,16,4,0,8", 8, True),        # 8 as 8
    (18, "1,32,7,0,8", 4, True),        # 2 x 7 as four rectangles of 2 x 2
])
def test_rectangles_of_output_tiles_overhang_only_so_far(width, tile, waves, blocked):
    src = "def f(float(N, C, H, W) I, float(M, C, KH, KW) W1) -> (O) { O(n, m, h, w) +=! I(n, r_c, h + r_kh, w + r_kw) * W1(m, r_c, r_kh, r_kw) }"
    text, _ = mapped(src, "f", [(256, 64, width, width), (96, 64, 3, 3)],
                     f"naive;tile={tile};mapToThreads=64,{waves};mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert bool(re.search(r"float ra_\[\d+\]\[", text)) == blocked


def test_sizes_that_keep_a_stream_and_a_half_tile_as_given():
    src = "def f(float(N, M) A, float(N, M) B) -> (O) { O(n, m) = A(n, m) + B(n, m) }"
    for options, launch in (("tile=256;mapToThreads=256;mapToBlocks=64", ((64, 1, 1), (256, 1, 1))),
                            ("tile=512;mapToThreads=256;mapToBlocks=64;vectorWidth=2", ((64, 1, 1), (256, 1, 1))),
                            ("tile=32;mapToThreads=32;mapToBlocks=64", ((64, 1, 1), (32, 1, 1)))):
        assert tc.map_only(src, "f", [ShapeOnly((512, 1000))] * 2, f"naive;{options}")[1] == [launch]
    text, _ = tc.map_only(HALF_PRODUCT, "f", [ShapeOnly((512, 512), "float16")] * 2, f"naive;tile=64,64,32;{MATRIX.replace(';prefetchShared=1', '')}")
    assert depths(text) == {32}


def test_a_deepened_tile_that_does_not_pay_leaves_the_given_one():
    """15 output tiles on four wavefronts form no rectangles: 160 points stay five tiles of 32."""
    text, _ = tc.map_only(HALF_PRODUCT, "f", [ShapeOnly((480, 160), "float16")] * 2,
                          f"naive;tile=48,80,32;{MATRIX.replace('64,8', '64,4')}")
    assert depths(text) == {32} and "for (int t_r_k" in text


ANY_HALF_PRODUCT = "def f(float16(%s) A, float16(%s) B) -> (O) { O(m, n) +=! float(A(%s)) * float(B(%s)) }"


@pytest.mark.parametrize("m,n,k,tile,changes,large", [
    (4096, 4096, 4096, "128,256,32", "", True),
    (2512, 3432, 256, "128,256,32", "", True),                  # as many outputs a round
    (1808, 3688, 384, "128,128,64", "", True),                  # 120 blocks compute twice as many
    (1784, 3256, 256, "128,128,64", "", False),                 # 91 blocks do
    (4096, 4096, 248, "128,256,32", "", False),                 # a short reduction
    (4096, 4096, 4092, "128,256,32", "", False),                # rows that are no whole vectors
    (4095, 4096, 4096, "128,256,32", "", True),                 # (rows of the output may be any number)
    (4096, 4095, 4096, "128,256,32", "", False),                # rows of B
    (4096, 4096, 4096, "128,256,32", "maxSharedMemory=131071", False),
    (4096, 4096, 4096, "128,256,32", "prefetchShared=0", False),
    (4096, 4096, 4096, "128,256,32", "mapToThreads=64,4", False),
    (4096, 4096, 4096, "128,256,32", "mapToBlocks=16,16", False),
    (4096, 4096, 4096, "128,256,32", "reductionBlocks=2", False),
])
def test_large_half_products(m, n, k, tile, changes, large):
    text, launches = tc.map_only(ANY_HALF_PRODUCT % ("M, K", "K, N", "m, r_k", "r_k, n"), "f", [ShapeOnly((m, k), "float16"), ShapeOnly((k, n), "float16")],
                                 f"naive;tile={tile};{MATRIX};{changes}")
    assert ("__tc::largeHalfProduct<true, false, " in text) == large
    if large:
        assert launches == [((-(-m // 256) * -(-n // 256), 1, 1), (64, 8, 1))]


@pytest.mark.parametrize("src,dtype", [
    (ANY_HALF_PRODUCT % ("M, K", "K, N", "m, r_k", "r_k, n"), "float16"),
    (ANY_HALF_PRODUCT.replace("+=!", "+=") % ("M, K", "K, N", "m, r_k", "r_k, n"), "float16"),                     # adds to what is there
    ((ANY_HALF_PRODUCT % ("M, K", "K, N", "m, r_k", "r_k, n")).replace(" }", " O(m, n) = fmax(O(m, n), 0) }"), "float16"),
    ((ANY_HALF_PRODUCT % ("M, K", "L, N", "m, r_k + 8", "r_k, n")).replace(" }", " where r_k in 0:4096 }"), "float16"),  # rows not read whole
    ((ANY_HALF_PRODUCT % ("M, K", "K, N", "4095 - m, r_k", "r_k, n")).replace(" }", " where m in 0:4096 }"), "float16"),
    ("def f(float(M, K) A, float(K, N) B) -> (O) { O(m, n) +=! A(m, r_k) * B(r_k, n) }", "float32"),
])
def test_other_products_keep_their_tiles(src, dtype):
    plain = src == ANY_HALF_PRODUCT % ("M, K", "K, N", "m, r_k", "r_k, n")
    text, _ = tc.map_only(src, "f", [ShapeOnly((4096, 4104 if "+ 8" in src else 4096), dtype), ShapeOnly((4096, 4096), dtype)], f"naive;tile=128,256,32;{MATRIX}")
    assert ("__tc::largeHalfProduct<" in text) == plain


@pytest.mark.parametrize("shape,blocks,grid", [
    ((1, 11, 16), "1,11", (11, 11, 1)),          # a variable of one tile uses up no axis, and no block size either
    ((1, 11, 16), "4,3", (4, 3, 1)),
    ((1, 1, 16), "1,1,5", (5, 1, 1)),
    ((3, 1, 16), "2,1,5", (2, 5, 1)),
    ((3, 5, 7), "2,4,6", (2, 4, 6)),             # none: as given
    ((1, 5, 7), "9,2,3", (5, 3, 1)),
])
def test_block_sizes_keep_their_variables(shape, blocks, grid):
    src = "def f(float(N, G, H) A, float(H, K) W) -> (O) { O(n, g, h) +=! A(n, g, h) * W(h, r_k) }"
    _, launches = mapped(src, "f", [shape, (shape[2], 8)], f"naive;tile=1,1,1;mapToThreads=1;mapToBlocks={blocks};collapseContiguous=0")
    assert launches[0][0] == grid


FLOAT_PRODUCT = "def f(float(M, K) A, float(K, N) B) -> (O) { O(m, n) +=! A(m, r_k) * B(r_k, n) }"


@pytest.mark.parametrize("m,k,n,tile,changes,grid", [
    (215, 1188, 1305, "64,64,32", "", (4, 41)),             # 84 blocks of 64x64: columns are halved
    (430, 1367, 1095, "64,64,32", "", (7, 35)),
    (691, 1840, 792, "64,64,32", "", (11, 13)),             # 275 would run in two rounds
    (215, 224, 1305, "64,64,32", "", (4, 21)),              # a short reduction
    (215, 1188, 1305, "64,64,32", "maxSharedMemory=65536", (4, 21)),
    (215, 1188, 1305, "64,64,32", "prefetchShared=0", (4, 21)),
    (215, 1188, 1305, "64,64,32", "mapToBlocks=4,21", (4, 21)),
    (254, 1500, 292, "16,32,128", "", (16, 10)),            # wavefronts already share a tile
])
def test_products_halve_a_side_to_fill_the_device(m, k, n, tile, changes, grid):
    _, launches = mapped(FLOAT_PRODUCT, "f", [(m, k), (k, n)], f"naive;tile={tile};{MATRIX};{changes}")
    assert sorted(launches[0][0][:2]) == sorted(grid)


@pytest.mark.parametrize("sizes,kernel,tile,blocks", [
    ((13, 83, 38, 7, 38), 3, "1,32,5,0,8", 13 * 2 * 5),     # one row a block: wavefronts share the reduction of six tiles
    ((4, 118, 21, 30, 38), 1, "1,32,15,0,8", 4 * 30),       # a reduction whose given tile is dropped
    ((4, 118, 21, 30, 38), 1, "1,32,15,0,0", 4 * 2),        # one that is given whole
    ((1, 64, 64, 57, 57), 3, "1,32,11,0,8", 2 * 55),
])
def test_convolutions_get_small_tiles_where_units_are_idle(sizes, kernel, tile, blocks):
    n, c, m, h, w = sizes
    src = "def f(float(N, C, H, W) I, float(M, C, KH, KW) W1) -> (O) { O(n, m, h, w) +=! I(n, r_c, h + r_kh, w + r_kw) * W1(m, r_c, r_kh, r_kw) }"
    _, launches = mapped(src, "f", [(n, c, h, w), (m, c, kernel, kernel)],
                         f"naive;tile={tile};mapToThreads=64,8;mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;prefetchShared=1")
    grid = launches[0][0]
    assert grid[0] * grid[1] * grid[2] == blocks


TENSORDOT = "def f(float(N, C1, C2, H, W) A, float(N, C2, C3, H, W) B) -> (O) { O(n, c1, c3, h, w) +=! A(n, c1, r_c2, h, w) * B(n, r_c2, c3, h, w) }"
STREAM = "naive;tile=1,8,2,0;mapToThreads=256;mapToBlocks=32,64;unroll=128;vectorWidth=4;useReadOnlyCache=1"


@pytest.mark.parametrize("sizes,changes,grid,sums", [
    ((32, 512, 8, 2, 28, 28), "", (32, 64, 1), 64),                 # blocks enough: as given
    ((16, 286, 3, 2, 25, 30), "", (16, 36, 1), 48),                 # nine wavefronts a compute unit
    ((4, 17, 8, 4, 47, 25), "", (4, 9, 5), 8),                      # 47 x 25 points to five blocks, then two of the 17
    ((4, 17, 8, 4, 47, 25), "useSharedMemory=1", (4, 3, 1), 80),
    ((4, 17, 8, 4, 47, 25), "mapToThreads=128,2", (4, 3, 1), None),
    ((4, 17, 8, 4, 47, 25), "mapToBlocks=4,2", (4, 2, 1), 80),      # fewer blocks than tiles: the ones asked for
    ((4, 17, 8, 4, 47, 25), "mapToBlocks=4,3", (4, 3, 5), 32),      # no more blocks along c1
    ((1, 93, 3, 3, 25, 25), "", (47, 2, 3), 4),                     # (with one n, c3 has a block axis)
    ((32, 512, 8, 4, 28, 28), "", (32, 64, 1), 64),                 # 128 sums would not fit
    ((32, 512, 8, 3, 7, 7), "", (32, 64, 1), 24),                   # all of c3 at once
    ((32, 512, 8, 3, 7, 7), "unroll=16", (32, 64, 1), 16),          # ... where the loops may be unrolled
])
def test_tiles_made_for_other_sizes(sizes, changes, grid, sums):
    n, c1, c2, c3, h, w = sizes
    text, launches = mapped(TENSORDOT, "f", [(n, c1, c2, h, w), (n, c2, c3, h, w)], f"{STREAM};{changes}")
    assert launches[0][0] == grid
    if sums is not None:
        assert f"float acc_[{sums}];" in text


@pytest.mark.parametrize("m,k,n,tile,changes,grid", [
    (881, 655, 2389, "128,128,16", "", (12, 19, 1)),            # 80 x 128: five tiles a wavefront for eight
    (1500, 800, 1700, "128,128,16", "", (12, 18, 1)),           # 128 x 96, a fifth less
    (1500, 112, 1700, "128,128,16", "", (12, 14, 1)),           # seven reduction tiles: as given
    (2048, 512, 2048, "128,128,16", "", (16, 16, 1)),           # blocks enough
    (2100, 900, 2100, "128,128,16", "", (15, 17, 1)),           # 144 x 128: one round of blocks for two
    (1100, 2000, 1100, "64,64,32", "", (12, 18, 1)),            # 96 x 64
    (1400, 600, 1100, "64,64,32", "", (22, 18, 1)),             # 128 x 64 is no gain
    (116, 2960, 204, "16,32,128", "", (8, 13, 1)),              # 16 x 16: half the staging a block
    (116, 896, 204, "16,32,128", "", (8, 7, 1)),
    (128, 2960, 1024, "16,32,128", "", (32, 8, 1)),
    (116, 2960, 204, "16,32,128", "mapToBlocks=8,7", (8, 7, 1)),
    (1100, 2000, 1100, "64,64,32", "maxSharedMemory=160000", (18, 18, 1)),
    (881, 655, 2389, "128,128,16", "mapToThreads=64,4", (12, 19, 1)),
    (881, 655, 2389, "128,128,16", "mapToBlocks=7,19", (7, 19, 1)),
])
def test_sides_of_products_fit_the_device(m, k, n, tile, changes, grid):
    text, launches = mapped("def f(float(M, K) A, float(K, N) B) -> (O) { O(m, n) +=! A(m, r_k) * B(r_k, n) }", "f", [(m, k), (k, n)],
                            f"naive;tile={tile};{MATRIX};{changes}")
    assert launches[0][0] == grid


@pytest.mark.parametrize("divisor,known", [
    ("(float(uint32(3 - 5)) + 11)", False),     # 4294967305
    ("(float(uint32(3) - uint32(5)) + 11)", False),
    ("(float(uint64(N - 5)) + 11)", False),
    ("(N - 5 + 11)", False),                    # (9: a step of it is negative)
    ("(float(uint32(N)) + 6)", True),
    ("(N + 11 - 5)", True),
])
def test_divisors_of_unsigned_steps(divisor, known):
    """A divisor counts as a known whole number only where no step of it is negative."""
    text, _ = mapped("def f(float(N) A) -> (O) { O(n) = A(n) / %s }" % divisor, "f", [(3,)], "naive;tile=256;mapToThreads=256")
    assert ("/ __tc::Whole<9>()" in text.split('extern "C"')[-1]) == known


ROWS = "def f(float(N, C1, C2, H) A, float(N, C2, C3, H) B) -> (O) { O(n, c1, c3, h) +=! A(n, c1, r_c2, h) * B(n, r_c2, c3, h) }"


@pytest.mark.parametrize("sizes,options,grid", [
    ((8, 8, 4, 100, 64), "tile=8,1,1,0;mapToThreads=64;mapToBlocks=200,200", (8, 100, 1)),      # a halved n would take c1's axis, c1 that of c3
    ((2, 8, 2, 4, 56, 56), "tile=1,8,4,0;mapToBlocks=32,64,8", (2, 8, 4)),                       # c3 that of the points in rows
    ((2, 64, 16, 4, 40, 36), "tile=1,8,4,0;mapToBlocks=32,64,8", (2, 64, 2)),
    ((3, 7, 15, 79, 14, 13), "", (3, 40, 1)),                                                    # c1 that of c3, of 79 points
    ((2, 8, 2, 3, 56, 56), "", (2, 4, 4)),                                                       # all three points of c3 fit the registers
])
def test_variables_keep_their_blocks_when_others_are_halved(sizes, options, grid):
    n, c1, c2, c3 = sizes[:4]
    plane = sizes[4:]
    source = ROWS if len(plane) == 1 else TENSORDOT
    base = "naive" if len(plane) == 1 else STREAM
    text, launches = mapped(source, "f", [(n, c1, c2) + plane, (n, c2, c3) + plane], f"{base};{options}")
    assert launches[0][0] == grid
    assert not re.search(r"for \(int t_(?!r_)", text.split('extern "C"')[-1])     # no block walks the tiles of a variable


@pytest.mark.parametrize("m,n,k,large", [
    (2048, 4096, 256, False), (2048, 4096, 320, False), (1808, 3688, 320, False),
    (2048, 4096, 384, False),                                   # 512 given blocks fill their two rounds
    (1808, 3688, 384, True),                                    # 435 of them do not
    (2048, 4096, 392, True), (2048, 4096, 712, True),           # the last tile is partial
    (2048, 4096, 512, True), (2048, 4096, 704, False), (2048, 4096, 1280, True),
    (2816, 2816, 1216, False), (2816, 2816, 1344, True),
    (2880, 2904, 256, True), (2880, 2904, 320, True),           # three rounds of given blocks: a third more outputs
    (4096, 4096, 320, True),                                    # as many
])
def test_twice_as_many_outputs_need_a_deep_reduction(m, n, k, large):
    text, _ = tc.map_only(ANY_HALF_PRODUCT % ("M, K", "N, K", "m, r_k", "n, r_k"), "f", [ShapeOnly((m, k), "float16"), ShapeOnly((n, k), "float16")],
                          f"naive;tile=128,128,64;{MATRIX}")
    assert ("__tc::largeHalfProduct<" in text.split('extern "C"')[-1]) == large


CONVOLUTION = "def f(%s(N, C, H, W) I, %s(M, C, KH, KW) W1) -> (O) { O(n, m, h, w) +=! %s * %s }"


@pytest.mark.parametrize("dtype,sizes,tile,waves,steps,half", [
    ("float16", (16, 84, 128, 22, 18), "1,128,7,0,7", 4, 16, True),     # 18 would leave the half instruction (and 4x4 tiles be dealt one by one)
    ("float16", (32, 84, 16, 26, 26), "1,64,16,0,7", 4, 16, True),
    ("float16", (2, 84, 128, 22, 40), "1,32,3,0,7", 8, 18, False),      # eight wavefronts have half the registers each
    ("float16", (16, 25, 256, 11, 42), "1,32,6,0,5", 8, 12, True),      # 18 for 12 does not pay on eight either
    ("float16", (32, 84, 256, 27, 12), "1,64,4,0,14", 4, 32, True),
    ("float16", (16, 72, 256, 29, 17), "1,128,1,0,6", 4, 14, False),    # the same instruction: the fewer steps
    ("float", (16, 28, 128, 42, 40), "1,128,6,0,7", 8, 16, False),     # 18 would lose the rectangles of 4x4 tiles
    ("float", (32, 56, 96, 32, 28), "1,32,23,0,7", 8, 18, False),
    ("float", (16, 42, 64, 17, 27), "1,16,5,0,14", 8, 36, False),       # one tile a wavefront
    ("float", (32, 60, 32, 35, 35), "1,32,3,0,5", 4, 12, False),        # 18 for 12
])
def test_whole_points_in_a_quarter_of_the_reduction(dtype, sizes, tile, waves, steps, half):
    n, c, m, h, w = sizes
    load = "%s" if dtype == "float" else "float(%s)"
    source = CONVOLUTION % (dtype, dtype, load % "I(n, r_c, h + r_kh, w + r_kw)", load % "W1(m, r_c, r_kh, r_kw)")
    name = "float32" if dtype == "float" else dtype
    text, _ = tc.map_only(source, "f", [ShapeOnly((n, c, h, w), name), ShapeOnly((m, c, 3, 3), name)],
                          f"naive;tile={tile};mapToThreads=64,{waves};mapToBlocks=256,256,256;useMfma=1;useSharedMemory=1;sharedDepth=7")
    body = text.split('extern "C"')[-1]
    assert f", {steps} steps of " in body
    assert ("__tc::multiplyHalves(" in body) == half


@pytest.mark.parametrize("blocks", ["256,256,256", "1,256,256", "1,2,256"])
def test_tiles_that_fill_the_device_see_the_block_sizes_of_their_variables(blocks):
    """One image: its variable uses up no block axis, and no block size."""
    source = CONVOLUTION % ("float", "float", "I(n, r_c, h + r_kh, w + r_kw)", "W1(m, r_c, r_kh, r_kw)")
    _, launches = mapped(source, "f", [(1, 64, 57, 57), (64, 64, 3, 3)],
                         f"naive;tile=1,32,11,0,8;mapToThreads=64,8;mapToBlocks={blocks};useMfma=1;useSharedMemory=1;prefetchShared=1")
    assert launches[0][0] == (2, 55, 1)


@pytest.mark.parametrize("blocks,large", [("1,8", True), ("1,7", False), ("8,1", True)])
def test_large_half_products_see_the_block_sizes_of_their_variables(blocks, large):
    text, _ = tc.map_only(ANY_HALF_PRODUCT % ("M, K", "N, K", "m, r_k", "n, r_k"), "f", [ShapeOnly((256, 1024), "float16"), ShapeOnly((2048, 1024), "float16")],
                          f"naive;tile=256,256,32;{MATRIX};mapToBlocks={blocks}")
    assert ("__tc::largeHalfProduct<" in text.split('extern "C"')[-1]) == large


@pytest.mark.parametrize("sizes,blocks,grid", [
    ((2, 70000), "1,2,100000", [1, 2, 65535]), ((70000, 2), "1,100000,2", [1, 2, 65535]), ((2, 70000), "1,1,4294967296", [1, 1, 65535]),
    ((70000, 1), "100000,1", [1, 1, 70000]),                # the axis's own size is as given
])
def test_block_sizes_of_places_fit_every_axis(sizes, blocks, grid):
    """A variable that moves up to another axis brings no more blocks than a launch takes on the second and third."""
    _, launches = mapped("def f(float(G, H) A) -> (O) { O(n, g, h) = A(g, h) + 1 where n in 0:1 }", "f", [sizes],
                         f"naive;tile=1,1,1;mapToThreads=1;mapToBlocks={blocks};collapseContiguous=0")
    assert sorted(launches[0][0]) == grid


@pytest.mark.parametrize("m,k,n,tile,blocks", [(126, 81, 44, "16,16,13", "3,256"), (70, 81, 50, "16,16", "2,2"), (191, 105, 34, "4,4,2", "1,256")])
def test_shifted_vectors_of_a_tile_requested_ahead(m, k, n, tile, blocks):
    """Rows of an odd number of halves, walked by blocks that request the next tile's operands while they multiply: the stores
    shift vectors across the tensor's end by the place of that tile."""
    source = ANY_HALF_PRODUCT % ("M, K", "K, N", "m, r_k", "r_k, n")
    shapes = [ShapeOnly((m, k), "float16"), ShapeOnly((k, n), "float16")]
    options = f"naive;tile={tile};mapToThreads=64,4;mapToBlocks={blocks};useMfma=1;useSharedMemory=1;prefetchShared=1"
    text, _ = tc.map_only(source, "f", shapes, options)
    stores = text.split('extern "C"')[-1].rsplit("if (more_)", 1)[1]
    assert "__tc::shiftDown(" in stores and re.search(r"const int lo0_\w+_\d = .*\(t_\w+ \+ \d+\)", stores)
    tc.compile(source, "f", shapes, options)


@pytest.mark.parametrize("tile,threads,later", [
    ("32,32,16", "64,4", True),             # rectangles
    ("16,16,16", "64,8", True),             # tile by tile
    ("16,16,0", "64,2", True),              # the whole reduction: 22 steps a quarter, no vector of four
    ("48,16,128", "64,2", False),           # 32 steps of a reduction tile, tile by tile
])
def test_loads_from_memory_are_tested_together(tile, threads, later):
    """A load with its test beside it is waited for before the next one leaves: values from memory get their zeros afterwards."""
    text, _ = mapped(FLOAT_PRODUCT, "f", [(70, 85 if tile.endswith(",0") else 333), (85 if tile.endswith(",0") else 333, 70)],
                     f"naive;tile={tile};mapToThreads={threads};mapToBlocks=64,64;useMfma=1;useSharedMemory=0")
    body = text.split('extern "C"')[-1]
    assert "kok_" in body
    assert bool(re.search(r"__tc::keep\(kok_, p[AB]\[", body)) != later
    assert bool(re.search(r"\[[a-z_]+\] = __tc::keep\(kok_, (ra|rb|aq|bq)_\[", body)) == later
