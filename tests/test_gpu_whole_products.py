"""Batches of products with two tiles of rows or columns, taken whole by a block each: sizes around the tiles and around where the rule ends."""
import pytest
import torch

import tensorcomprehensions_amd as tc
from tensorcomprehensions_amd import ShapeOnly

SOURCE = "def f(float(B, N, M) X, float(B, M, K) Y) -> (Z) { Z(b, n, k) +=! X(b, n, r_m) * Y(b, r_m, k) }"


def options(b, n, k):
    return f"naive;tile=1,{min(n, 64)},{min(k, 64)};mapToThreads=64,4;mapToBlocks={b},2,2;useMfma=1;useSharedMemory=1"


@pytest.mark.gpu
@pytest.mark.parametrize("b,n,m,k", [(512, 65, 1, 65), (512, 65, 4, 65), (513, 97, 60, 97), (512, 112, 91, 112), (512, 112, 88, 112), (768, 65, 33, 64), (769, 96, 104, 9), (512, 17, 41, 65), (600, 120, 80, 66),
                                     (1024, 64, 64, 128), (512, 1, 130, 128)])
def test_products_taken_whole(b, n, m, k):
    print(b, n, m, k, flush=True)
    g = torch.Generator().manual_seed(n)
    for draw in (lambda *s: torch.randint(-8, 9, s, generator=g).float(), lambda *s: torch.randn(s, generator=g)):
        x, y = draw(b, n, m), draw(b, m, k)
        ins = [x.cuda(), y.cuda()]
        executor = tc.compile(SOURCE, "f", ins, options(b, n, k))
        # (the first one has too few points, and the operands of the 91 are more than half of the LDS)
        assert (executor.grid()[0] == b and max(executor.grid()[1:]) == 1) == (m not in (1, 91))
        out = torch.full((b, n, k), float("nan"), device="cuda")
        tc.run(executor, ins, [out])
        want, magnitudes = torch.bmm(x.double(), y.double()), torch.bmm(x.double().abs(), y.double().abs())
        # one rounding a term (sums of whole numbers are exact)
        bound = 0 * magnitudes if torch.equal(x, x.round()) else (m + 1) * 2.0 ** -24 * magnitudes
        assert ((out.cpu().double() - want).abs() <= bound).all()


@pytest.mark.parametrize("b,n,m,k,opts,blocks", [
    (512, 65, 33, 65, "", (512, 1, 1)),
    (511, 65, 33, 65, "", (511, 2, 2)),                       # fewer than two products a compute unit
    (768, 96, 33, 64, "", (768, 1, 1)),
    (767, 96, 33, 64, "", (767, 2, 1)),                       # rows alone: three products a compute unit
    (768, 97, 33, 64, "", (768, 2, 1)),
    (512, 64, 33, 65, "", (512, 1, 1)),                       # columns alone
    (512, 121, 33, 65, "", (512, 2, 2)),
    (512, 113, 33, 97, "", (512, 2, 2)),                      # 56 output tiles
    (512, 65, 300, 65, "", (512, 2, 2)),                      # operands beyond half of the LDS
    (512, 65, 33, 65, ";maxSharedMemory=16384", (512, 2, 2)),
    (512, 129, 33, 65, "", (512, 2, 2)),
    (512, 65, 3, 65, "", (512, 2, 2)),                        # fewer than four points
    (768, 96, 33, 8, "", (768, 2, 1)),                        # 5 to 8 columns on four wavefronts
    (768, 96, 33, 5, "", (768, 2, 1)),
    (768, 96, 33, 4, "", (768, 1, 1)),
    (768, 96, 33, 9, "", (768, 1, 1)),
    (768, 96, 33, 8, ";mapToThreads=64,8", (768, 1, 1)),
    (1023, 65, 33, 65, ";mapToThreads=64,2", (1023, 2, 2)),   # fewer than eight wavefronts a compute unit
    (1024, 65, 33, 65, ";mapToThreads=64,2", (1024, 1, 1)),
])
def test_which_products_are_taken_whole(b, n, m, k, opts, blocks):
    _, launches = tc.map_only(SOURCE, "f", [ShapeOnly((b, n, m)), ShapeOnly((b, m, k))], options(b, n, k) + opts)
    assert launches[0][0] == blocks
