"""The split GEMM at tiles around 2 GB of limbs, where the kernel with 32-bit
offsets inside a tile (the largest of them) hands over to those with 64-bit
addresses.  Integer data are split exactly and every sum is exact, so both
sides are compared bit for bit with a FP64 product; on random data the limbs
in one tile above the limit and in two tiles below it give the same bits."""
import pytest
import torch

from tiledarray_amd import DistArray, TiledRange, TiledRange1
from tiledarray_amd import engine as E

pytestmark = pytest.mark.gpu

LIMIT = 1 << 31  # bytes of limbs of a tile
ROWS, COLS = 1040, 33  # a last macro tile of one 16-row block; ragged columns
PRECISIONS = [f"{t}x{s}" for t in ("i8", "bf16") for s in range(2, 7)]


def extents(precision):
    """The largest k with less than LIMIT bytes of limbs, the next with more."""
    quantum, size = (64, 1) if precision.startswith("i8") else (32, 2)
    per_k = int(precision.split("x")[1]) * size * ROWS
    below = (LIMIT - 1) // per_k // quantum * quantum
    assert below * per_k < LIMIT <= (below + quantum) * per_k
    return below, below + quantum


def product(ctx, pool, rows, k, b, precision):
    """C = A B^T of the `rows`-tiled A in `pool` and the one-tile b."""
    tk = TiledRange1([0, k])
    A = DistArray(TiledRange([rows, tk]), pool, k * rows.boundaries[:-1])
    B = DistArray(TiledRange([TiledRange1([0, COLS]), tk]), b, [0])
    c = E.Contraction(ctx, "m,n", A, "m,k", B, "n,k", precision=precision)
    c.run()
    torch.cuda.synchronize()
    return c.C.view(ROWS, COLS)


@pytest.mark.parametrize("precision", PRECISIONS)
def test_integer_exact_on_both_sides_of_the_limit(ctx, precision):
    for n, k in enumerate(extents(precision)):
        g = torch.Generator(device="cuda").manual_seed(5100 + 2 * PRECISIONS.index(precision) + n)
        rnd = lambda count: torch.randint(-8, 9, (count,), dtype=torch.int8, device="cuda",
                                          generator=g).double()
        a, b = rnd(ROWS * k), rnd(COLS * k)
        C = product(ctx, a, TiledRange1([0, ROWS]), k, b, precision)
        assert torch.equal(C, a.view(ROWS, k) @ b.view(COLS, k).t().contiguous()), k


@pytest.mark.parametrize("precision", PRECISIONS)
def test_same_bits_on_both_sides_of_the_limit(ctx, precision):
    k = extents(precision)[1]
    g = torch.Generator(device="cuda").manual_seed(5200 + PRECISIONS.index(precision))
    rnd = lambda count: torch.rand(count, dtype=torch.float64, device="cuda", generator=g) - 0.5
    a, b = rnd(ROWS * k), rnd(COLS * k)
    half = ROWS // 2 // 16 * 16
    a.view(ROWS, k)[[0, half], 5] = 0.75  # the same scale in every tile
    one = product(ctx, a, TiledRange1([0, ROWS]), k, b, precision)
    two = product(ctx, a, TiledRange1([0, half, ROWS]), k, b, precision)
    assert torch.equal(one, two)
    assert bool(one.ne(0).all())
