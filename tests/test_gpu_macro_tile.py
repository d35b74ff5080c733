"""The macro tile of an FP64 or FP32 product without a configuration: which
one runs, by the extents of the result tiles that are there and not by the
size of the result buffer, found out anew in every pass, with the bits of an
explicit 64 x 64."""
import pytest
import torch

from tiledarray_amd import DistArray, TiledRange, TiledRange1
from tiledarray_amd import engine as E

pytestmark = pytest.mark.gpu

F64, F32 = (64, 64, 16), (64, 64, 32)
WIDE = (128, 128, 16)
K = 24


def product(ctx, rows, cols, dtype=torch.float64, threshold=None):
    """C(m,n) over K, result tiles of all `rows` x `cols` combinations."""
    g = torch.Generator(device="cuda").manual_seed(len(rows) * 31 + len(cols) + rows[0])
    ext = lambda x: TiledRange1([0] + torch.cumsum(torch.tensor(x), 0).tolist())
    tm, tn, tk = ext(rows), ext(cols), TiledRange1([0, K])
    A = DistArray.allocate(TiledRange([tm, tk]), dtype=dtype)
    B = DistArray.allocate(TiledRange([tk, tn]), dtype=dtype)
    for X in (A, B):
        X.pool.copy_(torch.rand(X.pool.numel(), dtype=dtype, device="cuda", generator=g) - 0.5)
        if threshold is not None:
            E.make_sparse(ctx, X, threshold)
    kw = {} if threshold is None else {"threshold": threshold}
    return E.Contraction(ctx, "m,n", A, "m,k", B, "k,n",
                         precision="f64" if dtype == torch.float64 else "f32", **kw)


def check(c, expected):
    c.run()
    assert c.macro_tile() == expected
    C0 = c.C.clone()
    c.set_tile(F64)
    c.C.zero_()
    c.gemm_step()
    assert c.macro_tile() == F64
    c.set_tile(None)
    assert torch.equal(c.C, C0) and bool(C0.ne(0).any())


@pytest.mark.parametrize("rows,cols,expected", [
    ([256] * 16, [1024] * 4, WIDE),
    ([4096], [4096], WIDE),
    ([2047, 2000], [2040, 1999], WIDE),
    ([2047, 2000], [2050, 1999], F64),  # just above four items a CU
    ([225] * 4, [5625] * 4, WIDE),  # 225 = 128 + 97: no more blocks than in 64s
    ([2048], [2048], F64),          # one item a CU
    ([320] * 13, [320] * 13, F64),  # half-filled macro tiles
    ([300] * 10, [3500] * 2, F64),
    ([36] * 200, [4096] * 2, F64),  # flat
    ([4096] * 2, [36] * 200, F64),
    ([128] * 32, [4096], F64),
    ([64, 100], [100], F64),
], ids=lambda x: None if isinstance(x, tuple) else "%dx%d" % (len(x), x[0]))
def test_choice_by_the_extents(ctx, rows, cols, expected):
    check(product(ctx, rows, cols), expected)


def test_single_precision(ctx):
    c = product(ctx, [1024] * 4, [1024] * 4, torch.float32)
    c.run()
    assert c.macro_tile() == F32


@pytest.mark.parametrize("rows,cols,expected", [([512] * 8, [512] * 8, WIDE), ([512] * 2, [512], F64)])
def test_choice_regardless_of_the_buffer(ctx, rows, cols, expected):
    c = product(ctx, rows, cols)
    c.c_capacity *= 8
    c.C = torch.zeros(c.c_capacity, dtype=torch.float64, device="cuda")
    c._desc.c_capacity = c.c_capacity
    check(c, expected)


def test_choice_by_what_the_screening_leaves(ctx):
    # the same object and graph, first with all result tiles, then with the
    # first column of them only, then with all again
    c = product(ctx, [512] * 8, [512] * 8, threshold=1e-6)
    norms = c.B.shape_norms.clone()
    graph = E.Graph(ctx, c.run)
    for factor, expected in ((1.0, WIDE), (0.0, F64), (1.0, WIDE)):
        c.B.shape_norms.copy_(norms)
        c.B.shape_norms[1:].mul_(factor)
        graph.replay()
        torch.cuda.synchronize()
        assert c.counters()["ntasks"] == (64 if factor else 8)
        n = c.counters()["celems"]
        C0 = c.C[:n].clone()
        c.C.zero_()
        c.run()
        assert c.macro_tile() == expected
        assert torch.equal(c.C[:n], C0)
        c.set_tile(F64)
        c.C.zero_()
        c.gemm_step()
        c.set_tile(None)
        assert torch.equal(c.C[:n], C0) and bool(C0.ne(0).any())


def test_no_launch_yet_and_a_refused_one(ctx):
    c = product(ctx, [64], [64])
    with pytest.raises(E._lib.TamxError):
        c.macro_tile()
    c.run()
    c.set_tile((48, 64, 16))
    with pytest.raises(E._lib.TamxError):
        c.gemm_step()
    assert c.macro_tile() == F64
