"""The default split GEMM (64 x 64 macro tiles, chunks multiplied out of
registers) at its edges: result tiles one row past and short of every block
of the macro tile, contracted extents around a chunk and half of one, pairs
longer than a fold joins (448 k) and result tiles of more than 64 pairs.
Integer data are split exactly and every sum is exact, so results are
compared bit for bit with the oracle; on random data the other split kernels
must give the same bits."""
import numpy as np
import pytest
import torch

from tiledarray_amd import TiledRange1
from tiledarray_amd import engine as E
from test_gpu_contract import c_off_mask, matrix_ops_arrays, oracle_contract

pytestmark = pytest.mark.gpu

ROWS = TiledRange1(np.cumsum([0, 1, 15, 16, 17, 32, 33, 48, 49, 64, 65, 100]))
COLS = TiledRange1(np.cumsum([0, 65, 31, 64, 1, 47, 16, 129]))
# chunk edges, then more pairs than one descriptor table holds, then folds
K_MIXED = TiledRange1(np.cumsum([0, 1, 31, 32, 33, 63, 64, 65, 97] + [3] * 70 + [448, 449, 700]))
PRECISIONS = [f"{t}x{s}" for t in ("i8", "bf16") for s in range(2, 7)]


@pytest.mark.parametrize("precision", PRECISIONS)
def test_staged_integer_exact(ctx, precision):
    rng = np.random.default_rng(4100 + PRECISIONS.index(precision))
    A, B = matrix_ops_arrays(rng, ROWS, K_MIXED, COLS, 0, 1, torch.float64, True, fill=0.9)
    c = E.Contraction(ctx, "m,n", A, "m,k", B, "n,k", alpha=2.0, precision=precision)
    c.run()
    torch.cuda.synchronize()
    Cref, _, c_off = oracle_contract(c, A, B)
    mask = c_off_mask(c_off, c)
    np.testing.assert_array_equal(c.C.cpu().numpy()[mask], Cref[mask])


@pytest.mark.parametrize("exponent", [0, -480])
@pytest.mark.parametrize("precision", PRECISIONS[:5] + PRECISIONS[5:8])
def test_staged_same_bits(ctx, precision, exponent):
    # exponent -480: scales below the range in which a fold joins the levels
    rng = np.random.default_rng(4200 + PRECISIONS.index(precision))
    A, B = matrix_ops_arrays(rng, ROWS, K_MIXED, COLS, 0, 1, torch.float64, True, fill=0.9)
    for X in (A, B):
        X.pool.copy_(torch.as_tensor(rng.standard_normal(X.pool.numel())))
        X.pool.mul_(2.0 ** exponent)
    c = E.Contraction(ctx, "m,n", A, "m,k", B, "n,k", precision=precision)
    c.run()
    torch.cuda.synchronize()
    C0 = c.C.clone()
    c.set_tile((64, 64, 32) if precision.startswith("i8") else (128, 64))
    c.C.zero_()
    c.gemm_step()
    torch.cuda.synchronize()
    mask = torch.as_tensor(c_off_mask(c.c_off.cpu().numpy(), c), device="cuda")
    assert torch.equal(c.C[:mask.numel()][mask], C0[:mask.numel()][mask])
    assert bool(C0[:mask.numel()][mask].ne(0).any())
