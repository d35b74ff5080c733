"""The macro tile the library picks by itself: FP32 chunks of 32 k, and 128 x
128 for FP64 results whose tiles are many macro tiles wide, give the same
bits as 64 x 64 x 16, which adds the same products in the same order."""
import numpy as np
import pytest
import torch

from tiledarray_amd import TiledRange1
from tiledarray_amd import engine as E
from test_gpu_contract import matrix_ops_arrays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("op_a,op_b", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("dtype,rows,cols", [
    (torch.float32, [1, 63, 64, 65, 129], [17, 100, 128]),
    # four result tiles of 2000 x 1999 elements and up: above the mean size and
    # with 3.9 items of 128 x 128 a CU, so that macro tile is taken
    (torch.float64, [2047, 2000], [2050, 1999]),
])
def test_default_macro_tile_same_bits(ctx, dtype, rows, cols, op_a, op_b):
    rng = np.random.default_rng(4300 + op_a * 2 + op_b)
    trm, trn = TiledRange1(np.cumsum([0] + rows)), TiledRange1(np.cumsum([0] + cols))
    trk = TiledRange1(np.cumsum([0, 1, 15, 31, 33, 64]))
    A, B = matrix_ops_arrays(rng, trm, trk, trn, op_a, op_b, dtype, False, fill=0.9)
    c = E.Contraction(ctx, "m,n", A, "k,m" if op_a else "m,k", B, "n,k" if op_b else "k,n",
                      precision="f32" if dtype == torch.float32 else "f64")
    c.run()
    torch.cuda.synchronize()
    C0 = c.C.clone()
    c.set_tile((64, 64, 16))
    c.C.zero_()
    c.gemm_step()
    torch.cuda.synchronize()
    assert torch.equal(c.C, C0)
    assert bool(C0.ne(0).any())
