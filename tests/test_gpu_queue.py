"""The item queue of the grouped GEMM kernels at the edges of its ranges: no
item, fewer items than XCD ranges, one more or less than the workgroups of
the launch, several per workgroup.  Integer products, so every launch must
give the exact result (an item left out or run twice under beta = 1 shows)."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f64", "i8x4", "bf16x3"])
@pytest.mark.parametrize("rows,cols", [(1, 1), (1, 7), (2, 4), (3, 3), (15, 17), (16, 16), (1, 257),
                                       (17, 31), (40, 52)])
def test_every_item_runs_once(precision, rows, cols):
    from tiledarray_amd import DistArray, TiledRange, TiledRange1
    from tiledarray_amd import _lib
    from tiledarray_amd import engine as E
    ctx = E.Context(0)
    w, k = 16, 5  # one 64 x 64 macro tile per result tile
    rng = np.random.default_rng(rows * 1000 + cols)
    a = rng.integers(-8, 9, (rows * w, k)).astype(np.float64)
    b = rng.integers(-8, 9, (k, cols * w)).astype(np.float64)
    tm, tn = TiledRange1.uniform(rows * w, w), TiledRange1.uniform(cols * w, w)
    tk = TiledRange1([0, k])
    A = DistArray.from_dense(a, TiledRange([tm, tk]))
    B = DistArray.from_dense(b, TiledRange([tk, tn]))
    # one workgroup per CU where the precision takes the setting: 256 of them
    c = E.Contraction(ctx, "m,n", A, "m,k", B, "k,n", precision=precision,
                      tile=(64, 64, 16, 1) if precision == "f64" else None)
    for _ in range(3):  # the counters are cleared for every launch
        c.C.fill_(float("nan"))
        c.run()
        got = c.C.cpu().numpy()
        want = np.concatenate([t.reshape(-1) for r in np.split(a @ b, rows, 0)
                               for t in np.split(r, cols, 1)])
        np.testing.assert_array_equal(got, want)
    if precision != "f64":
        return
    # every task accumulates into its tile: a second run of an item would
    # add its product twice
    tasks, _, _ = c.wl.buffers()
    n = rows * cols
    torch.cuda.synchronize()
    t = torch.empty(n * 32, dtype=torch.uint8)
    hip = ctypes.CDLL("libamdhip64.so")
    assert hip.hipMemcpy(ctypes.c_void_p(t.data_ptr()), ctypes.c_void_p(tasks),
                         ctypes.c_size_t(n * 32), 2) == 0
    t.numpy().view(np.int32).reshape(n, 8)[:, 7] |= _lib.TAMX_TASK_BETA1  # flags
    assert hip.hipMemcpy(ctypes.c_void_p(tasks), ctypes.c_void_p(t.data_ptr()),
                         ctypes.c_size_t(n * 32), 1) == 0
    c.gemm_step()
    np.testing.assert_array_equal(c.C.cpu().numpy(), 2.0 * want)
