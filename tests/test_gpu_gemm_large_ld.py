"""Leading dimensions around the largest that the plain grouped GEMM stages
through 32-bit offsets and well above it, where units have 64-bit addresses:
several loads of rows, ragged rows, columns and k, the pool ending with the
last row's last element and NaN between the rows.  Integer data make every
sum exact, so results are compared bit for bit."""
import ctypes

import pytest
import torch

from tiledarray_amd import _lib
from tiledarray_amd import engine as E
from test_gpu_gemm_edges import hip

pytestmark = pytest.mark.gpu


def strided(x, ld):
    """The rows of x `ld` elements apart, eight NaN after each but the last."""
    rows, cols = x.shape
    pool = torch.empty((rows - 1) * ld + cols, dtype=x.dtype, device="cuda")
    for r in range(rows):
        pool[r * ld:r * ld + cols] = x[r]
        pool[r * ld + cols:r * ld + cols + 8] = float("nan")
    return pool


def gemm(ctx, dtype, ops, m, n, pairs, pools, tile):
    """One task over `pairs`: (a_off, b_off, k, lda, ldb)."""
    C = torch.full((m * n,), 7.0, dtype=dtype, device="cuda")
    wl = E.WorkList(ctx, 4, len(pairs), 4096)
    tasks, ppairs, counters = wl.buffers()
    task = _lib.GemmTask(0, m, n, n, 0, len(pairs), 0)
    pr = (_lib.GemmPair * len(pairs))(*[_lib.GemmPair(*p, 0, 0, 0) for p in pairs])
    cnt = (ctypes.c_int64 * 8)(1, len(pairs), m * n, 0, 0, 0, 0, 0)
    for dst, src in ((tasks, task), (ppairs, pr), (counters, cnt)):
        assert hip().hipMemcpy(dst, ctypes.byref(src), ctypes.sizeof(src), 1) == 0
    cfg = _lib.GemmConfig(*tile, 0)
    f64 = dtype == torch.float64
    E.call("tamx_grouped_gemm_f64_config" if f64 else "tamx_grouped_gemm_f32_config",
           ctx.ptr, wl.ptr, *ops, ctypes.c_double(1.0) if f64 else ctypes.c_float(1.0),
           pools[0].data_ptr(), pools[1].data_ptr(), C.data_ptr(), ctypes.byref(cfg), ctx.stream())
    torch.cuda.synchronize()
    return C.view(m, n).cpu()


def operands(g, dtype, ops, m, n, k):
    rnd = lambda r, c: torch.randint(-3, 4, (r, c), dtype=torch.int32, device="cuda",
                                     generator=g).to(dtype)
    return rnd(*((k, m) if ops[0] else (m, k))), rnd(*((n, k) if ops[1] else (k, n)))


def reference(a, b, ops):
    return (a.t() if ops[0] else a).double().cpu() @ (b.t() if ops[1] else b).double().cpu()


OPS = pytest.mark.parametrize("ops", [(0, 0), (1, 0), (0, 1), (1, 1)],
                              ids=["NN", "TN", "NT", "TT"])
DTYPES = pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])


@DTYPES
@OPS
@pytest.mark.parametrize("tile", [(64, 64, 16), (64, 64, 32), (128, 128, 16), (32, 32, 32)],
                         ids=lambda t: "x".join(map(str, t)))
@pytest.mark.parametrize("ld,m,n,k", [((1 << 20) + 1, 131, 70, 33),
                                      # the limit with k contiguous, 64 and 32 rows
                                      (1 << 22, 65, 9, 19), ((1 << 22) + 1, 70, 37, 35),
                                      ((1 << 23) + 3, 37, 66, 33), ((1 << 24) + 2, 7, 21, 18),
                                      # the limit with rows contiguous, 32 and 16 k
                                      (1 << 24, 3, 5, 33), ((1 << 25) + 1, 9, 11, 19)])
def test_large_leading_dimension(ctx, dtype, ops, tile, ld, m, n, k):
    g = torch.Generator(device="cuda").manual_seed(ld % 97 + m + n + k)
    a, b = operands(g, dtype, ops, m, n, k)
    C = gemm(ctx, dtype, ops, m, n, [(0, 0, k, ld, ld)], (strided(a, ld), strided(b, ld)), tile)
    assert torch.equal(C, reference(a, b, ops).to(dtype))


@DTYPES
@OPS
@pytest.mark.parametrize("far", [0, 1, 2])
def test_large_leading_dimension_among_others(ctx, dtype, ops, far):
    # pair `far` of three has one, in A or in B: the sum starts anew there
    m, n, ks = 70, 67, (33, 18, 40)
    g = torch.Generator(device="cuda").manual_seed(6100 + far)
    pairs, pools, offs, ref = [], ([], []), [0, 0], 0
    for i, k in enumerate(ks):
        ab = operands(g, dtype, ops, m, n, k)
        ref = ref + reference(*ab, ops)
        lds = [(1 << 25) + 1 if i == far and w == far % 2 else x.shape[1] for w, x in enumerate(ab)]
        pairs.append((*offs, k, *lds))
        for w in range(2):
            x = strided(ab[w], lds[w]) if lds[w] != ab[w].shape[1] else ab[w].reshape(-1)
            pools[w].append(x)
            offs[w] += x.numel()
    C = gemm(ctx, dtype, ops, m, n, pairs, [torch.cat(p) for p in pools], (64, 64, 16))
    assert torch.equal(C, ref.to(dtype))
