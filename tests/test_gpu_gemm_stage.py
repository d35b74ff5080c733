"""Staging of the plain grouped GEMM at its edges, through the C ABI on
hand-built work lists: results one block past and short of every tile of the
macro tile in both directions, several pairs with k around a chunk and a
staged unit (odd k, k of one), tile offsets of every residue of the 16-byte
units, and values of infinity and NaN that lie next to the operands in the
pool but in no operand.  Integer data make every sum exact, so results are
compared bit for bit with torch."""
import ctypes

import pytest
import torch

from tiledarray_amd import _lib
from tiledarray_amd import engine as E
from test_gpu_gemm_edges import hip

pytestmark = pytest.mark.gpu


def run_pairs(ctx, dtype, op_a, op_b, m, n, ks, shift, tile, fence):
    """One task of len(ks) pairs; every stored tile lies in the pool with
    `fence` elements of infinity and NaN around it."""
    g = torch.Generator(device="cuda").manual_seed(m * 7919 + n * 104729 + sum(ks) + shift)
    bad = torch.tensor([float("inf"), float("nan"), -float("inf")], dtype=dtype, device="cuda")

    def fenced(parts):
        pool, offs, at = [bad.repeat(fence)[: fence + shift]], [], fence + shift
        for x in parts:
            offs.append(at)
            pool += [x.reshape(-1), bad.repeat(fence)[:fence]]
            at += x.numel() + fence
        return torch.cat(pool), offs

    def rnd(r, c):
        return torch.randint(-3, 4, (r, c), dtype=torch.int32, device="cuda", generator=g).to(dtype)

    As = [rnd(k, m) if op_a else rnd(m, k) for k in ks]
    Bs = [rnd(n, k) if op_b else rnd(k, n) for k in ks]
    A, aoff = fenced(As)
    B, boff = fenced(Bs)
    C = torch.full((m * n,), 7.0, dtype=dtype, device="cuda")
    wl = E.WorkList(ctx, 4, len(ks), 4096)
    tasks, pairs, counters = wl.buffers()
    task = _lib.GemmTask(0, m, n, n, 0, len(ks), 0)
    pr = (_lib.GemmPair * len(ks))(*[
        _lib.GemmPair(aoff[i], boff[i], k, m if op_a else k, k if op_b else n, 0, 0, 0)
        for i, k in enumerate(ks)])
    cnt = (ctypes.c_int64 * 8)(1, len(ks), m * n, 0, 0, 0, 0, 0)
    for dst, src in ((tasks, task), (pairs, pr), (counters, cnt)):
        assert hip().hipMemcpy(dst, ctypes.byref(src), ctypes.sizeof(src), 1) == 0
    cfg = _lib.GemmConfig(*tile, 0)
    f64 = dtype == torch.float64
    E.call("tamx_grouped_gemm_f64_config" if f64 else "tamx_grouped_gemm_f32_config",
           ctx.ptr, wl.ptr, op_a, op_b, ctypes.c_double(1.0) if f64 else ctypes.c_float(1.0),
           A.data_ptr(), B.data_ptr(), C.data_ptr(), ctypes.byref(cfg), ctx.stream())
    torch.cuda.synchronize()
    ref = sum((a.double().t() if op_a else a.double()).cpu() @ (b.double().t() if op_b else b.double()).cpu()
              for a, b in zip(As, Bs)).to(dtype)
    return C.view(m, n).cpu(), ref


TILES = [(64, 64, 16), (64, 64, 32), (128, 128, 16), (128, 64, 16), (64, 128, 16), (32, 32, 16),
         (32, 32, 32), (128, 64, 32), (64, 128, 32)]


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32], ids=["f64", "f32"])
@pytest.mark.parametrize("ops", [(0, 0), (1, 0), (0, 1), (1, 1)], ids=["NN", "TN", "NT", "TT"])
@pytest.mark.parametrize("tile", TILES, ids=lambda t: "x".join(map(str, t)))
def test_edges_and_neighbours(ctx, dtype, ops, tile):
    bm, bn, bk = tile
    shapes = [(bm, bn), (bm + 1, bn - 1), (bm - 17, bn + 16), (1, 2), (9 * bm + 5, 3)]
    for i, (m, n) in enumerate(shapes):
        ks = [[bk], [1, bk - 1, bk + 3], [2 * bk + 1, 5], [bk + 2, 2, 3 * bk]][i % 4]
        C, ref = run_pairs(ctx, dtype, *ops, m, n, ks, i % 4, tile, 3 * (i % 3) + 3)
        assert torch.equal(C, ref), (m, n, ks)
