"""GPU tests of merged line groups (the second pass of lengths odd * 2^a) at batches whose own tiles
exceed what runs at once, told by the launch trace: tiles that span two or more groups, a partial last
tile, full and small tiles, each against the same lines in a batch too small to merge, bit for bit."""
import ctypes

import pytest

from .helpers import complex_input, to_device

FMT = {"split_fp16": "c16", "fp16": "c16", "bf16": "cbf16", "fp32": "c32"}


def _exec(plan, x):
    """Output and the names of the launches."""
    import torch

    from fft_demo_amd import _lib as L
    from fft_demo_amd.hiptime import EventPool

    lib, cap = L.load(), 16
    recs, pool, n = (L.LaunchRecord * cap)(), EventPool(cap + 1), ctypes.c_int()
    L.check(lib.mfft_trace_begin(pool.arr, recs, cap), "mfft_trace_begin")
    y = plan.exec(x)
    L.check(lib.mfft_trace_end(ctypes.c_void_p(torch.cuda.current_stream().cuda_stream), ctypes.byref(n)), "mfft_trace_end")
    torch.cuda.synchronize()
    pool.close()
    return y, [recs[i].kernel.decode() for i in range(n.value)]


def _check(dev, n, batch, want, in_fmt=None, **desc):
    import torch

    import fft_demo_amd as F

    fmt = in_fmt or FMT[desc["precision"]]
    few, reps = 7, -(-batch // 7)
    dt = {"c16": torch.float16, "cbf16": torch.bfloat16, "c32": torch.float32}[fmt]
    base = to_device(complex_input((few, n), n, fmt), dt, dev)
    x = base.repeat(reps, 1, 1)[:batch].contiguous()
    fm = dict(in_fmt=in_fmt, out_fmt=in_fmt) if in_fmt else {}
    for inverse in (False, True):
        d = dict(direction=F.INVERSE if inverse else F.FORWARD, workspace_limit=4 << 30, **fm, **desc)
        with F.Plan((n,), batch, **d) as plan, F.Plan((n,), few, **d) as small:
            y, names = _exec(plan, x)
            ref, own = _exec(small, base)
        assert len(names) == 2 and ("merged" in names[1]) == want and "merged" not in own[1], (names, own)
        assert torch.equal(y, ref.repeat(reps, 1, 1)[:batch])


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(FMT))
@pytest.mark.parametrize("n,batch", [(6144, 1801), (5120, 1701), (4608, 1801), (7680, 1303), (8704, 1203), (4352, 1801)])
def test_matrix_core_rows(dev, prec, n, batch):
    # lines a group / lines a tile: 3/2, 5/4, 9/8, 15/8, 17/8, 17/16
    _check(dev, n, batch, True, precision=prec)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(FMT))
@pytest.mark.parametrize("batch", [900, 50003])  # small tiles; full ones
@pytest.mark.parametrize("n", [96, 80, 288, 480, 272])
def test_tile_kernel_rows(dev, prec, n, batch):
    _check(dev, n, batch, True, precision=prec, split_hint=2)  # the two passes that the planner would make one


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch,want", [(192, 6001, True), (192, 700, False), (1152, 4001, True), (3072, 1000, False)])
def test_tile_kernel_rows_of_longer_lines(dev, n, batch, want):
    # fp16 arithmetic on 32-bit words has no matrix-core row kernel
    _check(dev, n, batch, want, in_fmt="c32", precision="fp16", split_hint=2)
