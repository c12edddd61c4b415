"""GPU tests of the mixed-radix kernels (lengths 2^a 3^b 5^c 17^d up to 4096): every radix as a
first, middle and last stage, partial tiles, in place, 16- and 32-bit ends, and the work queue
with few items, more items than its arguments hold and more tiles than its grid."""
import ctypes

import numpy as np
import pytest

import oracle

from .helpers import complex_input, from_device, rel_errors, to_device

TOL = {"split_fp16": (1e-3, 4e-3), "fp16": (4e-3, 2e-2), "bf16": (3e-2, 1e-1), "fp32": (1e-5, 4e-5)}
# 15 5 16 | 17 17 2 | 9 9 9 3 | 5 5 5 5 5 | 15 15 ... | 17 15 16 | 12 10 | 10 10 | one stage (15, 17) | largest
LENGTHS = [1200, 578, 2187, 3125, 450, 4080, 120, 100, 15, 17, 4050, 1530, 1000, 75]


def _dtype(prec):
    import torch

    return {"split_fp16": torch.float16, "fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}[prec]


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(TOL))
@pytest.mark.parametrize("n", LENGTHS)
def test_mixed_rows(dev, prec, n):
    import fft_demo_amd as F

    fmt = {"bf16": "cbf16", "fp32": "c32"}.get(prec, "c16")
    for batch, inverse in ((1, False), (2600, True)):  # one line; several lines per tile, the last tile partial
        x = complex_input((batch, n), n + batch, fmt)
        with F.Plan((n,), batch, precision=prec, direction=F.INVERSE if inverse else F.FORWARD) as plan:
            xd = to_device(x, _dtype(prec), dev)
            y = from_device(plan.exec(xd, out=xd)) / plan.out_scale  # in place
        ref = oracle.fft(x.conj()).conj() if inverse else oracle.fft(x)
        l2, mx = rel_errors(y, ref)
        assert l2 <= TOL[prec][0] and mx <= TOL[prec][1], (batch, l2, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("inf,outf", [("c16", "c32"), ("c32", "c16"), ("c32", "c32")])
def test_mixed_rows_32bit_ends(dev, inf, outf):
    import torch

    import fft_demo_amd as F

    x = complex_input((7, 1200), 3)
    with F.Plan((1200,), 7, precision="split_fp16", in_fmt=inf, out_fmt=outf) as plan:
        xd = to_device(x, torch.float32 if inf == "c32" else torch.float16, dev)
        y = from_device(plan.exec(xd)) / plan.out_scale
    l2, mx = rel_errors(y, oracle.fft(x))
    assert l2 <= 1e-3 and mx <= 4e-3, (l2, mx)


@pytest.mark.gpu
def test_mixed_rows_of_a_2d_plan(dev):
    import torch

    import fft_demo_amd as F

    x = complex_input((3, 64, 720), 4)
    with F.Plan((64, 720), 3, precision="split_fp16") as plan:
        y = from_device(plan.exec(to_device(x, torch.float16, dev))) / plan.out_scale
    l2, mx = rel_errors(y, oracle.fft2d(x))
    assert l2 <= 1e-3 and mx <= 4e-3, (l2, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(TOL))
@pytest.mark.parametrize("what", ["few", "many_items", "many_tiles"])
def test_queue(dev, prec, what):
    import torch

    import fft_demo_amd as F
    from fft_demo_amd import _lib as L

    cases = {"few": [(2, 3), (16, 700), (4096, 3), (1200, 5), (17, 9), (512, 40), (8, 1), (2187, 2)],
             "many_items": [((16, 48, 100, 256, 1530)[i % 5], 1 + i % 7) for i in range(70)],
             "many_tiles": [(4096, 900), (1024, 33), (3125, 400)]}[what]
    lib = L.load()
    desc = F.make_desc(precision=prec)
    bh = ctypes.c_void_p()
    L.check(lib.mfft_batcher_create(ctypes.byref(bh), ctypes.byref(desc), len(cases)), "batcher")
    fmt = {"bf16": "cbf16", "fp32": "c32"}.get(prec, "c16")
    data, items = [], (L.BatchItem * len(cases))()
    for i, (n, c) in enumerate(cases):
        x = complex_input((c, n), 70 + i, fmt)
        xd = to_device(x, _dtype(prec), dev)
        od = torch.zeros_like(xd)
        data.append((x, xd, od))
        items[i].in_, items[i].out, items[i].n, items[i].count = xd.data_ptr(), od.data_ptr(), n, c
    s = torch.cuda.current_stream(dev)
    for rep in range(6):  # every slot more than once: the counters start from zero each time
        if rep == 5:
            for _, _, od in data:
                od.zero_()
        L.check(lib.mfft_batcher_exec(bh, items, len(cases), ctypes.c_void_p(s.cuda_stream)), "exec")
    torch.cuda.synchronize()
    for (n, c), (x, _, od) in zip(cases, data):
        y = from_device(od) * (n if prec == "split_fp16" else 1)
        l2, mx = rel_errors(y, oracle.fft(x))
        assert l2 <= TOL[prec][0] and mx <= TOL[prec][1], (n, c, l2, mx)
    lib.mfft_batcher_destroy(bh)


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(TOL))
@pytest.mark.parametrize("nx,ny,b", [(96, 80, 3),       # 32 lines a tile, partial last tile
                                     (480, 100, 2),     # 16 lines a tile, 4 in the last
                                     (1088, 64, 2),     # the large tile, full
                                     (2176, 72, 1),     # 8 lines a tile
                                     (272, 5, 2)])      # fewer lines than a tile
def test_mixed_columns(dev, prec, nx, ny, b):
    import fft_demo_amd as F

    fmt = {"bf16": "cbf16", "fp32": "c32"}.get(prec, "c16")
    x = complex_input((b, nx, ny), nx + ny, fmt)
    for inverse in (False, True):
        with F.Plan((nx, ny), b, precision=prec, direction=F.INVERSE if inverse else F.FORWARD) as plan:
            assert len(plan.info["passes"]) == 2 or (nx > 1088 and prec != "fp32")
            xd = to_device(x, _dtype(prec), dev)
            y = from_device(plan.exec(xd, out=xd)) / plan.out_scale  # in place
        ref = oracle.fft2d(x.conj()).conj() if inverse else oracle.fft2d(x)
        l2, mx = rel_errors(y, ref)
        assert l2 <= TOL[prec][0] and mx <= TOL[prec][1], (inverse, l2, mx)
