"""GPU tests of plans on the mixed-radix kernels beside other plans and at their limits: two plans that
share a kernel and take different amounts of LDS, batches of more workgroups than one launch may
have, transforms in place that change the element size, what a plan reports of them, and the columns
whose number of passes depends on their pitch."""
import numpy as np
import pytest

import oracle

from .helpers import complex_input, from_device, rel_errors, to_device


@pytest.mark.gpu
@pytest.mark.parametrize("prec,first,second", [("fp32", 2176, 544), ("split_fp16", 1088, 544), ("fp32", 510, 272)])
def test_plans_that_share_a_kernel(dev, prec, first, second):
    import torch

    import fft_demo_amd as F

    dt = torch.float32 if prec == "fp32" else torch.float16
    x = complex_input((1, first, 24), 1, "c32" if prec == "fp32" else "c16")
    with F.Plan((first, 24), 1, precision=prec) as a, F.Plan((second, 24), 1, precision=prec) as b:
        b.exec(torch.zeros((1, second, 24, 2), dtype=dt, device=dev))
        y = from_device(a.exec(to_device(x, dt, dev))) / a.out_scale
    l2, mx = rel_errors(y, oracle.fft2d(x))
    assert l2 <= (1e-5 if prec == "fp32" else 1e-3) and mx <= (4e-5 if prec == "fp32" else 4e-3), (l2, mx)


@pytest.mark.gpu
def test_more_workgroups_than_a_launch_takes(dev):
    import torch

    import fft_demo_amd as F

    # one workgroup of 256 threads per transform's columns: 2^24 of them are 2^32 threads; the workspace
    # holds all, so that the batch is not cut into chunks before
    batch = (1 << 24) + 3
    base = to_device(complex_input((1024, 48, 2), 5), torch.float16, dev)
    x = base.repeat(batch // 1024 + 1, 1, 1, 1)[:batch].contiguous()
    with F.Plan((48, 2), batch, precision="split_fp16", workspace_limit=16 << 30) as plan, \
            F.Plan((48, 2), 1024, precision="split_fp16") as one:
        assert plan.info["batch_chunk"] == batch
        y = plan.exec(x)
        want = one.exec(base)
    del x
    whole = batch // 1024 * 1024
    assert torch.equal(y[:whole].view(-1, 1024, 48, 2, 2), want.expand(whole // 1024, 1024, 48, 2, 2))
    assert torch.equal(y[whole:], want[:batch - whole])


@pytest.mark.gpu
@pytest.mark.parametrize("n,batch", [(480, 3000), (1152, 901), (2304, 5), (3840, 300)])
@pytest.mark.parametrize("inf,outf", [("c16", "c32"), ("c32", "c16")])
def test_in_place_with_another_element_size(dev, n, batch, inf, outf):
    import torch

    import fft_demo_amd as F

    dt = {"c16": torch.float16, "c32": torch.float32}
    x = complex_input((batch, n), n)
    with F.Plan((n,), batch, precision="split_fp16", in_fmt=inf, out_fmt=outf) as plan:
        xd = to_device(x, dt[inf], dev)
        buf = torch.empty(batch * n * 8, dtype=torch.uint8, device=dev)  # holds either format
        buf[:xd.numel() * xd.element_size()] = xd.view(-1).view(torch.uint8)
        plan.exec_ptr(buf.data_ptr(), buf.data_ptr(), torch.cuda.current_stream(dev).cuda_stream)
        y = buf.view(dt[outf])[:2 * batch * n].view(batch, n, 2)
        scale = plan.out_scale
    l2, mx = rel_errors(from_device(y) / scale, oracle.fft(x))
    assert l2 <= 1e-3 and mx <= 4e-3, (l2, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("timed", ["events", "pass"])
def test_in_place_with_another_element_size_timed(dev, timed):
    import torch

    import fft_demo_amd as F
    from fft_demo_amd import _lib, hiptime

    lib = _lib.load()
    n, batch = 480, 3000
    x = complex_input((batch, n), n)
    with F.Plan((n,), batch, precision="split_fp16", in_fmt="c32", out_fmt="c16") as plan:
        want = from_device(plan.exec(to_device(x, torch.float32, dev)))
        buf = to_device(x, torch.float32, dev)
        s, ptr, pool = torch.cuda.current_stream(dev).cuda_stream, buf.data_ptr(), hiptime.EventPool(2)
        if timed == "events":
            assert lib.mfft_exec_events(plan._h, ptr, ptr, s, pool.slice(0), 2) == 0
        else:
            assert lib.mfft_exec_pass(plan._h, 0, ptr, ptr, s, pool.arr[0], pool.arr[1]) == 0
        assert pool.elapsed_ms(0, 1) > 0
        y = from_device(buf.view(torch.float16).view(-1)[:2 * batch * n].view(batch, n, 2))
        pool.close()
    l2, mx = rel_errors(y, want)
    assert l2 <= 1e-3 and mx <= 4e-3, (l2, mx)


@pytest.mark.gpu
def test_reported_passes(dev):
    import fft_demo_amd as F

    with F.Plan((1200,), 3001, precision="split_fp16") as plan:
        (p,) = plan.info["passes"]
        assert p["kernel"] == "mixed_rows" and p["lines_per_tile"] == 3 and p["tiles"] == 1001
    with F.Plan((48, 300), 5, precision="split_fp16") as plan:  # 5 x 48 rows, 5 x 300 columns
        rows, cols = plan.info["passes"]
        assert rows["kernel"] == "mixed_rows" and rows["lines_per_tile"] * rows["tiles"] >= 240
        assert cols["kernel"] == "mixed_cols" and cols["lines_per_tile"] == 8 and cols["tiles"] == 5 * 38


@pytest.mark.gpu
@pytest.mark.parametrize("prec", ["fp32", "split_fp16", "bf16"])
@pytest.mark.parametrize("nx,ny,batch", [(48, 16, 1), (48, 16, 700), (60, 32, 3), (60, 34, 3), (68, 32, 3), (1020, 2, 5),
                                         (1020, 3, 2), (24, 2, 33)])
def test_columns_of_small_tiles(dev, prec, nx, ny, batch):
    import torch

    import fft_demo_amd as F

    fmt = {"fp32": "c32", "split_fp16": "c16", "bf16": "cbf16"}[prec]
    x = complex_input((batch, nx, ny), nx + ny, fmt)
    with F.Plan((nx, ny), batch, precision=prec) as plan:
        assert plan.info["passes"][-1]["kernel"] == "mixed_cols"
        y = from_device(plan.exec(to_device(x, plan.in_dtype(), dev))) / plan.out_scale
    l2, mx = rel_errors(y, oracle.fft2d(x))
    tol = {"fp32": (1e-5, 4e-5), "split_fp16": (1e-3, 4e-3), "bf16": (1e-2, 4e-2)}[prec]
    assert l2 <= tol[0] and mx <= tol[1], (l2, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("ny,passes", [(1024, 2), (2048, 3)])  # one pass of columns; at a wide pitch two
def test_columns_of_1088_points(dev, ny, passes):
    import torch

    import fft_demo_amd as F

    x = complex_input((1, 1088, ny), ny)
    with F.Plan((1088, ny), 1, precision="split_fp16", mid_fmt="c16") as plan:
        assert len(plan.info["passes"]) == passes
        y = from_device(plan.exec(to_device(x, torch.float16, dev))) / plan.out_scale
    l2, mx = rel_errors(y, oracle.fft2d(x))
    assert l2 <= 1e-3 and mx <= 4e-3, (l2, mx)
