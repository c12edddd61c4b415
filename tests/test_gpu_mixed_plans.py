"""GPU test of two plans on the mixed-radix kernels that share a kernel and take different amounts of
LDS."""
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
