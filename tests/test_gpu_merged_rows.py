"""GPU tests of the transposed-store row kernels (matrix-core and, for 16 and 32 points, tile kernels) on
merged line groups (the second pass of lengths odd * 2^a): tiles that span two or more groups, a partial last tile, one group alone, every precision, the
three-level form of the conv operator's rows against the same operator on single images."""
import pytest

import oracle

from .helpers import complex_input, from_device, rel_errors, to_device

TOL = {"split_fp16": (1e-3, 4e-3), "fp16": (4e-3, 2e-2), "bf16": (3e-2, 1e-1), "fp32": (1e-5, 4e-5)}


@pytest.mark.gpu
@pytest.mark.parametrize("prec", list(TOL))
@pytest.mark.parametrize("n,batch", [(4352, 1), (4352, 7), (4608, 33), (5120, 5), (6144, 3), (7680, 2), (8704, 9), (3 * 4096, 2)])
def test_merged_rows(dev, prec, n, batch):
    import torch

    import fft_demo_amd as F

    fmt = {"bf16": "cbf16", "fp32": "c32"}.get(prec, "c16")
    dt = {"split_fp16": torch.float16, "fp16": torch.float16, "bf16": torch.bfloat16, "fp32": torch.float32}[prec]
    x = complex_input((batch, n), n + batch, fmt)
    for inverse in (False, True):
        with F.Plan((n,), batch, precision=prec, direction=F.INVERSE if inverse else F.FORWARD) as plan:
            y = from_device(plan.exec(to_device(x, dt, dev))) / plan.out_scale
        ref = oracle.fft(x.conj()).conj() if inverse else oracle.fft(x)
        l2, mx = rel_errors(y, ref)
        assert l2 <= TOL[prec][0] and mx <= TOL[prec][1], (inverse, l2, mx)


@pytest.mark.gpu
@pytest.mark.parametrize("pad", [(64, 192), (72, 320), (128, 576), (64, 960), (96, 1088), (64, 1536),
                                 (64, 48), (40, 80), (64, 272), (48, 96), (64, 480), (36, 544), (4096, 480)])
@pytest.mark.parametrize("option", [{}, {"mid_fp16": True}, {"spec_fp16": True}])
def test_merged_rows_of_the_conv(dev, pad, option):
    import torch

    from fft_demo_amd.conv import Conv2d

    g = torch.Generator(device=dev)
    g.manual_seed(5)
    h, w = pad[0] - 4, pad[1] - 8
    x = torch.rand((6, 1, h, w), generator=g, device=dev)
    f = torch.rand((1, 1, 5, 9), generator=g, device=dev)
    op, one = (Conv2d(b, 1, 1, h, w, 5, 9, mode="same", pad=pad, **option) for b in (6, 2))
    op.set_filters(f)
    one.set_filters(f)
    y = op.forward(x)
    for i in range(0, 6, 2):
        assert torch.equal(y[i:i + 2], one.forward(x[i:i + 2]))
    ref = torch.fft.irfft2(torch.fft.rfft2(x.double().cpu(), s=pad) * torch.fft.rfft2(f.double().cpu(), s=pad), s=pad)
    ref = ref[..., 2:2 + h, 4:4 + w]
    # fp16 words at the pass boundaries: 4 roundings of 2^-12 rms relative to values of one size
    assert (y.double().cpu() - ref).norm() <= 1e-3 * ref.norm()
