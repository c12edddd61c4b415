"""GPU tests of the conv transforms with fused ends (rows read from real planes, columns stored as
cropped real planes): every line length they exist for on each axis, mixed with an axis that has none,
odd batches, partial tiles, filters of one tap (a cyclic offset of zero). fp64 planes take the separate
packing and cropping kernels, so for inputs that fp32 holds both must give the same values."""
import pytest


@pytest.mark.gpu
@pytest.mark.parametrize("B,C,F,pad,h,w,fh,fw", [(3, 2, 3, (64, 64), 61, 50, 5, 4), (2, 1, 1, (128, 64), 128, 64, 1, 1),
                                                 (1, 3, 2, (64, 128), 64, 127, 3, 7), (5, 2, 2, (256, 256), 250, 129, 13, 13),
                                                 (2, 1, 2, (512, 64), 300, 60, 9, 2), (3, 1, 1, (64, 512), 33, 512, 2, 33),
                                                 (2, 1, 1, (1024, 256), 1000, 200, 31, 31), (3, 1, 1, (128, 1024), 100, 1000, 4, 5),
                                                 (3, 2, 2, (80, 64), 79, 64, 6, 6), (3, 2, 2, (128, 68), 128, 67, 6, 6),
                                                 (4, 1, 3, (256, 36), 200, 36, 40, 3)])
def test_fused_ends_match_separate_passes(dev, B, C, F, pad, h, w, fh, fw):
    import torch

    from fft_demo_amd.conv import Conv2d

    g = torch.Generator(device=dev)
    g.manual_seed(7)
    x = torch.rand((B, C, h, w), generator=g, device=dev)
    f = torch.rand((F, C, fh, fw), generator=g, device=dev) - 0.5
    d = torch.rand((B, F, h - fh + 1, w - fw + 1), generator=g, device=dev) - 0.5
    op = Conv2d(B, C, F, h, w, fh, fw, mode="valid_corr", pad=pad)
    op.set_filters(f)
    got = (op.forward(x), op.forward(x, filter=F - 1), *op.backward(d, x))
    want = (op.forward(x.double()), op.forward(x.double(), filter=F - 1), *op.backward(d.double(), x.double()))
    for a, b in zip(got, want):
        assert torch.equal(a, b.float())
    if h + fh - 1 <= pad[0] and w + fw - 1 <= pad[1]:
        op = Conv2d(B, C, F, h, w, fh, fw, mode="same", pad=pad)
        op.set_filters(f)
        assert torch.equal(op.forward(x), op.forward(x.double()).float())


@pytest.mark.gpu
@pytest.mark.parametrize("option", [{}, {"mid_fp16": True}, {"spec_fp16": True}])
@pytest.mark.parametrize("pad,h,w,k", [((192, 64), 180, 50, 5), ((1088, 80), 1080, 70, 9), ((384, 128), 380, 100, 3),
                                       ((768, 96), 700, 90, 7), ((2560, 68), 2500, 60, 5), ((3072, 64), 3066, 64, 1),
                                       ((512, 48), 500, 40, 8)])
def test_crop_in_the_last_pass_of_split_columns(dev, option, pad, h, w, k):
    import torch

    from fft_demo_amd.conv import Conv2d

    g = torch.Generator(device=dev)
    g.manual_seed(11)
    x = torch.rand((3, 1, h, w), generator=g, device=dev)
    f = torch.rand((1, 1, k, k), generator=g, device=dev)
    op = Conv2d(3, 1, 1, h, w, k, k, mode="same", pad=pad, **option)
    op.set_filters(f)
    assert torch.equal(op.forward(x), op.forward(x.double()).float())
