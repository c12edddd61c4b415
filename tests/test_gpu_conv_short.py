"""GPU tests of the short-filter kernel (spectra straight from the taps) and of inverse transforms of a
filter gradient's columns alone: filter heights at the ends of each register size and one past the last,
widths up to the limit, planes whose columns are not whole blocks of 64 and with an odd row count."""
import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("B,C,F,h,w,fh,fw,pad", [(1, 1, 1, 32, 32, 1, 1, None), (3, 2, 5, 40, 70, 4, 32, None),
                                                 (2, 3, 4, 64, 64, 5, 3, None), (5, 1, 9, 60, 130, 12, 13, None),
                                                 (2, 2, 2, 45, 51, 13, 16, (45, 51)), (2, 1, 3, 100, 40, 16, 17, None),
                                                 (1, 2, 2, 68, 64, 24, 24, None), (2, 1, 2, 90, 65, 25, 31, None),
                                                 (2, 2, 1, 96, 96, 32, 32, None), (2, 1, 2, 96, 96, 33, 8, None)])
def test_short_filter_layer(dev, B, C, F, h, w, fh, fw, pad):
    import torch

    from fft_demo_amd.conv import Conv2d

    x = oracle.uniform(B * C * h * w, 1, 0.0, 1.0).reshape(B, C, h, w)
    f = oracle.uniform(F * C * fh * fw, 2).reshape(F, C, fh, fw)
    oh, ow = h - fh + 1, w - fw + 1
    d = oracle.uniform(B * F * oh * ow, 3).reshape(B, F, oh, ow)
    op = Conv2d(B, C, F, h, w, fh, fw, mode="valid_corr", pad=pad)
    s = (h + fh - 1, w + fw - 1)
    X, W, D = (np.fft.rfft2(a.astype(np.float32).astype(np.float64), s) for a in (x, f, d))
    want = (np.fft.irfft2(np.einsum("bcuv,fcuv->bfuv", X, W.conj()), s)[..., :oh, :ow],
            np.fft.irfft2(np.einsum("bfuv,fcuv->bcuv", D, W), s)[..., :h, :w],
            np.fft.irfft2(np.einsum("bcuv,bfuv->fcuv", X, D.conj()), s)[..., :fh, :fw])
    for dt in (torch.float32, torch.float64):
        xd, fd, dd = (torch.from_numpy(np.ascontiguousarray(a)).float().to(device=dev, dtype=dt) for a in (x, f, d))
        op.set_filters(fd)
        got = (op.forward(xd),) + tuple(op.backward(dd, xd))
        # the operator's tolerances on these sizes (fp32 spectra of split fp16 transforms)
        for g, ref, tol in zip(got, want, (1e-4, 1e-4, 1e-3)):
            g = g.double().cpu().numpy()
            assert np.linalg.norm(g - ref) <= tol * np.linalg.norm(ref)
