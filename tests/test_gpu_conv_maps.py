"""GPU tests of the conv operator's elementwise kernels where their tiles are partial: map counts
around the 4 x 4 tile (pairs, channels, filters), odd batches, odd and self-mirrored planes, rows
narrower and wider than a block."""
import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("B,C,F,h,w,fh,fw,pad", [(1, 1, 1, 20, 24, 3, 3, None),    # one map everywhere
                                                 (9, 5, 6, 33, 30, 4, 5, None),    # 5 pairs, a second tile of one map
                                                 (8, 4, 4, 40, 16, 3, 2, None),    # whole tiles
                                                 (3, 2, 7, 25, 31, 5, 5, (45, 51)),  # odd planes: no self-mirrored middle row
                                                 (2, 1, 2, 12, 700, 3, 9, None)])  # rows wider than 512 columns
def test_layer_maps(dev, B, C, F, h, w, fh, fw, pad):
    import torch

    from fft_demo_amd.conv import Conv2d

    x = oracle.uniform(B * C * h * w, 1, 0.0, 1.0).reshape(B, C, h, w)
    f = oracle.uniform(F * C * fh * fw, 2).reshape(F, C, fh, fw)
    oh, ow = h - fh + 1, w - fw + 1
    d = oracle.uniform(B * F * oh * ow, 3).reshape(B, F, oh, ow)
    op = Conv2d(B, C, F, h, w, fh, fw, mode="valid_corr", pad=pad)
    xd, fd, dd = (torch.from_numpy(np.ascontiguousarray(a)).float().to(dev) for a in (x, f, d))
    op.set_filters(fd)
    out = op.forward(xd).double().cpu().numpy()
    gi, gw = (t.double().cpu().numpy() for t in op.backward(dd, xd))
    s = (h + fh - 1, w + fw - 1)
    X, W, D = (np.fft.rfft2(a.astype(np.float32).astype(np.float64), s) for a in (x, f, d))
    want_out = np.fft.irfft2(np.einsum("bcuv,fcuv->bfuv", X, W.conj()), s)[..., :oh, :ow]
    want_gi = np.fft.irfft2(np.einsum("bfuv,fcuv->bcuv", D, W), s)[..., :h, :w]
    want_gw = np.fft.irfft2(np.einsum("bcuv,bfuv->fcuv", X, D.conj()), s)[..., :fh, :fw]
    # the operator's tolerances on these sizes (fp32 spectra of split fp16 transforms)
    for got, want, tol in ((out, want_out, 1e-4), (gi, want_gi, 1e-4), (gw, want_gw, 1e-3)):
        assert np.linalg.norm(got - want) <= tol * np.linalg.norm(want)
