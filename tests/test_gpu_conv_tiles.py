"""GPU tests of the conv operator's pointwise kernels in every tile they choose: one map a thread
(small planes, single maps), 2 x 2 and 4 x 4 tiles, whole and partial, with and without the split
over filters. Every choice must give what the operator gives map by map."""
import pytest


# batch, channels, filters and planes that take: one map everywhere | one map (few blocks), 2 x 2 gw,
# split gi | 4 x 4 forward, 2 x 2 gw, split gi | 4 x 4 everywhere, gi unsplit | partial 4 x 4 tiles
CASES = [(3, 2, 3, 12, 12, 3), (16, 6, 9, 40, 40, 3), (8, 3, 16, 150, 256, 5), (16, 16, 16, 128, 128, 3),
         (10, 5, 17, 136, 256, 3), (1, 16, 16, 64, 64, 5), (32, 4, 1, 64, 64, 5), (128, 3, 8, 16, 16, 3)]


def _layer(dev, B, C, F, h, w, k, amp):
    import torch

    from fft_demo_amd.conv import Conv2d

    g = torch.Generator(device=dev)
    g.manual_seed(B + C + F)
    x = (torch.rand((B, C, h, w), generator=g, device=dev) - 0.5) * amp
    f = torch.rand((F, C, k, k), generator=g, device=dev) - 0.5
    op = Conv2d(B, C, F, h, w, k, k, mode="valid_corr")
    d = (torch.rand(op.out_shape, generator=g, device=dev) - 0.5) * amp
    op.set_filters(f)
    s = tuple(-(-(n + k - 1) // 16) * 16 for n in (h, w))
    return op, x, f, d, s, tuple(torch.fft.rfft2(t.double().cpu(), s) for t in (x, f, d))


def _error(got, want):  # of the worst map
    return ((got.double().cpu() - want).flatten(2).norm(dim=2) / want.flatten(2).norm(dim=2)).max()


# fp32 spectra of split fp16 transforms: 1e-5
@pytest.mark.gpu
@pytest.mark.parametrize("B,C,F,h,w,k", CASES)
def test_forward_and_input_gradient(dev, B, C, F, h, w, k):
    import torch

    op, x, _, d, s, (X, W, D) = _layer(dev, B, C, F, h, w, k, 1.0)
    want = torch.fft.irfft2(torch.stack([(X * W[j].conj()).sum(1) for j in range(F)], 1), s)[..., :h - k + 1, :w - k + 1]
    assert _error(op.forward(x), want) <= 1e-5
    want = torch.fft.irfft2(torch.stack([(D * W[:, j]).sum(1) for j in range(C)], 1), s)[..., :h, :w]
    assert _error(op.backward(d, grad_w=False)[0], want) <= 1e-5


# Inputs of 256: both spectra carry 1 / P, their products (about amp^2 / 12 P) then lie above 2^-14, where
# fp16 keeps its precision, and the gradient's inverse is as good as the others
@pytest.mark.gpu
@pytest.mark.parametrize("B,C,F,h,w,k", CASES)
def test_filter_gradient(dev, B, C, F, h, w, k):
    import torch

    op, x, _, d, s, (X, _, D) = _layer(dev, B, C, F, h, w, k, 256.0)
    want = torch.fft.irfft2(torch.stack([(X * D[:, j:j + 1].conj()).sum(0) for j in range(F)]), s)[..., :k, :k]
    assert _error(op.backward(d, x, grad_in=False)[1], want) <= 1e-5
