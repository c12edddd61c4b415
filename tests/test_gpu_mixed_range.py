"""GPU tests of the range and precision of split fp16 lines odd * 2^a with one matrix-core stage on
the mixed-radix kernels (rows and columns): unscaled inputs that a radix-`odd` pass and a power-of-two
pass carry through fp16 operands without overflow, and scaled inputs so small that the operands' low
words are near fp16's smallest value; and of columns of odd * 16 points, which stay in fp32."""
import numpy as np
import pytest

import oracle

from .helpers import complex_input, from_device, rel_errors, to_device

# odd factor, power of two (16 * 4 or 16 * 8)
LINES = [(3, 64), (5, 64), (3, 128), (9, 64), (5, 128), (15, 64), (17, 64), (9, 128), (15, 128)]


def _run(dev, n, cols, x, scale):
    import torch

    import fft_demo_amd as F

    shape = (n, 4) if cols else (n,)
    with F.Plan(shape, x.shape[0], precision="split_fp16", in_fmt="c32", out_fmt="c32", scale=scale) as plan:
        return from_device(plan.exec(to_device(x, torch.float32, dev))) / plan.out_scale


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [False, True])
@pytest.mark.parametrize("odd,p", LINES)
def test_unscaled_range(dev, odd, p, cols):
    import fft_demo_amd as F

    # the largest power of two that the odd pass's sum keeps below 65504; columns: after the rows'
    # 4-point sum
    n, m = odd * p, 2.0 ** np.floor(np.log2(65504 / odd / (4 if cols else 1)))
    x = np.full((3, n, 4) if cols else (3, n), m * (1 - 1j))
    y = _run(dev, n, cols, x, F.SCALE_NONE)
    assert np.isfinite(y).all()
    ref = np.zeros_like(x)
    ref[(slice(None),) + (0,) * (x.ndim - 1)] = x[0].size * m * (1 - 1j)
    # a constant: 22-bit operands, fp32 sums
    assert np.abs(y - ref).max() <= 1e-6 * np.abs(ref).max()


@pytest.mark.gpu
@pytest.mark.parametrize("odd,p", LINES)
def test_scaled_small_inputs(dev, odd, p):
    import fft_demo_amd as F

    n, amp = odd * p, 2.0 ** -8
    x = complex_input((64, n), n, "c32") * amp
    l2, _ = rel_errors(_run(dev, n, False, x, F.SCALE_STAGE), oracle.fft(x))
    # operands round to multiples of 2^-24 (rms 2^-24 / sqrt 12); behind a scaled radix-odd pass the
    # signal's rms amp / sqrt 3 has become amp / sqrt(3 odd)
    assert l2 <= 1.2 * (2.0 ** -24 / np.sqrt(12)) * np.sqrt(3 * odd) / amp, l2


@pytest.mark.gpu
@pytest.mark.parametrize("odd", [3, 5, 9, 15, 17])
def test_columns_in_fp32(dev, odd):
    import torch

    import fft_demo_amd as F

    # rows of 4 points, columns of odd * 16: no matrix-core stage. Scaled and small, unscaled and large
    x = complex_input((16, 16 * odd, 4), odd, "c32")
    for amp, scale in ((2.0 ** -12, F.SCALE_STAGE), (2.0 ** 16, F.SCALE_NONE)):
        with F.Plan((16 * odd, 4), 16, precision="split_fp16", in_fmt="c32", out_fmt="c32", scale=scale) as plan:
            y = from_device(plan.exec(to_device(x * amp, torch.float32, dev))) / plan.out_scale
        l2, _ = rel_errors(y, oracle.fft2d(x * amp))
        assert l2 <= 1e-6, (amp, l2)  # four fp32 stages
