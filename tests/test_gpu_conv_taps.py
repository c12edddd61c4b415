"""GPU test of the precision of short filters' spectra: a constant image leaves only the spectrum's
first value, the sum of the taps, whose rounding is told from the transforms' by filters of one tap
that hold the sums themselves."""
import numpy as np
import pytest

import oracle


@pytest.mark.gpu
@pytest.mark.parametrize("k", [31, 32])
def test_sum_of_the_taps(dev, k):
    import torch

    from fft_demo_amd.conv import Conv2d

    F = 1024
    w = oracle.uniform(F * k * k, k, 0.0, 1.0).astype(np.float32).reshape(F, 1, k, k)
    total = w.astype(np.float64).sum((1, 2, 3))
    x = torch.ones((1, 1, 32, 32), device=dev)

    def error(f, want):
        op = Conv2d(1, 1, F, 32, 32, f.shape[2], f.shape[3], mode="valid_corr", pad=32)
        op.set_filters(torch.from_numpy(f).to(dev))
        y = op.forward(x)[0, :, 0, 0].double().cpu().numpy()
        return np.sqrt(np.mean((y / want - 1) ** 2))

    sums = total.astype(np.float32)
    e = error(w, total)
    e1 = error(sums.reshape(F, 1, 1, 1), sums.astype(np.float64))
    # the rounding of k taps of a row, then k rows, summed in one chain each
    rows = np.zeros((F, k), np.float32)
    for i in range(k):
        rows += w[:, 0, :, i]
    chain = np.zeros(F, np.float32)
    for i in range(k):
        chain += rows[:, i]
    serial = np.sqrt(np.mean((chain / total - 1) ** 2))
    # parts of at most 8 terms: about 0.45 (31 taps) and 0.56 (32) of it
    assert np.sqrt(max(0.0, e * e - e1 * e1)) <= 0.8 * serial, (e, e1, serial)
