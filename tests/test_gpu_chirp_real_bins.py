"""R2C at lengths with prime factors above 19: the bins of a real input that are real (0, and n/2 of
an even length) come with an imaginary part of exactly zero, in 1D and as the rows of a 2D
transform, and a row that is not finite stays visible in both parts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def run(kind, dims, batch, inverse, x):
    import torch

    from sip_amd.fft import Plan
    p = Plan(kind, dims, batch, inverse)
    try:
        return p.execute(torch.from_numpy(x).cuda()).cpu().numpy()
    finally:
        p.close()


@pytest.mark.parametrize("n", [23, 31, 37, 46, 62, 74, 254, 509, 997, 1994, 4093, 4106, 8188, 8191])
@pytest.mark.parametrize("inverse", [False, True])
def test_real_bins_1d(n, inverse):
    x = np.random.default_rng(n).uniform(-1, 1, (7, n)).astype(np.float32)
    y = run("r2c", (n,), 7, inverse, x)
    assert np.all(y[:, 0].imag == 0)
    if n % 2 == 0:
        assert np.all(y[:, n // 2].imag == 0)
    assert np.all(y[:, 1].imag != 0)


def test_real_bins_2d():
    x = np.random.default_rng(1).uniform(-1, 1, (3, 8, 74)).astype(np.float32)
    y = run("r2c", (8, 74), 3, False, x)
    for i in (0, 4):
        for k in (0, 37):
            assert np.all(y[:, i, k].imag == 0), (i, k)


def test_not_finite_rows():
    x = np.ones((3, 74), np.float32)
    x[1, 5] = np.nan
    y = run("r2c", (74,), 3, False, x)
    assert np.isnan(y[1, 0].real) and np.isnan(y[1, 0].imag) and np.isnan(y[1, 37].imag)
    assert np.all(np.isfinite(y[[0, 2]]))
