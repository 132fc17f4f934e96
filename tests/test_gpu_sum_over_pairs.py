"""Lengths to 127 with prime factors above 19 on both sides of the batch that moves them from the sum over
pairs to the chirp transform, even and odd (the middle element of an even length is its own pair), all
kinds and planes, against the FP64 oracle at relative L2 <= 1e-6 * log2(N) per transform."""
import math

import numpy as np
import pytest

LENGTHS = [37, 46, 62, 69, 86, 124, 127]


def rows(rng, shape):
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


@pytest.mark.parametrize("n", LENGTHS)
def test_route(n):
    from sip_amd.fft import Plan
    for batch, kernel in ((1, " sum over pairs"), (2048, " sum over pairs"), (2049, " chirp m=")):
        p = Plan("c2c", (n,), batch)
        text = p.describe()
        p.close()
        assert (" sum over pairs" if "sum over pairs" in text else " chirp m=") == kernel, text
    p = Plan("c2c", (129,), 1)
    assert "sum over pairs" not in p.describe()
    p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("batch", [1, 5, 2048, 2049])
@pytest.mark.parametrize("inverse", [False, True])
def test_matches_oracle(oracle, n, batch, inverse):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    rng = np.random.default_rng(n + batch)
    tol = 1e-6 * math.log2(n)

    def run(kind, x):
        p = Plan(kind, (n,), batch, inverse)
        try:
            return p.execute(torch.from_numpy(x).cuda()).cpu().numpy()
        finally:
            p.close()

    x = rows(rng, (batch, n))
    want = oracle.c2c(x, inverse)
    assert rel_l2_per_row(run("c2c", x), want).max() <= tol
    r = rng.uniform(-1, 1, (batch, n)).astype(np.float32)
    got = run("r2c", r)
    assert rel_l2_per_row(got, oracle.r2c_nd(r, 1, inverse)).max() <= tol
    assert np.all(got[:, 0].imag == 0) and (n % 2 or np.all(got[:, n // 2].imag == 0))
    h = rows(rng, (batch, n // 2 + 1))
    assert rel_l2_per_row(run("c2r", h), oracle.c2r_nd(h, (n,), inverse)).max() <= tol
    re, im = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x.real, x.imag))
    p = Plan("c2c_sep", (n,), batch, inverse)
    try:
        p.execute_separated(re, im, re, im)
    finally:
        p.close()
    assert rel_l2_per_row(re.cpu().numpy() + 1j * im.cpu().numpy(), want).max() <= tol


@pytest.mark.gpu
def test_istft_frames(oracle):
    """ISTFT frames of 46 points: strided columns of the spectrum."""
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd import Istft
    rng = np.random.default_rng(3)
    spec = rows(rng, (2, 46, 9))
    w = (0.6 + 0.4 * np.sin(2.0 * np.pi * np.arange(46) / 46 + 0.7)).astype(np.float32)
    p = Istft(2, 46, 9, 11)
    try:
        assert "sum over pairs" in p.describe()
        got = p.execute(torch.from_numpy(spec).cuda(), torch.from_numpy(w).cuda()).cpu().numpy()
    finally:
        p.close()
    assert rel_l2_per_row(got, oracle.istft(spec, w, 11), 1).max() <= 1e-6 * math.log2(46)
