"""Lengths with prime factors above 19 (the sum over pairs at 23, 29 and 31, the chirp transform,
bluestein.hip, above) against the FP64 oracle at
relative L2 <= 1e-6 * log2(N) per transform.

The lengths are the shortest and the longest that each convolution length M takes; the batches
leave lanes, whole transforms of the last workgroup, or nothing empty."""
import math

import numpy as np
import pytest

# (shortest, longest) length with a prime factor above 19 for M = 128, 256, ..., 16384
EDGES = [(37, 62), (69, 127), (129, 254), (257, 511), (514, 1021), (1027, 2047), (2051, 4093), (4099, 8191)]
LENGTHS = [23, 29, 31] + [n for pair in EDGES for n in pair]


def tol(n):
    return 1e-6 * math.log2(n)


def smooth(n):
    for p in (2, 3, 5, 7, 11, 13, 17, 19):
        while n % p == 0:
            n //= p
    return n == 1


def test_every_length_has_a_convolution_length():
    from sip_amd.fft import Plan
    for n in [v for v in range(37, 8193) if not smooth(v)][::29] + LENGTHS[3:]:
        p = Plan("c2c", (n,), 3)
        text = p.describe()
        p.close()
        m = int(text.split("chirp m=")[1].split()[0])
        assert 2 * n - 1 <= m < 4 * n and m & (m - 1) == 0, text


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from sip_amd import _native
    _native.lib()
    return torch.device("cuda:0")


def _complex(rng, shape):
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


def _run(torch_dev, kind, n, batch, inverse, x):
    import torch

    from sip_amd.fft import Plan
    p = Plan(kind, (n,), batch, inverse)
    try:
        return p.execute(torch.from_numpy(x).to(torch_dev)).cpu().numpy()
    finally:
        p.close()


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("inverse", [False, True])
def test_chirp_matches_oracle(torch_dev, oracle, n, inverse):
    from oracle.oracle import rel_l2_per_row
    rng = np.random.default_rng(n)
    for batch in (1, 13, 515 if n < 600 else 3):
        x = _complex(rng, (batch, n))
        got = _run(torch_dev, "c2c", n, batch, inverse, x)
        assert rel_l2_per_row(got, oracle.c2c(x, inverse)).max() <= tol(n), batch
    batch = 5
    x = rng.uniform(-1, 1, (batch, n)).astype(np.float32)
    assert rel_l2_per_row(_run(torch_dev, "r2c", n, batch, inverse, x), oracle.r2c_nd(x, 1, inverse)).max() <= tol(n)
    x = _complex(rng, (batch, n // 2 + 1))
    assert rel_l2_per_row(_run(torch_dev, "c2r", n, batch, inverse, x), oracle.c2r_nd(x, (n,), inverse)).max() <= tol(n)


@pytest.mark.gpu
@pytest.mark.parametrize("n", [31, 997, 2047])
def test_chirp_in_place_and_planes(torch_dev, oracle, n):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    rng = np.random.default_rng(n)
    batch = 37
    x = _complex(rng, (batch, n))
    want = oracle.c2c(x, True)
    buf = torch.from_numpy(x).to(torch_dev)
    p = Plan("c2c", (n,), batch, True)
    try:
        p.execute(buf, out=buf)
        assert rel_l2_per_row(buf.cpu().numpy(), want).max() <= tol(n)
    finally:
        p.close()
    re, im = (torch.from_numpy(np.ascontiguousarray(v)).to(torch_dev) for v in (x.real, x.imag))
    p = Plan("c2c_sep", (n,), batch, True)
    try:
        p.execute_separated(re, im, re, im)
        assert rel_l2_per_row(re.cpu().numpy() + 1j * im.cpu().numpy(), want).max() <= tol(n)
    finally:
        p.close()
