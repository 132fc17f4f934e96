"""Run-time kernels on up to 1024 threads (rows of one transform per workgroup, 16, 8 or 4
columns) against the FP64 oracle at relative L2 <= 1e-6 * log2(N) per transform.

Row lengths: the last on 256 threads and the first above it, 1024 threads exactly, the first
whose passes need 32 points per thread.  Column lengths: the longest that keep 16, 8 and 4
columns with a second workgroup on the CU, and the next one; row lengths that leave partial
column tiles and rows off the 128-byte line."""
import math

import numpy as np
import pytest

ROWS = [2560, 2592, 4320, 9216, 10240, 10935, 14400, 16128]
COLUMNS = [(588, 33), (600, 16), (1134, 19), (1260, 8), (1280, 37), (2016, 5), (2058, 9)]


def tol(n):
    return 1e-6 * math.log2(n)


@pytest.fixture(scope="module")
def torch_dev():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a HIP device"
    from sip_amd import _native
    _native.lib()
    return torch.device("cuda:0")


def _complex(rng, shape):
    return (rng.uniform(-1, 1, shape) + 1j * rng.uniform(-1, 1, shape)).astype(np.complex64)


def _run(torch_dev, kind, dims, batch, inverse, x):
    import torch

    from sip_amd.fft import Plan
    p = Plan(kind, dims, batch, inverse)
    try:
        return p.execute(torch.from_numpy(x).to(torch_dev)).cpu().numpy()
    finally:
        p.close()


def test_workgroups_hold_every_pass():
    """Every butterfly of every pass has a slot: threads x (budget / radix) >= N / radix."""
    import re

    from sip_amd.fft import Plan
    for dims in [(n,) for n in ROWS] + COLUMNS:
        p = Plan("c2c", dims, 3)
        text = p.describe()
        p.close()
        for line in (s for s in text.splitlines() if "stockham" in s):
            f = dict(re.findall(r"(\w+)=([\w.x]+)", line))
            n, t, emax = int(f["n"]), int(f["T"]), int(f["emax"])
            assert int(f["block"]) <= 1024 and int(f["lds"]) <= 160 * 1024, line
            for r in map(int, f["radices"].split("x")):
                assert t * (emax // r) >= n // r, line


@pytest.mark.gpu
@pytest.mark.parametrize("n", ROWS)
@pytest.mark.parametrize("inverse", [False, True])
def test_rows(torch_dev, n, inverse):
    from oracle import oracle
    rng = np.random.default_rng(n)
    x = _complex(rng, (5, n))
    assert oracle.rel_l2_per_row(_run(torch_dev, "c2c", (n,), 5, inverse, x), oracle.c2c(x, inverse)).max() <= tol(n)
    r = rng.uniform(-1, 1, (3, 2 * n)).astype(np.float32)
    if not inverse:
        got, gold = _run(torch_dev, "r2c", (2 * n,), 3, False, r), oracle.r2c(r)
    else:
        h = np.fft.rfft(r).astype(np.complex64)
        got, gold = _run(torch_dev, "c2r", (2 * n,), 3, True, h), oracle.c2r(h, 2 * n, True)
    assert oracle.rel_l2_per_row(got, gold).max() <= tol(2 * n)


@pytest.mark.gpu
@pytest.mark.parametrize("dims", COLUMNS)
@pytest.mark.parametrize("inverse", [False, True])
def test_columns(torch_dev, dims, inverse):
    from oracle import oracle
    x = _complex(np.random.default_rng(dims[0]), (2,) + dims)
    got = _run(torch_dev, "c2c", dims, 2, inverse, x)
    assert oracle.rel_l2_per_row(got, oracle.c2c_nd(x, 2, inverse), 2).max() <= tol(dims[0] * dims[1])
