"""Batches of lengths 1, 23, 29, 31 and the chirp transform whose workgroups take several rows of the
grid (65536 a row), and the first batch of 23 points past 2^32 threads, against the FP64 oracle at
relative L2 <= 1e-6 * log2(N) per transform: the first and last transforms and those around the ends
of the rows."""
import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def in_place(oracle, n, batch, spots):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    x = torch.empty((batch, n), dtype=torch.complex64, device="cuda")
    step = 1 << 24
    for i in range(0, batch, step):
        torch.view_as_real(x[i:i + step]).uniform_(-1.0, 1.0)
    rows = torch.tensor(sorted({min(max(0, s + d), batch - 1) for s in spots for d in range(-20, 20)}), device="cuda")
    before = x[rows].cpu().numpy()
    p = Plan("c2c", (n,), batch)
    try:
        p.execute(x, out=x)
        after = x[rows].cpu().numpy()
    finally:
        p.close()
    assert rel_l2_per_row(after, oracle.c2c(before, False)).max() <= 1e-6 * math.log2(n)


@pytest.mark.parametrize("n,per_workgroup", [(23, 16), (31, 16), (37, 32)])
def test_two_rows(oracle, n, per_workgroup):
    batch = 65537 * per_workgroup + 3  # 65538 workgroups: rows of 32769
    in_place(oracle, n, batch, [0, 32769 * per_workgroup, batch])


def test_unit_rows():
    """The length-1 axis of a 2D C2R: 65536 * 257 elements copied in rows of workgroups of 256."""
    import torch

    from sip_amd.fft import Plan
    batch = 1 << 16
    x = torch.randn(batch, 1, 257, dtype=torch.complex64, device="cuda")
    p, q = Plan("c2r", (1, 512), batch, True), Plan("c2r", (512,), batch, True)
    try:
        assert "direct n=1" in p.describe() and "grid=65792" in p.describe(), p.describe()
        assert torch.equal(p.execute(x).view(batch, 512), q.execute(x.view(batch, 257)))
    finally:
        p.close()
        q.close()


def test_more_than_2_to_32_threads(oracle):
    import torch
    torch.cuda.empty_cache()
    if torch.cuda.mem_get_info()[0] < 60 << 30:
        pytest.skip("needs 60 GiB of free device memory")
    batch = (1 << 28) + 37
    in_place(oracle, 23, batch, [0, 1 << 27, 1 << 28, batch])
    torch.cuda.empty_cache()
