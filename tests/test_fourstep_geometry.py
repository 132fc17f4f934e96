"""First passes of four-step transforms and shifted columns (cols_config in planner.cpp): workgroups of 32
points a thread stay within 512 threads, and what this moves against the FP64 oracle at relative L2 <=
1e-6 * log2(N) per transform."""
import math
import re

import numpy as np
import pytest

LENGTHS = [468160, 536085, 795600, 841568, 1290240, 1462050]


def first_pass(n, batch):
    from sip_amd.fft import Plan
    p = Plan("c2c", (n,), batch)
    text = p.describe()
    p.close()
    return [int(v) for v in re.search(r"variant=6 n=(\d+) .*?emax=(\d+) T=(\d+) tpb=(\d+) block=(\d+)", text).groups()], text


@pytest.mark.parametrize("n", LENGTHS)
@pytest.mark.parametrize("batch", [1, 9])
def test_first_pass_stays_within_its_threads(n, batch):
    (_, emax, threads, tpb, block), text = first_pass(n, batch)
    assert block == threads * tpb <= (1024 if emax == 16 else 512), text


@pytest.mark.gpu
@pytest.mark.parametrize("n", LENGTHS)
def test_long_lengths_match_oracle(oracle, n):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    rng = np.random.default_rng(n)
    x = (rng.uniform(-1, 1, (2, n)) + 1j * rng.uniform(-1, 1, (2, n))).astype(np.complex64)
    p = Plan("c2c", (n,), 2)
    try:
        got = p.execute(torch.from_numpy(x).cuda()).cpu().numpy()
    finally:
        p.close()
    assert rel_l2_per_row(got, oracle.c2c(x, False)).max() <= 1e-6 * math.log2(n)


SHIFTED = [(1156, 30), (1197, 85), (833, 75)]


@pytest.mark.parametrize("dims", SHIFTED)
def test_shifted_columns_stay_within_their_threads(dims):
    from sip_amd.fft import Plan
    p = Plan("c2c", dims, 2, in_shift="ifft", out_shift="fft")
    text = p.describe()
    p.close()
    assert int(re.search(r"variant=18 .*?block=(\d+)", text).group(1)) <= 512, text


@pytest.mark.gpu
@pytest.mark.parametrize("dims", SHIFTED)
def test_shifted_columns_match_oracle(oracle, dims):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    rng = np.random.default_rng(dims[0])
    x = (rng.uniform(-1, 1, (2,) + dims) + 1j * rng.uniform(-1, 1, (2,) + dims)).astype(np.complex64)
    p = Plan("c2c", dims, 2, in_shift="ifft", out_shift="fft")
    try:
        got = p.execute(torch.from_numpy(x).cuda()).cpu().numpy()
    finally:
        p.close()
    # "ifft" rolls by floor(n / 2), "fft" by ceil(n / 2), as asdIfftShift and asdFftShift do
    want = oracle.c2c_nd(np.roll(x, [d // 2 for d in dims], (1, 2)), 2, False)
    want = np.roll(want, [(d + 1) // 2 for d in dims], (1, 2))
    assert rel_l2_per_row(got, want, 2).max() <= 1e-6 * math.log2(dims[0] * dims[1])
