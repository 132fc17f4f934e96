"""Which register budget a row launch takes (rows_share_a_cu in planner.cpp), at both sides of its rules,
and the lengths that it moves against the FP64 oracle at relative L2 <= 1e-6 * log2(N) per transform."""
import math
import re

import numpy as np
import pytest

# kind, length, batch, points per thread
BUDGETS = [
    # planar rows: three workgroups of 32 points on a CU, no more transforms than CUs, one that is already shared
    ("c2c_sep", 5670, 694, 32), ("c2c_sep", 5040, 2902, 32), ("c2c_sep", 5670, 256, 16), ("c2c_sep", 3780, 2000, 16),
    # two of them: in one round instead of two, and in more
    ("c2c_sep", 8320, 272, 32), ("c2c_sep", 8320, 512, 32), ("c2c_sep", 8320, 513, 16),
    ("c2r", 13860, 285, 32), ("c2r", 15552, 2738, 16), ("r2c", 18816, 290, 32), ("r2c", 18816, 700, 16),
    ("r2c", 18000, 2872, 32),
    # two of 16 points share a CU; a specialised kernel
    ("c2c", 5670, 694, 16), ("c2c_sep", 8192, 700, 16),
]


@pytest.mark.parametrize("kind,n,batch,points", BUDGETS)
def test_budget(kind, n, batch, points):
    from sip_amd.fft import Plan
    p = Plan(kind, (n,), batch, kind == "c2r")
    text = p.describe()
    p.close()
    assert int(re.search(r"emax=(\d+)", text).group(1)) == points, text


@pytest.mark.gpu
@pytest.mark.parametrize("kind,n,batch", [("c2c_sep", 5670, 258), ("c2c_sep", 8320, 257), ("c2r", 13860, 257), ("r2c", 18816, 257)])
def test_rows_match_oracle(oracle, kind, n, batch):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd.fft import Plan
    rng = np.random.default_rng(n)
    p = Plan(kind, (n,), batch, kind == "c2r")
    try:
        assert "emax=32" in p.describe()
        if kind == "r2c":
            x = rng.uniform(-1, 1, (batch, n)).astype(np.float32)
            got, want = p.execute(torch.from_numpy(x).cuda()).cpu().numpy(), oracle.r2c(x)
        elif kind == "c2r":
            x = np.fft.rfft(rng.uniform(-1, 1, (batch, n))).astype(np.complex64)
            got, want = p.execute(torch.from_numpy(x).cuda()).cpu().numpy(), oracle.c2r(x, n, True)
        else:
            x = (rng.uniform(-1, 1, (batch, n)) + 1j * rng.uniform(-1, 1, (batch, n))).astype(np.complex64)
            re_, im = (torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x.real, x.imag))
            p.execute_separated(re_, im, re_, im)
            got, want = re_.cpu().numpy() + 1j * im.cpu().numpy(), oracle.c2c(x, False)
    finally:
        p.close()
    assert rel_l2_per_row(got, want).max() <= 1e-6 * math.log2(n)
