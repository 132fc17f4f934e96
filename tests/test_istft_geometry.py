"""Which launches an ISTFT plan takes and the frames per group of the one launch (build_istft_fused,
istft_two_launches_faster in planner.cpp): at both sides of each rule, and both forms against the
FP64 oracle at relative L2 <= 1e-6 * log2(nfft) per channel where the rules choose them anew."""
import math

import numpy as np
import pytest

# (channel, nfft, nframes, hop), frames per group of the one launch (0: two launches)
ROUTES = [
    # two groups, the first for its halo alone: too small a batch, and one large enough
    ((1, 630, 2, 78), 0), ((37, 1331, 3, 166), 0), ((4, 1024, 50, 64), 0), ((16, 1024, 1000, 64), 16),
    # the same overlap in one group
    ((1, 1024, 50, 64), 16), ((2, 128, 70, 8), 16),
    # groups of 4 on more than 512 threads: five groups within the device cache, past it, fewer groups
    ((12, 1320, 325, 1015), 0), ((10, 1386, 597, 1066), 0), ((13, 1323, 840, 661), 4), ((5, 1440, 21, 360), 4),
    # three workgroups of five wavefronts do not share a CU
    ((9, 700, 1531, 175), 8), ((10, 720, 363, 180), 8), ((24, 324, 692, 81), 16),
    # the spectrum's lines where groups of 4 read a quarter of each
    ((26, 440, 939, 146), 16), ((38, 432, 658, 108), 8),
    # no hop of nfft / 17 above what a group holds; frames of nfft > 1024 in groups of 8 at most
    ((1, 128, 40, 7), 0), ((1, 1440, 50, 160), 0), ((1, 1280, 50, 80), 0),
    ((16, 1024, 1000, 256), 16),
]


@pytest.mark.parametrize("shape,frames", ROUTES, ids=str)
def test_route(shape, frames):
    from sip_amd import Istft
    p = Istft(*shape)
    text = p.describe()
    p.close()
    if frames == 0:
        assert "istft fused" not in text, text
    else:
        assert f"istft fused frames/group={frames} " in text, text


@pytest.mark.parametrize("shape", [(1 << 21, 1024, 2, 64), (1 << 22, 1024, 2, 64), (1 << 23, 1024, 2, 256)], ids=str)
def test_launch_stays_within_2_to_32_threads(shape):
    """Where the one launch would pass them (one workgroup of 1024 threads for two frames of a
    channel, 2^22 channels: 69 GB), the two launches stay."""
    import re

    from sip_amd import Istft
    p = Istft(*shape)
    text = p.describe()
    p.close()
    m = re.search(r"istft fused frames/group=(\d+) T=(\d+) .*grid=(\d+)", text)
    assert (m is None) == (shape == (1 << 22, 1024, 2, 64)), text
    assert m is None or math.prod(map(int, m.groups())) < 1 << 32, text


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(1, 630, 2, 78), (3, 1024, 5, 64), (2, 1320, 33, 1015), (9, 700, 41, 175), (5, 440, 37, 146)],
                         ids=str)
@pytest.mark.parametrize("form", ["0", "1"])
def test_forms_match_oracle(oracle, monkeypatch, shape, form):
    import torch

    from oracle.oracle import rel_l2_per_row
    from sip_amd import Istft
    channel, nfft, nframes, hop = shape
    rng = np.random.default_rng(nfft)
    spec = (rng.uniform(-1, 1, (channel, nfft, nframes)) +
            1j * rng.uniform(-1, 1, (channel, nfft, nframes))).astype(np.complex64)
    w = (0.6 + 0.4 * np.sin(2.0 * np.pi * np.arange(nfft) / nfft + 0.7)).astype(np.float32)
    monkeypatch.setenv("ASDFFT_ISTFT_FUSED", form)
    p = Istft(*shape)
    try:
        assert ("istft fused" in p.describe()) == (form == "1"), p.describe()
        out = torch.full((channel, p.out_len), float("nan"), dtype=torch.complex64, device="cuda")
        p.execute(torch.from_numpy(spec).cuda(), torch.from_numpy(w).cuda(), out=out)
        got = out.cpu().numpy()
    finally:
        p.close()
    assert rel_l2_per_row(got, oracle.istft(spec, w, hop), 1).max() <= 1e-6 * math.log2(nfft)
