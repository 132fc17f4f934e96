"""Schedules are tuned in the kernel that their plan runs: a class tuned for one launch form, or for a
batch of another budget, is timed again, and the tuned plan keeps the launch of the untuned one."""
import re

import pytest

pytestmark = pytest.mark.gpu


def tuned(entries, **kw):
    import torch  # noqa: F401  (its HIP runtime is loaded first)

    from sip_amd.fft import RaggedPlan
    plain, plan = RaggedPlan(entries, **kw), RaggedPlan(entries, autotune=True, **kw)
    try:
        launch = re.findall(r"launch emax=(\d+) block=(\d+)", plain.describe())
        text = plan.describe()
        timings = int(re.search(r"autotuned: (\d+) timings", text).group(1))
        return timings, launch, re.findall(r"launch emax=(\d+) block=(\d+)", text), text
    finally:
        plain.close()
        plan.close()


def test_forms_are_tuned_apart():
    first, launch, got, text = tuned([("c2c", 8748, 5, False)])
    assert launch == got == [("24", "512")] and first > 1 and "block16" not in text, text
    again = tuned([("c2c", 8748, 3, False)])
    assert again[0] == 0, again  # the same class in the same kernel
    other, _, got, text = tuned([("c2c", 8748, 5, False)], per_budget=True)
    sweep = 2  # two workgroup sizes on the whole batch
    assert other > sweep and "block16" in text and got[0][0] != "24", text


def test_batches_are_tuned_in_their_launch():
    alone, launch, _, _ = tuned([("c2c", 288, 40, False)])
    assert launch == [("16", "256")] and alone > 2
    _, launch, got, _ = tuned([("c2c", 15552, 2, False)])
    assert launch == got == [("20", "1024")]
    mixed, launch, got, text = tuned([("c2c", 288, 40, False), ("c2c", 15552, 2, False)])
    assert launch == got == [("20", "1024")], text
    assert mixed > 2, text  # 288 in the 1024-thread kernel (more than two runs of the whole batch)
