"""Plans and wait counts of the one-group GEMM tiles (fixed_plan.h,
gemm_item_wide with 4 and 5 column blocks), checked in a host build.

Every plan must be one that the launch accepts: M tiles of whole 16-row blocks,
none of them empty and none taller than the kernel's accumulators, N tiles that
cover N, and K splits that leave each at least four stages and stay within the
caller's partials.
"""
import os
import random
import subprocess

import pytest

from test_split_pipeline import simulate_wide

DRIVER_DIR = os.path.join(os.path.dirname(os.path.abspath(__file__)), "fixed_plan")


def plans(cases):
    subprocess.run(["make", "-s", "-C", DRIVER_DIR], check=True)
    text = "".join(" ".join(map(str, c)) + "\n" for c in cases)
    out = subprocess.run([os.path.join(DRIVER_DIR, "driver")], input=text, capture_output=True, text=True, check=True)
    return [tuple(map(int, line.split())) for line in out.stdout.splitlines()]


def test_plans_cover_every_row_and_column():
    rng = random.Random(3)
    cases = [(T, 12288, 1, 4, 96, 32, 256) for T in range(1, 700)]
    cases += [(T, 154880, 0, 5, 96, 1, 256) for T in range(1, 129)]
    for _ in range(3000):
        cb = rng.choice([4, 5])
        pair = rng.choice([0, 1]) if cb == 4 else 0
        T = rng.randint(1, 128 if cb == 5 else 8192)
        cases.append((T, rng.randint(64 * cb * (2 - pair), 200000), pair, cb, rng.randint(1, 640), rng.randint(1, 32),
                      rng.choice([8, 64, 256, 304])))
    for c, (m, rows, n, ks, most_rows, cols) in zip(cases, plans(cases)):
        T, N, pair, cb, stages, most, blocks = c
        assert rows % 16 == 0 and 16 <= rows <= most_rows, c
        assert m * rows >= T > (m - 1) * rows, c
        assert n * cols >= N > (n - 1) * cols, c
        assert 1 <= ks <= most and (ks == 1 or 4 * ks <= stages), c


@pytest.mark.parametrize("cb,rows", [(4, 160), (5, 128)])
def test_waits_cover_their_loads(cb, rows):
    # A half-stage is cb DMA instructions of 8 weight rows, of which a sub-step
    # may leave one half-stage outstanding.
    w = dict(nad=-(-rows // 64), nwh=cb, after=cb, wper1=2, wper2=1)
    for H in (1, 2):
        for nk in range(1, 12):
            for nad in range(w["nad"] + 1):
                simulate_wide(w, H, nk, nad)
        with pytest.raises(AssertionError):
            simulate_wide(dict(w, after=cb + 1), H, 4, w["nad"])
