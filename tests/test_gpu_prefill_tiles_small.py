"""The prefill tiles at small layer shapes.

By default a layer whose prefill items do not fill the CUs takes the 128-row
kernel; with HFMOE_PREFILL_MIN_ROWS=4 it takes the prefill tiles from four rows
per expert on, as the full-shape layer does, so that their edges (ragged
widths, one K stage, no shared expert, tiles and items drawn from counters)
are checked without a 19 GB layer.  The tests are test_gpu_grouped's own, and
the rule itself: the choice changes a result in its last bits only.
"""
import numpy as np
import pytest

from hummingflight_amd import synth
from moe_harness import SMALL, Run
from test_gpu_grouped import (  # noqa: F401  (run here under the fixture below)
    test_grouped_fp32_activations, test_grouped_repeat_is_deterministic, test_grouped_small,
    test_grouped_small_prefill_tiles, test_grouped_without_shared_expert, test_prefill_tiles_edge_shapes,
    test_prefill_tiles_fp32_activations, test_tile_size_switch_boundary, test_wide_tiles_few_k_stages)

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def prefill_tiles_from_four_rows(monkeypatch):
    monkeypatch.setenv("HFMOE_PREFILL_MIN_ROWS", "4")


@pytest.mark.parametrize("T", [64, 767, 768])
def test_small_layer_choice(hf, monkeypatch, T):
    # 64 experts of 2048 x 1024: 264 items and more, a round of 256 CUs but not
    # four, so the prefill tiles from 96 rows per expert (T = 768) on.
    r = Run(SMALL, n_group=8, topk_group=4, seed=96, T=T)
    x = synth.make_x_dev(T, SMALL["hidden"], seed=96)
    wide = r.forward(x, T)["out"]
    monkeypatch.setenv("HFMOE_PREFILL_MIN_ROWS", "100000")
    narrow = r.forward(x, T)["out"]
    monkeypatch.delenv("HFMOE_PREFILL_MIN_ROWS")
    got = r.forward(x, T)["out"]
    assert not np.array_equal(wide, narrow)
    assert np.array_equal(got, wide if T >= 768 else narrow)
    assert np.linalg.norm(wide - narrow) <= 2.2e-5 * np.linalg.norm(narrow)  # two roundings of 16-bit operands
    x.free()
    r.free()
