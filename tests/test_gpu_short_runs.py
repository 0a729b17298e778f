"""Runs of few steps on FP64 2-D lattices without row conditions: a launch of
several steps is taken only where it is no slower than the half-steps one by
one (which a handle with forced 64-bit offsets always launches, and whose
fields are the same)."""
import time

import numpy as np
import pytest

import _pkg
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

CASES = {  # ni, nj, components, partial bounce-back, steps of a run
    "strips_of_51_columns": (102, 11500, 2, False, 2),
    "strips_of_51_columns_walsh": (102, 11500, 2, True, 2),
    "second_round_of_tiles": (420, 300, 1, False, 2),
    "second_round_of_large_tiles": (480, 340, 1, False, 2),
    "beyond_the_cache_walsh": (2100, 1900, 1, True, 2),
    "one_round_flow_solute_walsh": (200, 170, 2, True, 2),
    "one_round": (128, 128, 1, False, 2),
    "many_tiles": (1000, 1000, 1, False, 2),
    "three_steps": (102, 11500, 2, False, 3),
    "four_steps_second_round_walsh": (480, 340, 1, True, 4),
    "six_steps_second_round_walsh": (480, 340, 1, True, 6),
}


@pytest.mark.parametrize("case", list(CASES))
def test_few_steps_not_slower_than_single_ones(case, monkeypatch):
    ni, nj, nsubs, walsh, n = CASES[case]
    say(f"case short runs {case}")
    L = _pkg.load()
    rng = np.random.default_rng(ni + nj)
    mask = (rng.random((nj, ni)) < 0.3).astype(np.uint8)
    mask[0, 0] = 0
    lats = []
    for force in ("0", "1"):
        monkeypatch.setenv("LBM_OFFSET64", force)
        g = L.Lattice(mask=mask, dims=2, ni=ni, nj=nj, nsubs=nsubs, tau=(0.8, 0.75), gaccel=(1e-6, 0, 0, 0, 0, 0))
        if walsh:
            g.set_ns(np.full((nj, ni), 0.3))
        g.init_rest(np.random.default_rng(1).random(ni * nj))
        lats.append(g)
    best = [np.inf, np.inf]
    for rep in range(30):
        for q, g in enumerate(lats):
            t = time.perf_counter()
            for _ in range(20):
                g.run(n, write_last=False)
            best[q] = min(best[q], (time.perf_counter() - t) / (20 * n))
    say(f"{case}: {best[0] * 1e6:.2f} us a step, one by one {best[1] * 1e6:.2f}")
    for s in range(nsubs):
        assert np.array_equal(lats[0].download_f(s), lats[1].download_f(s))
    # a tenth for what two timings of one and the same run may differ by
    assert best[0] < 1.1 * best[1]
    for g in lats:
        g.close()
