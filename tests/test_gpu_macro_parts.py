"""Macroscopic fields of which a caller wants some components only."""
import time

import numpy as np
import pytest

import _pkg
from test_gpu_parity import say
from test_gpu_transfer import lattice

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(3, 5), (401, 700), (7, 9, 11), (61, 70, 83), (180, 181, 182)])
def test_download_of_some_components(shape):
    """lbm_download_macro with null components: the others arrive as they do
    all together, and only they are moved (one field of four, where the bus
    bounds the transfer, takes well under half the time: a quarter of the
    bytes)"""
    say(f"case some components {shape}")
    L = _pkg.load()
    rng = np.random.default_rng(sum(shape))
    _, g = lattice(L, shape, 0, rng)
    g.set_mv(1, *rng.standard_normal((1 + g.dims, g.N)))
    every = g.mv(1)
    out = [np.zeros(g.N) for _ in range(4)]

    def download(which):
        ptr = [L._dp(out[c]) if c in which else None for c in range(4)]
        t = time.perf_counter()
        L._check(L.lib().lbm_download_macro(g.h, 1, *ptr))
        return time.perf_counter() - t

    for k in range(16):
        which = [c for c in range(4) if k >> c & 1]
        for o in out:
            o[:] = -7.0
        download(which)
        for c in range(4):
            assert np.array_equal(out[c], every[c] if c in which else np.full(g.N, -7.0)), (shape, which, c)
    if g.N > 5_000_000:
        one, all4 = (min(download(w) for _ in range(9)) for w in ((0,), range(4)))
        say(f"one component {one * 1e3:.2f} ms, all {all4 * 1e3:.2f} ms")
        assert one < 0.5 * all4
    g.close()
