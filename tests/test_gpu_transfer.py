"""Dense host arrays to and from the GPU (k_dense_field / _get / _put through
pinned slots of 262,144 doubles): populations and fields come back as they
went in at fluid nodes and 0 at solid ones, for lattices below, at and above a
slot, pieces of several components and of parts of one, each storage type, and
handles used from several threads at once."""
import threading

import numpy as np
import pytest

import _pkg
from test_gpu_parity import random_state, say

pytestmark = pytest.mark.gpu

# values that FP16 storage holds exactly: multiples of 2^-10 (flow) and 2^-7
GRID = (2.0 ** -10, 2.0 ** -7)


def lattice(L, shape, storage, rng):
    mask = (rng.random(shape) < 0.3).astype(np.uint8)
    dims = len(shape)
    return mask.reshape(-1) != 1, L.Lattice(mask=mask, dims=dims, ni=shape[-1], nj=shape[-2],
                                            nk=shape[0] if dims == 3 else 1, nsubs=2, tau=(0.8, 0.75),
                                            storage=storage, compute=0 if storage == 0 else 1)


@pytest.mark.parametrize("storage", [0, 1, 2])
@pytest.mark.parametrize("shape", [(1, 1), (3, 5), (511, 513), (512, 512), (401, 700), (33, 90, 97)])
def test_dense_round_trip(shape, storage):
    say(f"case transfer {shape} storage={storage}")
    L = _pkg.load()
    rng = np.random.default_rng(sum(shape) + storage)
    fl, g = lattice(L, shape, storage, rng) if shape != (1, 1) else (
        np.array([True]), L.Lattice(mask=np.zeros((1, 1), np.uint8), dims=2, ni=1, nj=1, nsubs=2, tau=(0.8, 0.75),
                                    storage=storage, compute=0 if storage == 0 else 1))
    for s in range(2):
        f = rng.integers(-500, 500, (g.Q, g.N)) * GRID[s]
        g.upload_f(s, f)
        assert np.array_equal(g.download_f(s), f * fl), (shape, s)
    for s in range(2):
        fields = rng.standard_normal((1 + g.dims, g.N))
        g.set_mv(s, *fields)
        got = g.mv(s)
        for c in range(4):
            assert np.array_equal(got[c], fields[c] * fl if c <= g.dims else np.zeros(g.N)), (shape, s, c)
    g.close()


@pytest.mark.parametrize("points", [1, 64, 65, 50_000, 90_000])
def test_samples_equal_fields(points):
    """k_sample_field: values at listed nodes (repeats and solid nodes among
    them; more than one pinned slot holds) equal the downloaded fields"""
    L = _pkg.load()
    rng = np.random.default_rng(points)
    _, g = lattice(L, (19, 23, 29), 0, rng)
    for s in range(2):
        g.set_mv(s, *rng.standard_normal((4, g.N)))
    at = rng.integers(0, g.N, points)
    for s in range(2):
        assert np.array_equal(g.sample_mv(s, at), np.stack(g.mv(s), 1)[at])
    with pytest.raises(L.LbmError, match="outside the lattice"):
        g.sample_mv(0, [0, g.N])
    assert g.sample_mv(0, []).shape == (0, 4)
    g.close()


def test_transfers_from_several_threads():
    L = _pkg.load()
    bad = []

    def work(seed):
        rng = np.random.default_rng(seed)
        fl, g = lattice(L, (200 + seed, 301), 0, rng)
        for _ in range(4):
            f, _ = random_state(rng, 9, g.N, 1)
            g.upload_f(1, f)
            if not np.array_equal(g.download_f(1), f * fl):
                bad.append(seed)
        g.close()
    threads = [threading.Thread(target=work, args=(q,)) for q in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
