"""Device memory that an adjoint sweep holds: the states before the steps of
one replayed segment, the adjoint state and its small accumulators."""
import numpy as np
import pytest
import torch

import _pkg
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nsteps,every", [(8, 4), (7, 3), (3, 100), (2, 1)])
def test_sweep_holds_one_segment(nsteps, every):
    say(f"case adjoint memory nsteps={nsteps} every={every}")
    L = _pkg.load()
    n = 64
    g = L.Lattice(mask=np.zeros((n, n, n), np.uint8), dims=3, ni=n, nj=n, nk=n, nsubs=2, tau=(0.8, 0.75),
                  zface_pressure=1, rho_bot=1.001, rho_top=1.0, zface_solute=1, c_bot=1.0, flux_plane=n - 4)
    state = n ** 3 * 2 * 19 * 8
    # the runtime's own memory for these kernels (their scratch), which stays;
    # the lattice's is released with its geometry
    g.init_rest()
    g.objective(2, 1, 1)
    g.adjoint()
    g.set_solids(np.zeros((n, n, n), np.uint8))
    g.init_rest()
    g.time = 0
    J = g.objective(nsteps, 1, every)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    grad, cmap = g.adjoint()
    held = (free - torch.cuda.mem_get_info()[0]) / state
    say(f"{held:.3f} states held")
    # the segment's states and the adjoint's; a quarter of one for the rest
    # (gradient slots, the inlet map, allocation granularity)
    assert held < min(every, nsteps) + 1.25
    again, cmap2 = g.adjoint()  # the same workspace serves again
    assert np.array_equal(again, grad) and np.array_equal(cmap2, cmap) and np.isfinite(J)
    g.close()
