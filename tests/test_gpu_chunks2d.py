"""Captured chunks of steps on 2-D lattices: those that lbm_run does not send
through the tiles (FP32 and FP16 storage, FP64 with forced 64-bit offsets)
replay graphs of 64 steps, except where the boundary values change from step
to step (a ramp that still runs, a pressure series)."""
import numpy as np
import pytest

import _pkg
from test_gpu_parity import random_state, say

pytestmark = pytest.mark.gpu

KIND = {"fp32": dict(storage=1, compute=1), "fp32_f64": dict(storage=1, compute=0), "fp16": dict(storage=2, compute=1),
        "fp64_off64": dict(storage=0, compute=0)}
T = np.arange(23)
ROWS = {
    "rows": dict(pressure_s_in=(1, 0), pressure_n_out=(1, 0), rho_in=1.002, rho_out=0.999),
    "ramp": dict(pressure_s_in=(1, 0), pressure_n_out=(1, 0), rho_in=1.002, rho_out=0.999, bc_ramp_start=3,
                 bc_ramp_stop=500),
    "ramp_ends": dict(pressure_s_in=(1, 0), pressure_n_out=(1, 0), rho_in=1.002, rho_out=0.999, bc_ramp_start=3,
                      bc_ramp_stop=140),
    "series": dict(pressure_n_in=(2, 0), pressure_s_in=(2, 0), pfadd=1.0, pfmul=0.1,
                   pressure_n_series=(0.01 * np.sin(T), None), pressure_s_series=(0.01 * np.cos(T), None)),
    "velocity_ramp": dict(velocity_s_in=1, pressure_n_out=(1, 0), uy_in=2e-3, bc_ramp_start=10, bc_ramp_stop=400),
}


@pytest.mark.parametrize("rows", list(ROWS))
@pytest.mark.parametrize("kind", list(KIND))
def test_2d_chunks_equal_stepwise_launches(kind, rows, monkeypatch):
    say(f"case 2-D chunks {kind} {rows}")
    monkeypatch.setenv("LBM_OFFSET64", "1" if kind.endswith("off64") else "0")
    L = _pkg.load()
    rng = np.random.default_rng(616)
    ni, nj = 40, 32
    mask = (rng.random((nj, ni)) < 0.15).astype(np.uint8)
    mask[:2] = 0
    mask[-2:] = 0
    kw = dict(dims=2, ni=ni, nj=nj, nsubs=2, tau=(0.9, 0.75), zeroconcgrad_n=1, zeroconcgrad_s=1, **ROWS[rows],
              **KIND[kind])
    f, gg = random_state(rng, 9, ni * nj, 2)
    lats = []
    for _ in range(2):
        lat = L.Lattice(mask=mask, **kw)
        lat.upload_f(0, f)
        lat.upload_f(1, gg)
        lats.append(lat)
    a, b = lats
    for n in (150, 1, 200, 1, 129):
        if n == 1:
            a.step()
        else:
            a.run(n, write_last=True)
        for q in range(n):
            b.step(n > 1 and q == n - 1)
        for s in range(2):
            assert np.array_equal(a.download_f(s), b.download_f(s)), (n, s)
            if n > 1:
                assert all(np.array_equal(x, y) for x, y in zip(a.mv(s), b.mv(s))), (n, s)
    a.close()
    b.close()
