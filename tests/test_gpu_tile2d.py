"""2-D runs of several steps per launch (k_tile2d, k_sweep2d) against the FP64
oracle.

lbm_run advances FP64 D2Q9 lattices by even numbers of steps in LDS tiles;
the arithmetic is that of the half-steps, so every run must equal the oracle
bit for bit: tiles that wrap around the lattice, partial tiles, runs that
start and end at either parity, row conditions on open rows and on rows whose
wrapped source is solid, prescribed values that change every step, a solute
window that opens and closes inside a launch."""
import numpy as np
import pytest

from test_gpu_parity import build_pair, load_both, random_state, say

pytestmark = pytest.mark.gpu

ROWS = dict(pressure_s_in=(1, 0), pressure_n_out=(1, 0), rho_in=1.002, rho_out=0.999)
GRAD = dict(zeroconcgrad_n=1, zeroconcgrad_s=1)
T = np.arange(13)
CASES = {
    "flow": dict(nsubs=1, gaccel=(1e-4, -2e-4, 0, 0, 0, 0)),
    "solute": dict(nsubs=2, sink=1e-3),
    "walsh": dict(nsubs=1, walsh=True),
    "walsh_solute_rows": dict(nsubs=2, walsh=True, open_rows=True, **ROWS, **GRAD),
    "rows": dict(nsubs=2, open_rows=True, **ROWS, **GRAD),
    "rows_beside_solids": dict(nsubs=2, **ROWS, **GRAD),
    "flow_rows_beside_solids": dict(nsubs=1, **ROWS),
    "velocity": dict(nsubs=2, velocity_s_in=1, pressure_n_out=(1, 0), uy_in=2e-3, **GRAD),
    "series_ramp": dict(nsubs=2, sink=1e-4, pressure_n_in=(2, 0), pressure_s_in=(2, 0), pfadd=1.0, pfmul=0.1,
                        pressure_n_series=(0.01 * np.sin(T), None), pressure_s_series=(0.01 * np.cos(T), None),
                        bc_ramp_start=3, bc_ramp_stop=20, **GRAD),
    "series_open": dict(nsubs=2, open_rows=True, pressure_n_in=(2, 0), pressure_s_in=(2, 0), pfadd=1.0, pfmul=0.1,
                        pressure_n_series=(0.01 * np.sin(T), None), pressure_s_series=(0.01 * np.cos(T), None), **GRAD),
    "window_open": dict(nsubs=2, open_rows=True, sigma_t_on=6, sigma_t_off=21, **ROWS, **GRAD),
    "window": dict(nsubs=2, sigma_t_on=6, sigma_t_off=31, **ROWS, **GRAD),
}


def run_both(case, ni, nj, runs):
    kw = dict(CASES[case])
    walsh, open_rows = kw.pop("walsh", False), kw.pop("open_rows", False)
    rng = np.random.default_rng(ni * 1000 + nj)
    mask = (rng.random((nj, ni)) < 0.2).astype(np.uint8)
    mask[nj // 2, ni // 2] = 0
    if open_rows:
        mask[0] = mask[-1] = 0
    o, g = build_pair(mask, dims=2, ni=ni, nj=nj, tau=(0.8, 0.75), **kw)
    if walsh:
        ns = rng.uniform(0.0, 1.0, (nj, ni))
        o.set_ns(ns)
        g.set_ns(ns)
    f, gg = random_state(rng, 9, mask.size, kw["nsubs"])
    load_both(o, g, f, gg)
    fl = mask.reshape(-1) != 1
    for n, write in runs:
        o.run(n, write_last=bool(write))
        g.run(n, write_last=write)
        for s in range(kw["nsubs"]):
            assert np.array_equal(g.download_f(s)[:, fl], o.get_f(s)[:, fl]), (case, n, s)
            assert all(np.array_equal(a[fl], b[fl]) for a, b in zip(g.mv(s)[:3], o.mv(s)[:3])), (case, n, s)
    g.close()


@pytest.mark.parametrize("ni,nj", [(1, 5), (7, 3), (33, 40), (149, 83)])
@pytest.mark.parametrize("case", list(CASES))
def test_tiled_runs_match_oracle(case, ni, nj):
    say(f"case tiled run {case} {ni}x{nj}")
    run_both(case, ni, nj, ((1, 1), (2, 1), (9, 1), (26, 1), (5, 0), (16, 1)))


@pytest.mark.parametrize("case,ni,nj", [("solute", 1201, 967), ("rows", 1201, 967), ("walsh_solute_rows", 1201, 967),
                                        ("series_open", 1201, 967), ("window_open", 1201, 967), ("rows", 109, 10900),
                                        ("rows", 11003, 105), ("rows_beside_solids", 1201, 967)])
def test_swept_runs_match_oracle(case, ni, nj):
    """lattices above the size from which flow + solute runs sweep strips:
    ragged last strip and piece, one strip, pieces of two rows; rows beside
    solids stay with the tiles"""
    say(f"case swept run {case} {ni}x{nj}")
    run_both(case, ni, nj, ((1, 0), (11, 1), (6, 0), (8, 1)))
