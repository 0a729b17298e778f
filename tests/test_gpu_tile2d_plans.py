"""2-D runs of several steps per launch between the smallest lattices and those
swept in strips, against the FP64 oracle, bit for bit: each plan and kernel
form that a lattice of 2.5e4 to 1.2e6 nodes gets on 256 compute units.

form (KEEP: one tile per CU, one node per thread)   lattices here
flow, 8 steps, one tile per CU, not KEEP             413 x 307
flow, 10 steps, handed-on rows, halo 15, not KEEP    126 x 124
flow, second round of tiles                          480 x 340
flow, 32 x 16 cores, with and without partial
  bounce-back, open and handed-on rows               500 x 480, 601 x 499
flow + solute, 6 steps, KEEP                         300 x 200
flow + solute, second round of tiles, not KEEP       307 x 293, 421 x 303
flow + solute, largest square cores, open and
  handed-on rows, with partial bounce-back, resting
  solute                                             600 x 500
strips: one of 97 columns in pieces of 47 rows;
  resting solute with and without partial
  bounce-back                                        97 x 12000, 1201 x 967"""
import pytest

import test_gpu_tile2d as tile2d
from test_gpu_parity import say

pytestmark = pytest.mark.gpu

REST = dict(nsubs=2, sigma_t_on=1000, sigma_t_off=2000)
MORE = {
    "flow_rows_open": dict(nsubs=1, open_rows=True, **tile2d.ROWS),
    "walsh_rows_open": dict(nsubs=1, walsh=True, open_rows=True, **tile2d.ROWS),
    "rest": REST,
    "rest_walsh": dict(walsh=True, **REST),
    "rest_rows": dict(open_rows=True, **REST, **tile2d.ROWS, **tile2d.GRAD),
    "rest_rows_beside_solids": dict(**REST, **tile2d.ROWS, **tile2d.GRAD),
}

PLANS = [("flow", 413, 307), ("walsh", 413, 307), ("flow_rows_open", 413, 307), ("flow_rows_beside_solids", 126, 124),
         ("flow", 480, 340), ("walsh_rows_open", 480, 340),
         ("flow", 500, 480), ("walsh", 500, 480), ("flow_rows_open", 500, 480), ("walsh_rows_open", 601, 499),
         ("flow_rows_beside_solids", 601, 499),
         ("solute", 300, 200), ("rows", 307, 293), ("walsh_solute_rows", 300, 200), ("rest", 307, 293),
         ("solute", 600, 500), ("rows", 600, 500), ("walsh_solute_rows", 600, 500), ("rows_beside_solids", 600, 500),
         ("rest", 600, 500), ("rest_walsh", 600, 500), ("rest_rows", 600, 500), ("rest_rows_beside_solids", 600, 500),
         ("rows", 421, 303), ("rest_walsh", 421, 303), ("window_open", 600, 500),
         ("rows", 97, 12000), ("rest", 1201, 967), ("rest_walsh", 1201, 967), ("rest_rows", 1201, 967)]


@pytest.mark.parametrize("case,ni,nj", PLANS)
def test_plans_match_oracle(case, ni, nj, monkeypatch):
    say(f"case planned run {case} {ni}x{nj}")
    for name, kw in MORE.items():
        monkeypatch.setitem(tile2d.CASES, name, kw)
    # launches of every length a plan allows, odd steps between them
    tile2d.run_both(case, ni, nj, ((1, 0), (21, 1), (6, 0), (4, 1), (2, 0), (9, 1)))
