"""Transfers and samples where the system pins no host memory: in a process
whose hipHostMalloc is refused (a definition of it, loaded before the library,
that always fails) populations, fields and samples still go both ways, as
ordinary copies do."""
import os
import subprocess
import sys

import pytest

import _pkg

pytestmark = pytest.mark.gpu

REFUSE = r'''
#include <stddef.h>
static int calls;
int hipHostMalloc(void **p, size_t n, unsigned flags) {
  (void)n, (void)flags, calls++;
  *p = 0;
  return 2; /* hipErrorOutOfMemory */
}
int refused(void) { return calls; }
'''

WORK = r'''
import ctypes, sys
sys.path.insert(0, sys.argv[1])
refuse = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import _pkg
L = _pkg.load()
rng = np.random.default_rng(5)
for shape in ((3, 5), (33, 40), (19, 23, 29), (70, 80, 90)):
    mask = (rng.random(shape) < 0.3).astype(np.uint8)
    fl = mask.reshape(-1) != 1
    g = L.Lattice(mask=mask, dims=len(shape), ni=shape[-1], nj=shape[-2], nk=shape[0] if len(shape) == 3 else 1,
                  nsubs=2, tau=(0.8, 0.75))
    for s in range(2):
        f = rng.standard_normal((g.Q, g.N))
        g.upload_f(s, f)
        assert np.array_equal(g.download_f(s), f * fl), (shape, s)
        fields = rng.standard_normal((1 + g.dims, g.N))
        g.set_mv(s, *fields)
        got = g.mv(s)
        for c in range(4):
            assert np.array_equal(got[c], fields[c] * fl if c <= g.dims else np.zeros(g.N)), (shape, s, c)
        at = rng.integers(0, g.N, 5000)
        assert np.array_equal(g.sample_mv(s, at)[:, :1 + g.dims], np.stack(got, 1)[at][:, :1 + g.dims])
    # the buffer the copies went through serves reductions again
    assert abs(g.reduce_sums()[1] - g.mv(0)[1].sum()) <= 1e-9 * g.N
    g.close()
assert refuse.refused() > 0, "the refusal was not reached"
print("ok")
'''


def test_without_pinned_memory(tmp_path):
    src, so, work = tmp_path / "refuse.c", tmp_path / "refuse.so", tmp_path / "work.py"
    src.write_text(REFUSE)
    work.write_text(WORK)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    out = subprocess.run([sys.executable, str(work), here, str(so)], capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split()[-1] == "ok"
