"""Tables whose launch the runtime refuses are not read: in a process where a
chosen kernel launch is refused (a definition of hipLaunchKernel, loaded before
the library, that passes all others on), the run whose table is missing gives
the fields of the same steps launched one by one, and so does the run after
it."""
import os
import subprocess
import sys

import pytest

import _pkg

pytestmark = pytest.mark.gpu

REFUSE = r'''
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>
static int armed, refusals;
static hipError_t pending = hipSuccess;
static void *real(const char *name) {
  static void *lib = dlopen("libamdhip64.so.7", RTLD_NOW | RTLD_NOLOAD);
  return dlsym(lib, name);
}
extern "C" hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **a, size_t m, hipStream_t s) {
  static auto *fn = (hipError_t(*)(const void *, dim3, dim3, void **, size_t, hipStream_t))real("hipLaunchKernel");
  if (armed && --armed == 0) {
    refusals++;
    return pending = hipErrorOutOfMemory;
  }
  return fn(f, g, b, a, m, s);
}
extern "C" hipError_t hipGetLastError() {
  static auto *fn = (hipError_t(*)())real("hipGetLastError");
  const hipError_t e = pending;
  pending = hipSuccess;
  return e != hipSuccess ? e : fn();
}
extern "C" void arm(int n) { armed = n; }
extern "C" int refused() { return refusals; }
'''

WORK = r'''
import ctypes, sys
sys.path.insert(0, sys.argv[1])
refuse = ctypes.CDLL(sys.argv[2], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import _pkg
L = _pkg.load()
rng = np.random.default_rng(5)

def check(n, shape, **kw):
    """runs of n steps, the first launch of the first one refused, against
    single steps"""
    mask = (rng.random(shape) < 0.1).astype(np.uint8)
    mask[:2] = mask[-2:] = 0
    kw.update(dims=len(shape), ni=shape[-1], nj=shape[-2], nk=shape[0] if len(shape) == 3 else 1, nsubs=2, tau=(0.8, 0.75))
    a, b = L.Lattice(mask=mask, **kw), L.Lattice(mask=mask, **kw)
    f = [rng.uniform(-1e-3, 1e-3, (a.Q, a.N)), rng.uniform(0, 0.1, (a.Q, a.N))]
    for g in (a, b):
        for s in range(2):
            g.upload_f(s, f[s])
    before = refuse.refused()
    for run in range(3):
        refuse.arm(1 if run == 0 else 0)
        a.run(n)
        for q in range(n):
            b.step(q == n - 1)
        for s in range(2):
            assert np.array_equal(a.download_f(s), b.download_f(s)), (shape, run, s)
            assert all(np.array_equal(x, y) for x, y in zip(a.mv(s), b.mv(s))), (shape, run, s)
    assert refuse.refused() == before + 1, "the refusal was not reached"
    a.close()
    b.close()

rows = dict(pressure_s_in=(1, 0), pressure_n_out=(1, 0), rho_in=1.002, rho_out=0.999, zeroconcgrad_n=1, zeroconcgrad_s=1)
check(130, (12, 14, 16), gaccel=(1e-5, 0, 2e-5, 0, 0, 0))  # the location table
check(4, (40, 44), **rows)  # tiles
check(4, (1100, 1060), **rows)  # strips
print("ok")
'''


def test_tables_of_refused_launches_are_not_read(tmp_path):
    src, so, work = tmp_path / "refuse.cpp", tmp_path / "refuse.so", tmp_path / "work.py"
    src.write_text(REFUSE)
    work.write_text(WORK)
    subprocess.run(["g++", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", "/opt/rocm/include", "-o", str(so),
                    str(src), "-ldl"], check=True)
    here = os.path.dirname(os.path.abspath(__file__))
    out = subprocess.run([sys.executable, str(work), here, str(so)], capture_output=True, text=True, timeout=110)
    assert out.returncode == 0, out.stdout + out.stderr
    assert out.stdout.split()[-1] == "ok"
