"""A PME evaluation whose transform fails returns an error and leaves no atom
in the bins: the next evaluation gives the bits of an undisturbed one, also
with atoms beyond their bucket.  The failure is made on the host, by a library
that stands before hipFFT and returns HIPFFT_EXEC_FAILED once, in a process of
its own; every kernel that is launched runs to its end."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

FAILING = r"""
typedef int (*exec_t)(void *, void *, void *);
static exec_t d2z, z2d;
static int fail_d2z, fail_z2d;
void set_up(void *a, void *b) { d2z = (exec_t)a; z2d = (exec_t)b; }
void set_fail(int a, int b) { fail_d2z = a; fail_z2d = b; }
int hipfftExecD2Z(void *p, void *i, void *o) {
  if (fail_d2z > 0) { fail_d2z--; return 6; }
  return d2z(p, i, o);
}
int hipfftExecZ2D(void *p, void *i, void *o) {
  if (fail_z2d > 0) { fail_z2d--; return 6; }
  return z2d(p, i, o);
}
"""

CHILD = r"""
import ctypes, sys
stub = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import torch
from protomoladdon_amd import _lib, systems
from protomoladdon_amd.pme import NonbondedPMEwaldKSpace

lib = _lib.load()
with open("/proc/self/maps") as maps:
    real = [l.split()[-1] for l in maps if "libhipfft.so" in l]
real = [p for p in real if p.startswith("/opt/rocm")] or real
fft = ctypes.CDLL(real[0])
adr = lambda f: ctypes.cast(f, ctypes.c_void_p)
stub.set_up(adr(fft.hipfftExecD2Z), adr(fft.hipfftExecZ2D))

w = systems.small_water(n_mol=300, elec="coulomb")
w.positions = 0.2 * w.positions
force = w.make_force("fp64")
ks = NonbondedPMEwaldKSpace(force, (24, 24, 24), 9.0, order=4, alpha=0.35)
x = torch.tensor(w.positions, dtype=torch.float64, device="cuda:0")

def run():
    f = torch.zeros_like(x)
    out = torch.zeros(20, dtype=torch.float64, device="cuda:0")
    ks.evaluate_device(w.topology, x, f, out, flags=1)
    torch.cuda.synchronize()
    return f.cpu().numpy(), out.cpu().numpy()

ref = run()
assert np.abs(ref[0]).max() > 0
for which in ((1, 0), (0, 1)):
    for k in range(3):
        stub.set_fail(*which)
        try:
            run()
        except _lib.PmnbError as e:
            assert "hipFFT" in str(e), e
        else:
            raise SystemExit("the failing transform was not called")
        torch.cuda.synchronize()
    got = run()
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
ks.close()
force.close()
print("PME_AFTER_FAILURE_OK", flush=True)
"""


def test_evaluation_after_a_failed_transform(tmp_path):
    src, so = tmp_path / "failing.c", tmp_path / "libfailing.so"
    src.write_text(FAILING)
    subprocess.run(["gcc", "-shared", "-fPIC", "-o", str(so), str(src)],
                   check=True)
    env = dict(os.environ)
    env["PYTHONPATH"] = ROOT + os.pathsep + env.get("PYTHONPATH", "")
    r = subprocess.run([sys.executable, "-u", "-c", CHILD, str(so)], cwd=ROOT,
                       env=env, capture_output=True, text=True, timeout=100)
    assert "PME_AFTER_FAILURE_OK" in r.stdout, r.stdout + r.stderr
