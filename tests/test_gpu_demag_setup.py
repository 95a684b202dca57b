"""A demag set-up that runs out of device memory leaves the simulation as it
was: the call says so, the other terms go on, and a later call succeeds with
the same bits as on a new simulation.

A small library stands before the HIP runtime in a child process and lets the
k-th allocation of the set-up fail, for every k."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# hipMalloc that fails once, at the countdown's end (2: hipErrorOutOfMemory)
GATE = r"""
#include <dlfcn.h>
#include <stddef.h>
static int left = 0;
static int calls = 0;
void gate_arm(int k) { left = k; calls = 0; }
int gate_calls(void) { return calls; }
int hipMalloc(void **p, size_t n)
{
    static int (*real)(void **, size_t);
    if (!real) real = (int (*)(void **, size_t))dlsym(dlopen(GATE_HIP, RTLD_NOW), "hipMalloc");
    calls++;
    if (left > 0 && --left == 0) return 2;
    return real(p, n);
}
"""


def _child(gate, out):
    import ctypes

    g = ctypes.CDLL(gate, mode=ctypes.RTLD_GLOBAL)  # before libmmx is loaded
    import mmx

    res = {}

    def make(n, precision):
        N = n[0] * n[1] * n[2]
        rng = np.random.default_rng(N)
        s = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=3e-9, dz=4e-9, nx=n[0], ny=n[1], nz=n[2]), precision=precision)
        mmx.set_Ms(s, rng.uniform(4e5, 8e5, N))
        mmx.init_m0(s, rng.standard_normal(3 * N))
        mmx.add_exch(s, 1.3e-11)
        return s

    # one and two layers (one-kernel convolution), three (separate passes), a y
    # length of 5/8 of a power of two, a mesh whose last pass has more blocks
    # than the local kernels
    for n in ((40, 30, 1), (12, 9, 2), (12, 9, 3), (5, 40, 4), (2, 600, 15)):
        for precision in (mmx.F64, mmx.F32):
            ref = make(n, precision)
            h0, e0 = mmx.effective_field(ref), mmx.compute_system_energy(ref)
            g.gate_arm(0)
            mmx.add_demag(ref)
            total = g.gate_calls()
            h1 = mmx.effective_field(ref)
            e1 = mmx.compute_system_energy(ref)
            for k in range(1, total + 1):
                print(f"[case] set-up {n} fp{precision} allocation {k} of {total}", flush=True)
                s = make(n, precision)
                mmx.effective_field(s)
                g.gate_arm(k)
                try:
                    mmx.add_demag(s)
                    code = 0
                except mmx._lib.MmxError as e:
                    code = e.code
                g.gate_arm(0)
                assert code == mmx._lib.ENOMEM, (n, precision, k, code)
                assert np.array_equal(mmx.effective_field(s), h0), (n, precision, k)
                assert np.array_equal(mmx.compute_system_energy(s), e0), (n, precision, k)
                mmx.add_demag(s)
                assert np.array_equal(mmx.effective_field(s), h1), (n, precision, k)
                assert np.array_equal(mmx.compute_system_energy(s), e1), (n, precision, k)
            res[f"{n} {precision}"] = total
    with open(out, "w") as f:
        f.write(repr(res))


def test_failed_setup_leaves_no_state(tmp_path):
    import mmx

    src, lib, out = tmp_path / "gate.c", tmp_path / "libgate.so", tmp_path / "out"
    src.write_text(GATE)
    hip = os.environ.get("MMX_HIP_LIBRARY", "libamdhip64.so")
    subprocess.run(["gcc", "-O1", "-shared", "-fPIC", f'-DGATE_HIP="{hip}"', str(src), "-o", str(lib), "-ldl"],
                   check=True)
    r = subprocess.run([sys.executable, os.path.abspath(__file__), str(lib), str(out)], capture_output=True, text=True,
                       timeout=100, env=dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(mmx.__file__))))
    print(r.stdout[-2000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0
    assert min(eval(out.read_text()).values()) >= 9  # the gate was there


if __name__ == "__main__":
    _child(sys.argv[1], sys.argv[2])
