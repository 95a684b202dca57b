"""Transform lengths at the ends of what the demag passes are compiled for, field
against the oracle:

y lengths of 3 and 5 times a power of two from the shortest (48 of 64, ny = 17..24)
to the longest (1280 of 2048, ny = 513..640), on meshes of three layers and, where
two layers do not fit in LDS (FP64), of two; the one-kernel convolution of two
layers whose sequences go through LDS in several batches (Py = 2048, FP32); the z
pass with block barriers (Pz/4 > 64 threads a sequence in FP64, Pz/8 in FP32).

Tolerances: FP64 1e-12 of the largest value as every field check of this path;
FP32 1e-5 (24-bit transforms, a few dozen roundings of 6e-8)."""
import os
import subprocess
import sys

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [(4, 17, 3), (4, 24, 3), (2, 513, 3), (2, 640, 3), (3, 513, 2), (3, 640, 2), (2, 641, 2), (2, 1024, 2),
         (2, 1024, 3), (3, 33, 130), (2, 33, 260), (2, 20, 129), (3, 6, 257)]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", SIZES)
def test_field_vs_oracle(oracle, n, precision):
    import mmx

    print(f"[case] transform length {n} fp{precision}", flush=True)
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(5 * N + precision)
    m0, Ms = rng.standard_normal(3 * N), rng.uniform(4e5, 8e5, N)
    d = (2e-9, 3e-9, 4e-9)
    g = mmx.Sim(mmx.FDMesh(dx=d[0], dy=d[1], dz=d[2], nx=n[0], ny=n[1], nz=n[2]), precision=precision)
    o = oracle.OracleSim(*n, *d)
    mmx.set_Ms(g, Ms)
    mmx.init_m0(g, m0)
    mmx.add_demag(g)
    o.set_Ms(Ms)
    o.init_m0(m0)
    o.add_demag(0, 0, 0)
    hg, ho = mmx.effective_field(g), o.effective_field()
    assert np.max(np.abs(hg - ho)) <= (1e-12 if precision == 64 else 1e-5) * np.max(np.abs(ho))


def _batch_child():
    """Batches whose first plane launch, of more than 64 KB of LDS, is recorded
    into their graph, against the members alone."""
    import mmx

    for n, precision in (((3, 1024, 1), mmx.F64), ((3, 700, 2), mmx.F32)):
        print(f"[case] recorded plane {n} fp{precision}", flush=True)

        def make(q):
            s = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2]), integrator="Heun",
                        precision=precision)
            mmx.set_Ms(s, 5e5 + 1e4 * q)
            mmx.init_m0(s, np.random.default_rng(q).standard_normal(3 * n[0] * n[1] * n[2]))
            mmx.add_exch(s, 1.3e-11)
            mmx.add_demag(s)
            mmx.set_driver(s, integrator="Heun", step=1e-14)
            return s

        members, alone = [make(q) for q in range(3)], [make(q) for q in range(3)]
        batch = mmx.Batch(members)
        for steps in (4, 2):
            batch.advance(steps)
            for s in alone:
                mmx.run_step(s, n=steps)
            for a, b in zip(alone, members):
                assert np.array_equal(a.spin, b.spin)
    print("[done]", flush=True)


def test_large_plane_first_launched_in_a_recorded_graph():
    """In a process of its own, so that no launch before set the kernels' LDS limit."""
    import mmx

    r = subprocess.run([sys.executable, os.path.abspath(__file__)], capture_output=True, text=True, timeout=100,
                       env=dict(os.environ, PYTHONPATH=os.path.dirname(os.path.dirname(mmx.__file__))))
    print(r.stdout[-1000:], r.stderr[-2000:], flush=True)
    assert r.returncode == 0 and "[done]" in r.stdout


if __name__ == "__main__":
    _batch_child()
