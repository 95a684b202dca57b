"""The slot-form last pass at the edges of its launch shapes against the oracle:
4 or 8 elements per thread, threads that take cells only, rows per block with a
remainder, odd rows, rows as long as the transform.

Tolerances: FP64 1e-12 of the largest value after a few steps, as the
trajectory checks of this path; FP32 1e-5 (24-bit arithmetic over 12 to 21
evaluations)."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

SIZES = [(17, 5, 3), (32, 3, 5), (63, 4, 9), (128, 9, 7), (100, 6, 1), (256, 5, 3), (201, 33, 1), (300, 20, 3),
         (512, 3, 2), (120, 70, 20)]


def _pair(oracle, n, precision, maps, integrator, step):
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(N + precision)
    m0 = rng.standard_normal(3 * N)
    d = 2e-9
    D, Ku = (rng.uniform(1e-3, 3e-3, N), rng.uniform(4e5, 8e5, N)) if maps else (3e-3, 8e5)
    H = (0.0, 0.0, 79577.47)
    g = mmx.Sim(mmx.FDMesh(dx=d, dy=d, dz=d, nx=n[0], ny=n[1], nz=n[2], pbc="x"), integrator=integrator,
                precision=precision)
    o = oracle.OracleSim(*n, d, d, d, pbc="x")
    for s in (g, o):
        if s is g:
            mmx.set_Ms(s, 5.8e5)
            mmx.init_m0(s, m0)
            mmx.add_exch(s, 1.5e-11)
            mmx.add_dmi(s, D, type="interfacial")
            mmx.add_anis(s, Ku, axis=(0, 0, 1))
            if not maps:
                mmx.add_zeeman(s, H)
            mmx.add_demag(s)
            mmx.set_driver(s, integrator=integrator, step=step, tol=1e-6)
        else:
            s.set_Ms(np.full(N, 5.8e5))
            s.init_m0(m0)
            s.add_exch(1.5e-11)
            s.add_dmi(np.full(N, D) if not maps else D, type="interfacial")
            s.add_anis(np.full(N, Ku) if not maps else Ku, axis=(0, 0, 1))
            if not maps:
                s.add_zeeman(np.tile(H, N))
            s.add_demag(0, 0, 0)
    return g, o


@pytest.mark.parametrize("maps", [False, True])
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", SIZES)
def test_last_pass_rk4_vs_oracle(oracle, n, precision, maps):
    print(f"[case] last pass {n} fp{precision} maps={maps}", flush=True)
    g, o = _pair(oracle, n, precision, maps, "RungeKutta", 1e-14)
    o.set_integrator(0, step=1e-14)
    mmx.run_step(g, n=3)
    for _ in range(3):
        o.advance_step()
    assert np.max(np.abs(g.spin - o.spin)) <= (1e-12 if precision == 64 else 1e-5)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", SIZES)
def test_last_pass_heun_vs_oracle(oracle, n, precision):
    """A stage combination with an earlier stage."""
    print(f"[case] last pass heun {n} fp{precision}", flush=True)
    g, o = _pair(oracle, n, precision, False, "Heun", 1e-14)
    o.set_integrator(1, step=1e-14)
    mmx.run_step(g, n=3)
    for _ in range(3):
        o.advance_step()
    assert np.max(np.abs(g.spin - o.spin)) <= (1e-12 if precision == 64 else 1e-5)
