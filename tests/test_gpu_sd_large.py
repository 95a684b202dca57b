"""Steepest descent on meshes whose three block sums per step outgrow one value
per block of the largest launch (704 512 cells and more), and beyond the largest
number of blocks, against the oracle's restatement.

Tolerances: those of the small meshes' steps (tests/test_gpu_sd.py)."""
import numpy as np
import pytest

import mmx
from oracle import OracleSim
from oracle_sd import OracleSD

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [(1009, 701), (1500, 1451)])  # 2763 blocks; more cells than 8192 blocks' threads
def test_sd_steps_of_large_mesh(n):
    print(f"[case] steepest descent {n}", flush=True)
    nx, ny, d = n[0], n[1], 2.5e-9
    N = nx * ny
    rng = np.random.default_rng(N)
    m0 = np.array([1.0, 0.3, 0.2]) + 0.4 * rng.standard_normal((N, 3))
    o = OracleSim(nx, ny, 1, d, d, d)
    o.set_Ms(8e5)
    o.init_m0(m0.reshape(-1))
    o.add_exch(1.3e-11)
    o.add_anis(np.full(N, 5e4), axis=(0, 0, 1))
    sim = mmx.Sim(mmx.FDMesh(dx=d, dy=d, dz=d, nx=nx, ny=ny, nz=1), driver="SD")
    mmx.set_Ms(sim, 8e5)
    mmx.init_m0(sim, m0.reshape(-1))
    mmx.add_exch(sim, 1.3e-11)
    mmx.add_anis(sim, 5e4, axis=(0, 0, 1))
    osd = OracleSD(o, pins=np.zeros(N, dtype=bool))
    for i in range(5):
        osd.run_step()
        mmx.run_step(sim)
        tau = sim._integrator.step
        assert abs(tau - osd.tau) <= 1e-9 * osd.tau, (i, tau, osd.tau)
    assert np.abs(sim.spin - osd.spin.reshape(-1)).max() < 1e-9
