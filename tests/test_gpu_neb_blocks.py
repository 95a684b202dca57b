"""Bands of so many blocks that a block of the stage takes two or four shares of
the cells (launch_neb_stage: 2560 and 5120 blocks), on each side of the two
limits and with a last block that has fewer, against the oracle.

Tolerances: those of the band's trajectory checks (step size 1e-9, states
1e-10 in FP64, 1e-5 in FP32)."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
# 353 blocks per image of 300x301 cells: 2471, 2824, 4942, 5295 blocks
@pytest.mark.parametrize("images", [7, 8, 14, 15])
def test_stage_shares_vs_oracle(images, precision):
    from oracle import OracleSim
    from oracle_neb import OracleNEB

    nx, ny, d = 300, 301, 2e-9
    N = nx * ny
    rng = np.random.default_rng(images)
    Ms, A, H = np.full(N, 3.84e5), 3.25e-12, (0, 0, 1e5)
    o = OracleSim(nx, ny, 1, d, d, d, pbc="xy")
    o.set_Ms(Ms)
    o.add_exch(A)
    o.add_zeeman(H)
    sim = mmx.Sim(mmx.FDMesh(dx=d, dy=d, dz=d, nx=nx, ny=ny, nz=1, pbc="xy"), precision=precision)
    mmx.set_Ms(sim, Ms)
    mmx.add_exch(sim, A)
    mmx.add_zeeman(sim, H)
    ends = []
    for s in (1.0, -1.0):
        v = 0.2 * rng.standard_normal((N, 3)) + np.array([0.2, 0.4 * s, 1.0])
        ends.append((v / np.linalg.norm(v, axis=1, keepdims=True)).reshape(-1))
    on = OracleNEB(o, ends, [images], spring_constant=1e5, pins=np.zeros(N, dtype=bool))
    gn = mmx.NEB(sim, ends, [images], spring_constant=1e5)
    print(f"[case] band of {images} images fp{precision}", flush=True)
    on.advance_step()
    gn.advance(1)
    f64 = precision == mmx.F64
    assert abs(gn.state["step"] - on.step) <= (1e-9 if f64 else 1e-3) * on.step
    assert np.abs(gn.spin - on.spin).max() < (1e-10 if f64 else 1e-5)
