"""Batches of members without a term signature, none, some or all of them with a
stochastic field, or with one added after the batch was made: each member lands
bit for bit where it lands alone."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

SIZES = [(7, 5, 3), (33, 20, 2), (64, 9, 1), (1, 40, 4)]


def _members(integrator, precision, thermal):
    rng = np.random.default_rng(5)
    out = []
    for q, n in enumerate(SIZES):
        N = n[0] * n[1] * n[2]
        sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2], pbc=("x", "")[q % 2]),
                      integrator=integrator, precision=precision)
        Ms = np.full(N, 6e5)
        Ms[:: 6 + q] = 0.0
        mmx.set_Ms(sim, Ms)
        mmx.init_m0(sim, rng.standard_normal(3 * N))
        mmx.add_zeeman(sim, (0, 0, 4e4))  # before the exchange: no signature
        mmx.add_exch(sim, 1e-11)
        mmx.add_anis(sim, 5e5, axis=(0, 0, 1))
        if q in thermal:
            mmx.add_thermal_noise(sim, 300.0, seed=9 + q)
        mmx.set_driver(sim, integrator=integrator, step=1e-14)
        out.append(sim)
    return out


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("integrator", ["RungeKutta", "Heun"])
@pytest.mark.parametrize("thermal", [(), (1,), (0, 1, 2, 3)])
def test_members_land_where_they_land_alone(integrator, precision, thermal):
    print(f"[case] batch noise {integrator} fp{precision} {thermal}", flush=True)
    together, alone = (_members(integrator, precision, thermal) for _ in range(2))
    batch = mmx.Batch(together)
    for steps in (3, 2):
        batch.advance(steps)
        for a in alone:
            mmx.run_step(a, n=steps)
        for q, (b, a) in enumerate(zip(together, alone)):
            assert np.array_equal(b.spin, a.spin), (q, SIZES[q])
        if steps == 3 and 2 not in thermal:  # from here on the third member has one too
            for s in (together[2], alone[2]):
                mmx.add_thermal_noise(s, 200.0, seed=77)
