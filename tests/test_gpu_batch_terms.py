"""Batches whose members all have exchange, interfacial DMI, uniaxial anisotropy
and a uniform field, any of them a stochastic field on top, take kernels
compiled for these terms that draw the stochastic field once per step.  Every
member must land bit for bit where it lands alone, as must members of batches
that these kernels do not cover, meshes one cell wide, cells without moment and
members whose terms change after the batch was made."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

SIZES = [(1, 7, 5), (9, 1, 4), (33, 20, 3), (64, 16, 1), (5, 3, 1), (70, 41, 6)]


def _members(integrator, precision, covered):
    rng = np.random.default_rng(11)
    out = []
    for q, n in enumerate(SIZES):
        N = n[0] * n[1] * n[2]
        sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2], pbc=("", "xy", "x")[q % 3]),
                      integrator=integrator, precision=precision)
        Ms = np.full(N, 6e5 + 1e5 * q)
        Ms[:: 5 + q] = 0.0
        mmx.set_Ms(sim, Ms)
        mmx.init_m0(sim, rng.standard_normal(3 * N))
        if not covered and q == 2:  # another order of the terms
            mmx.add_zeeman(sim, (0, 0, 4e4))
        mmx.add_exch(sim, 1e-11 + 1e-12 * q)
        mmx.add_dmi(sim, 2e-3, type="interfacial")
        mmx.add_anis(sim, 5e5, axis=(0, 0, 1), name="Ku")
        if covered or q != 2:
            mmx.add_zeeman(sim, (0, 0, 4e4))
        if q % 2:
            mmx.add_thermal_noise(sim, 300.0 if q < 4 else rng.uniform(100.0, 300.0, N), seed=5 + q)
        mmx.set_driver(sim, integrator=integrator, step=1e-14)
        out.append(sim)
    return out


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("integrator", ["RungeKutta", "Heun"])
@pytest.mark.parametrize("covered", [True, False])
def test_batch_terms_match_members_alone(integrator, precision, covered):
    together = _members(integrator, precision, covered)
    alone = _members(integrator, precision, covered)
    batch = mmx.Batch(together)
    for steps in (3, 2):
        batch.advance(steps)
        for a in alone:
            mmx.run_step(a, n=steps)
        for q, (b, a) in enumerate(zip(together, alone)):
            assert np.array_equal(b.spin, a.spin), (q, SIZES[q])
        # from here on one member has a per-cell Ku, which those kernels do not take
        Ku = np.linspace(3e5, 6e5, 64 * 16)
        for s in (together[3], alone[3]):
            mmx.update_anis(s, Ku, name="Ku")
