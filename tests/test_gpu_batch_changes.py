"""A batch whose members change after it was made (a second term of a kind, which
the slot form does not hold; a demag term; another step; another scheme for all
of them): every member lands bit for bit where it lands alone."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

SIZES = [(9, 7, 4), (16, 5, 3), (9, 7, 4)]


def _members(integrator, precision, demag):
    rng = np.random.default_rng(3)
    out = []
    for q, n in enumerate(SIZES):
        N = n[0] * n[1] * n[2]
        sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2]), integrator=integrator,
                      precision=precision)
        mmx.set_Ms(sim, 6e5 + 1e4 * q)
        mmx.init_m0(sim, rng.standard_normal(3 * N))
        mmx.add_exch(sim, 1e-11)
        mmx.add_anis(sim, 5e5, axis=(0, 0, 1))
        if demag:
            mmx.add_demag(sim)
        mmx.set_driver(sim, integrator=integrator, step=1e-14)
        out.append(sim)
    return out


CHANGES = {
    "second anisotropy": lambda s: mmx.add_anis(s[1], 3e5, axis=(1, 0, 0), name="second"),
    "demag": lambda s: mmx.add_demag(s[1]) if not any(t.name == "demag" for t in s[1].interactions) else None,
    "step": lambda s: mmx.set_driver(s[2], integrator=s[2].integrator_name, step=2.5e-14),
    "scheme": lambda s: [mmx.set_driver(q, integrator="RungeKutta", step=1e-14) for q in s],
}


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("demag", [False, True])
@pytest.mark.parametrize("change", list(CHANGES))
def test_changed_members_match_alone(change, demag, precision):
    print(f"[case] batch change {change} demag={demag} fp{precision}", flush=True)
    together, alone = (_members("Heun", precision, demag) for _ in range(2))
    for s in together + alone:
        s.integrator_name = "Heun"
    batch = mmx.Batch(together)
    for steps in (3, 4, 1):
        batch.advance(steps)
        for a in alone:
            mmx.run_step(a, n=steps)
        for q, (b, a) in enumerate(zip(together, alone)):
            assert np.array_equal(b.spin, a.spin), (steps, q)
        if steps == 3:
            CHANGES[change](together)
            CHANGES[change](alone)


def test_time_dependent_member_is_refused():
    """As when the batch is made; the other calls go on."""
    sims = _members("Heun", mmx.F64, False)
    batch = mmx.Batch(sims)
    batch.advance(2)
    mmx.add_zeeman(sims[0], (0, 0, 1e4), lambda t: 1.0)
    with pytest.raises(mmx._lib.MmxError):
        batch.advance(1)
    mmx.run_step(sims[1], n=1)
