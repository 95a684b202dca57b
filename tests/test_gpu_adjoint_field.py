"""The pull-back of an RK4 trajectory recomputes its stages in slot form and
takes their kept field for the dL/dMs of the local terms when no other term is
in it.  A zero Zeeman field (the field is then evaluated for those terms alone)
and a zero second anisotropy (no slot form: the term list) change the route but
no value.

Tolerance: the routes differ by rounding only, accumulated over 12 steps of 8
evaluations: 1e-12 of the largest value in FP64, 2e-5 in FP32."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu


def _grads(n, precision, extra, demag):
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(N)
    sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2], pbc="x"),
                  integrator="RungeKutta", precision=precision)
    Ms = rng.uniform(5e5, 7e5, N)
    Ms[::7] = 0.0
    pins = np.zeros(N, dtype=bool)
    pins[3] = True
    mmx.set_Ms(sim, Ms)
    mmx.set_pinning(sim, pins)
    mmx.init_m0(sim, rng.standard_normal(3 * N))
    mmx.add_exch(sim, 1.5e-11)
    mmx.add_dmi(sim, rng.uniform(1e-3, 3e-3, N), type="interfacial", name="D")
    mmx.add_anis(sim, rng.uniform(4e5, 8e5, N), axis=(0, 0, 1), name="Ku")
    if extra == "zeeman":
        mmx.add_zeeman(sim, (0.0, 0.0, 0.0))
    if extra == "anis":
        mmx.add_anis(sim, 0.0, axis=(1, 0, 0), name="none")
    if demag:
        mmx.add_demag(sim)
    mmx.set_driver(sim, integrator="RungeKutta", step=2e-14)
    m, pullback = mmx.rk4_trajectory_rrule(sim, 12, every=5)
    out = pullback(rng.standard_normal(3 * N) / N)
    return dict(m=m, **{key: out[key] for key in ("m0", "Ms", "D", "Ku")})


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("n,demag", [((20, 7, 3), False), ((65, 9, 1), False), ((1, 5, 4), False), ((12, 6, 2), True)])
def test_adjoint_routes_agree(n, precision, demag):
    tol = 1e-12 if precision == mmx.F64 else 2e-5
    base = _grads(n, precision, None, demag)
    for extra in ("zeeman", "anis"):
        other = _grads(n, precision, extra, demag)
        for key, v in base.items():
            assert np.abs(v - other[key]).max() <= tol * np.abs(v).max(), (extra, key)
