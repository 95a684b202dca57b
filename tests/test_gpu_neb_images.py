"""Fields and energies of a band's images with demag: the kernels of a term
signature, the slot form and the term list (a zero second anisotropy) are the
same sums in another order of the terms.

Tolerance: rounding of one evaluation, 1e-12 of the energies' size in FP64 and
1e-5 in FP32; states after the first step (the same size for every route) 1e-10
and 1e-5."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu


def _band(n, precision, route):
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(N)
    sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2], pbc="x"), precision=precision)
    Ms = np.full(N, 5.8e5)
    Ms[::11] = 0.0
    mmx.set_Ms(sim, Ms)
    ends = []
    for s in (1.0, -1.0):
        v = 0.3 * rng.standard_normal((N, 3)) + np.array([0.2, 0.4 * s, 1.0])
        ends.append((v / np.linalg.norm(v, axis=1, keepdims=True)).reshape(-1))
    mmx.init_m0(sim, ends[0])
    if route == "slots":
        mmx.add_zeeman(sim, (0, 0, 4e4))
    mmx.add_exch(sim, 1.5e-11)
    mmx.add_dmi(sim, 3e-3, type="interfacial")
    mmx.add_anis(sim, 8e5, axis=(0, 0, 1))
    if route != "slots":
        mmx.add_zeeman(sim, (0, 0, 4e4))
    if route == "list":
        mmx.add_anis(sim, 0.0, axis=(1, 0, 0), name="none")
    mmx.add_demag(sim)
    return mmx.NEB(sim, ends, [3], spring_constant=1e5)


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("n", [(20, 7, 3), (65, 9, 1), (9, 4, 5), (130, 6, 2), (300, 3, 1)])
def test_image_routes_agree(n, precision):
    etol, stol = (1e-12, 1e-10) if precision == mmx.F64 else (1e-5, 1e-5)
    base = _band(n, precision, "signature")
    scale = np.abs(base.energy).max()
    start = np.array(base.energy)
    base.advance(1)
    for route in ("slots", "list"):
        other = _band(n, precision, route)
        assert np.abs(other.energy - start).max() <= etol * scale, route
        other.advance(1)
        assert np.abs(other.spin - base.spin).max() <= stol, route


@pytest.mark.parametrize("n,climb", [((16, 16), -1), ((150, 121), -1), ((260, 137), 2), ((401, 331), -1)])
def test_force_sums_over_many_blocks(n, climb):
    """The force's sums over the blocks of an image (1, 71, 140 and 512 of them),
    which every wave of a stage forms, against the oracle; tolerances of the
    band's trajectory checks."""
    from oracle import OracleSim
    from oracle_neb import OracleNEB

    nx, ny = n
    N, d = nx * ny, 2e-9
    rng = np.random.default_rng(N)
    o = OracleSim(nx, ny, 1, d, d, d, pbc="xy")
    sim = mmx.Sim(mmx.FDMesh(dx=d, dy=d, dz=d, nx=nx, ny=ny, nz=1, pbc="xy"))
    for s in (o, sim):
        Ms, A, H = np.full(N, 3.84e5), 3.25e-12, (0, 0, 1e5)
        if s is sim:
            mmx.set_Ms(s, Ms)
            mmx.add_exch(s, A)
            mmx.add_zeeman(s, H)
        else:
            s.set_Ms(Ms)
            s.add_exch(A)
            s.add_zeeman(H)
    ends = []
    for s in (1.0, -1.0):
        v = 0.2 * rng.standard_normal((N, 3)) + np.array([0.2, 0.4 * s, 1.0])
        ends.append((v / np.linalg.norm(v, axis=1, keepdims=True)).reshape(-1))
    on = OracleNEB(o, ends, [3], spring_constant=1e5, climbing_image=climb, pins=np.zeros(N, dtype=bool))
    gn = mmx.NEB(sim, ends, [3], spring_constant=1e5, clib_image=climb)
    for _ in range(2):
        on.advance_step()
        gn.advance(1)
        assert abs(gn.state["step"] - on.step) <= 1e-9 * on.step
        assert np.abs(gn.spin - on.spin).max() < 1e-10
