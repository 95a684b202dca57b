"""Fields and energies of a band's images with demag for every kind of term the
slot form holds: uniform and per-cell exchange, DMI, anisotropy, cubic anisotropy
and field.  The slot form and the term list (taken with a second anisotropy of
zero) evaluate the same sums in the same order of the terms.

Tolerance: rounding of one evaluation, 1e-12 of the energies' size in FP64 and
1e-5 in FP32; states after the first step (the same size for both) 1e-10 and
1e-5."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu


def _terms(sim, kind, N, rng):
    if kind == "bulk":
        mmx.add_exch(sim, 1.3e-11)
        mmx.add_dmi(sim, 2e-3, type="bulk")
        mmx.add_cubic_anis(sim, -5e4)
        mmx.add_zeeman(sim, (0, 0, 4e4))
    elif kind == "bulk-vector":
        mmx.add_exch(sim, rng.uniform(1e-11, 2e-11, N))
        mmx.add_dmi(sim, (1e-3, 2e-3, -1.5e-3), type="bulk")
        mmx.add_cubic_anis(sim, rng.uniform(-5e4, 5e4, N))
    else:
        axis = rng.standard_normal((N, 3))
        mmx.add_zeeman(sim, rng.uniform(-5e4, 5e4, 3 * N))
        mmx.add_exch(sim, rng.uniform(1e-11, 2e-11, N))
        mmx.add_dmi(sim, rng.uniform(1e-3, 3e-3, N), type="interfacial")
        mmx.add_anis(sim, rng.uniform(1e5, 8e5, N),
                     axis=(axis / np.linalg.norm(axis, axis=1, keepdims=True)).reshape(-1), name="Ku")


def _band(n, precision, kind, term_list):
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(N)
    sim = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=n[0], ny=n[1], nz=n[2], pbc="y"), precision=precision)
    Ms = rng.uniform(4e5, 6e5, N)
    Ms[::11] = 0.0
    mmx.set_Ms(sim, Ms)
    ends = []
    for s in (1.0, -1.0):
        v = 0.3 * rng.standard_normal((N, 3)) + np.array([0.2, 0.4 * s, 1.0])
        ends.append((v / np.linalg.norm(v, axis=1, keepdims=True)).reshape(-1))
    mmx.init_m0(sim, ends[0])
    _terms(sim, kind, N, rng)
    mmx.add_demag(sim)
    if term_list:
        mmx.add_anis(sim, 0.0, axis=(1, 0, 0), name="none")
        mmx.add_anis(sim, 0.0, axis=(0, 1, 0), name="nothing")
    return mmx.NEB(sim, ends, [3], spring_constant=1e5, clib_image=2)


@pytest.mark.parametrize("precision", [mmx.F64, mmx.F32])
@pytest.mark.parametrize("kind", ["bulk", "bulk-vector", "cells"])
@pytest.mark.parametrize("n", [(20, 7, 3), (65, 9, 1), (1100, 3, 1)])
def test_image_energies_of_every_term(n, kind, precision):
    print(f"[case] image terms {kind} {n} fp{precision}", flush=True)
    etol, stol = (1e-12, 1e-10) if precision == mmx.F64 else (1e-5, 1e-5)
    slot, list_ = (_band(n, precision, kind, t) for t in (False, True))
    a, b = np.array(slot.energy), np.array(list_.energy)
    assert np.abs(a - b).max() <= etol * np.abs(b).max()
    slot.advance(1)
    list_.advance(1)
    assert np.abs(slot.spin - list_.spin).max() <= stol
