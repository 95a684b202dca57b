"""The one-kernel y/z convolution of films of one or two layers against the
oracle at the edges of its range, and its wider blocks against the single ones.

Tolerances: FP64 as every other field check of this path (1e-12 of the largest
value); FP32 1e-5 (24-bit transforms of at most 2^11 x 2^3 points: a few dozen
roundings of 6e-8)."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

# (nx, ny, nz): shortest and longest y transforms, remainders on both sides of
# a power of two, one column (nx = 1), and the neighbours that keep the passes
# (ny = 4, nz = 3)
SIZES = [(1, 8, 1), (2, 9, 2), (5, 5, 1), (33, 7, 2), (17, 64, 1), (16, 65, 2), (31, 33, 1), (3, 513, 1), (4, 256, 2),
         (2, 1024, 1), (3, 300, 2), (40, 30, 1), (130, 20, 2), (6, 4, 2), (9, 9, 3)]


def _pair(oracle, n, precision):
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(7 * N + precision)
    m0, Ms = rng.standard_normal(3 * N), rng.uniform(4e5, 8e5, N)
    d = (2e-9, 3e-9, 4e-9)
    g = mmx.Sim(mmx.FDMesh(dx=d[0], dy=d[1], dz=d[2], nx=n[0], ny=n[1], nz=n[2]), precision=precision)
    o = oracle.OracleSim(*n, *d)
    mmx.set_Ms(g, Ms)
    mmx.init_m0(g, m0)
    mmx.add_exch(g, 1.3e-11)
    mmx.add_demag(g)
    o.set_Ms(Ms)
    o.init_m0(m0)
    o.add_exch(1.3e-11)
    o.add_demag(0, 0, 0)
    return g, o


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", SIZES)
def test_plane_field_vs_oracle(oracle, n, precision):
    print(f"[case] plane {n} fp{precision}", flush=True)
    g, o = _pair(oracle, n, precision)
    hg, ho = mmx.effective_field(g), o.effective_field()
    assert np.max(np.abs(hg - ho)) <= (1e-12 if precision == 64 else 1e-5) * np.max(np.abs(ho))


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nz", [1, 2])
def test_plane_wide_blocks_match_single(nz, precision):
    """Ten members of one geometry share launches with several kx columns per
    block; alone each column has a block of its own: the same bits."""
    print(f"[case] plane batch nz={nz} fp{precision}", flush=True)

    def make(q):
        s = mmx.Sim(mmx.FDMesh(dx=2e-9, dy=2e-9, dz=2e-9, nx=129, ny=21, nz=nz), integrator="Heun",
                    precision=precision)
        mmx.set_Ms(s, 5e5 + 1e4 * q)
        mmx.init_m0(s, np.random.default_rng(q).standard_normal(3 * 129 * 21 * nz))
        mmx.add_exch(s, 1.3e-11)
        mmx.add_demag(s)
        mmx.set_driver(s, integrator="Heun", step=1e-14)
        return s

    alone, members = [make(q) for q in range(10)], [make(q) for q in range(10)]
    for s in alone:
        mmx.run_step(s, n=3)
    mmx.Batch(members).advance(3)
    for a, b in zip(alone, members):
        assert np.array_equal(a.spin, b.spin)
