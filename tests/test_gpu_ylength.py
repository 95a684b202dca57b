"""y transforms of 3 and 5 times a power of two: field and tensor against the
oracle at both ends of each length's range, on meshes of three layers and more
(thinner ones take the one-kernel convolution).

Tolerances: FP64 1e-12 of the largest value as every field check of this path;
FP32 1e-5 (24-bit transforms, a few dozen roundings of 6e-8)."""
import numpy as np
import pytest

import mmx

pytestmark = pytest.mark.gpu

# ny: shortest and longest with 5/8, 3/4 and all of the power of two above
# 2 ny - 1, from the shortest cut length (80 of 128) to the longest (768 of 1024)
SIZES = [(6, 33, 3), (5, 40, 4), (4, 41, 3), (7, 48, 5), (3, 49, 3), (4, 56, 3), (5, 57, 3), (33, 65, 9), (9, 72, 33),
         (16, 80, 3), (17, 96, 4), (4, 100, 3), (3, 160, 3), (2, 161, 4), (3, 200, 3), (2, 300, 3), (2, 380, 3),
         (2, 448, 3)]


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("n", SIZES)
def test_field_vs_oracle(oracle, n, precision):
    print(f"[case] y length {n} fp{precision}", flush=True)
    N = n[0] * n[1] * n[2]
    rng = np.random.default_rng(3 * N + precision)
    m0, Ms = rng.standard_normal(3 * N), rng.uniform(4e5, 8e5, N)
    d = (2e-9, 3e-9, 4e-9)
    g = mmx.Sim(mmx.FDMesh(dx=d[0], dy=d[1], dz=d[2], nx=n[0], ny=n[1], nz=n[2]), precision=precision)
    o = oracle.OracleSim(*n, *d)
    mmx.set_Ms(g, Ms)
    mmx.init_m0(g, m0)
    mmx.add_demag(g, Nx=1, Ny=1)
    o.set_Ms(Ms)
    o.init_m0(m0)
    o.add_demag(1, 1, 0)
    hg, ho = mmx.effective_field(g), o.effective_field()
    assert np.max(np.abs(hg - ho)) <= (1e-12 if precision == 64 else 1e-5) * np.max(np.abs(ho))
