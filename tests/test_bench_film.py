"""bench.py's byte model of films of one or two layers, whose y and z transforms
are one kernel in place."""
import os
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
sys.path.insert(0, ROOT)
import bench  # noqa: E402


def test_byte_model_plane():
    # 1000x1000x1 FP32: Px, Py, Pz = 2048, 2048, 1; 1024 columns
    nx, ny, nz, w = 1000, 1000, 1, 4
    b, total = bench.byte_model(nx, ny, nz, 2048, 2048, 1, w, 2, chained=True, plane=True)
    N, S1 = nx * ny * nz, 1024 * ny * nz
    assert b["P2"] == b["P4"] == 0
    assert b["P3"] == 2 * 3 * 2 * w * S1 + 6 * w * 1025 * 1025 * 1
    assert b["P5"] == 2 * 3 * 2 * w * S1 + 7 * w * N + N
    assert total == b["P3"] + b["P5"]


def test_plane_form_follows_the_launches():
    five = {"P1": (0.1, 1), "P2": (0.1, 8), "P3": (0.1, 8), "P4": (0.1, 8), "P5": (0.1, 8), "LOCAL": (None, 0)}
    assert not bench.plane_form(five)
    assert bench.plane_form(dict(five, P2=(None, 0), P4=(None, 0)))
    assert not bench.plane_form({k: (None, 0) for k in five})
