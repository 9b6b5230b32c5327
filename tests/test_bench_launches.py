"""bench.py names the kernel that an evolve call runs, and does not take two steps per
launch for granted."""
import importlib.util
import os

import pytest

from tsmi.lattice import Lattice2D

ROOT = os.path.join(os.path.dirname(os.path.abspath(__file__)), "..")


@pytest.fixture(scope="module")
def bench():
    spec = importlib.util.spec_from_file_location("bench", os.path.join(ROOT, "bench.py"))
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


@pytest.mark.parametrize("n,steps,tile_rows,tiles", [(1024, 100, 0, True), (8192, 100, 0, False), (1024, 100, 16, False),
                                                     (2100, 100, 0, True), (2100, 1, 0, False)])
def test_tile_launch(bench, n, steps, tile_rows, tiles):
    lat = Lattice2D(n, 64.0, periodic_x=True, periodic_y=True)
    assert bench.tile_launch(lat, dict(dt=5e-4, mass=1.0, g=50.0), 32, steps, tile_rows) is tiles


def test_dominant_kernel(bench):
    def kt(fused, single):
        return dict(fused_ms=0.5 * fused, fused_launches=fused, single_ms=0.25 * single, single_launches=single)
    assert bench.dominant_kernel(kt(499, 2), 1000, False) == ("step2_kernel", 499, 0.5, 2)
    assert bench.dominant_kernel(kt(0, 9), 9, False) == ("step_kernel", 9, 0.25, 1)
    assert bench.dominant_kernel(kt(250, 0), 1000, True) == ("tile_kernel", 250, 0.5, 4)
    assert bench.dominant_kernel(kt(333, 2), 1000, True)[3] == pytest.approx(998 / 333)
    assert bench.dominant_kernel(kt(0, 1), 1, True) == ("tile_kernel", 1, 0.25, 1)
