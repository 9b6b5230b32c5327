"""Tile passes (several real-time steps of a small lattice per launch) against
the oracle: sizes at the edges of tiles, closed, periodic and mixed axes, every
scaled form of the pair updates and of the merged pass, step counts around a
pass's own.

Tolerances: FP64 1e-12 over at most 13 steps, as everywhere.  FP32: some 40
roundings of at most 6e-8 per cell and step, independent of each other, stay
below 6e-8 sqrt(40 * 13) = 1.4e-6 of the state; the bound is three times that.
"""
import numpy as np
import pytest

from tsmi import workloads as W
from tsmi.lattice import Lattice2D

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 5e-6}


def case(nx, ny, px, py, beta=0.05, ratio=1.0, g=5.0, g_lhy=0.0, steps=13, v_scale=1.0):
    """A lattice whose horizontal pair angle is beta (vertical: beta ratio^2) and
    whose state does not vanish at the edges."""
    dt = 1e-3
    dx = np.sqrt(dt / (4.0 * beta))
    lat = Lattice2D(nx, nx * dx, ny, ny * dx / ratio, px, py)
    X, Y = lat.mesh()
    lx, ly = lat.length_x, lat.length_y
    psi = (1.0 + 0.5 * np.cos(2 * np.pi * X / lx) * np.sin(2 * np.pi * Y / ly + 0.3)) * np.exp(
        1j * (0.7 * np.sin(2 * np.pi * X / lx) + 0.4 * np.cos(4 * np.pi * Y / ly)))
    psi = W.normalise(lat, psi)
    v = v_scale * (3.0 * np.cos(2 * np.pi * X / lx + 0.2) + 4.0 * np.sin(2 * np.pi * Y / ly) + 5.0)
    return W.Workload("tile", lat, psi, v, dt, steps, g=g * lx * ly, g_lhy=g_lhy * (lx * ly) ** 1.5)


def run(wl, oracle, precision, calls):
    from tsmi.hip import kernel_for
    k = kernel_for(wl, precision=precision, e_planes=oracle.exp_potential(wl.v, wl.dt, False))
    try:
        for n in calls:
            k.evolve(n)
        return k.sample()
    finally:
        k.close()


def check(wl, oracle, precision, calls=None):
    calls = calls or [wl.steps]
    ref = wl.psi
    for n in calls:
        ref = oracle.evolve(wl, n, ref)
    psi = run(wl, oracle, precision, calls)
    err = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
    assert err < TOL[precision], err


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nx,ny,px,py", [
    (2, 2, False, False), (5, 3, False, False), (127, 31, False, False), (128, 32, False, False),
    (129, 33, False, False), (255, 50, False, False), (300, 131, False, False),
    (8, 8, True, True), (10, 14, True, True), (120, 24, True, True), (136, 90, True, True), (45, 38, True, True),
    (38, 45, True, False), (90, 61, False, True)])
def test_tile_sizes(nx, ny, px, py, precision, oracle):
    check(case(nx, ny, px, py, g_lhy=0.7 if nx % 3 == 0 else 0.0), oracle, precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("beta,ratio", [(0.6, 1.0), (1.0, 1.0), (1.6, 1.0), (2.9, 1.0), (0.3, 2.0), (1.0, 0.5)])
def test_tile_forms(beta, ratio, per, precision, oracle):
    check(case(140, 76, per, per, beta=beta, ratio=ratio), oracle, precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("v_scale", [30.0, 300.0, 40000.0])
def test_tile_angles(v_scale, per, precision, oracle):
    """Potential angles up to 0.36, 3.6 and 480 per step."""
    check(case(64, 64, per, per, v_scale=v_scale), oracle, precision)


@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("calls", [[1], [2], [3], [4], [1, 2, 5], [7, 0, 6], [9, 3]])
def test_tile_calls(calls, per, oracle):
    check(case(150, 70, per, per), oracle, 64, calls)
