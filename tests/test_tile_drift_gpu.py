"""Norm drift of the register tiles over long runs.  With V = 0 and g = 0 every cell
takes the same factor at the potential stage, so a rounding of its modulus repeats at
every cell and step and drifts the norm.  Tiles merge the neighbouring half passes of
two steps, whose modulus is rounded anew (delta, relative); what a pass's middle steps
leave its last step takes back, and what that leaves the passes after it.

FP64, 64^2 periodic, 6000 steps, against the streamed one-step passes: without the
correction the norm would differ by 2 x 4000 delta, at least 1.9e-13 at the angles
taken (computed here); each step's own roundings are independent from cell to cell
and leave far less than the bar, 1e-13.  A batch's passes come in 8 sets, whose last
rounding repeats every 8 passes: at most 2 x 250 x 1.1e-16 = 5.5e-14 besides.

FP32, as the streamed passes' own drift tests: 1e-7 over 1000 and 400 steps."""
import math

import numpy as np
import pytest

from tsmi import workloads as W
from tsmi.lattice import Lattice2D

pytestmark = pytest.mark.gpu

STEPS = 6000
ANGLES = [0.043, 0.199, 0.238, 0.277, 0.303, 0.316, 0.9, 1.2, 1.3]


def delta(beta):
    """Relative rounding error of the merged pass's modulus in FP64."""
    def axis(a, b):
        m, t = (1.0, b / a) if abs(a) >= abs(b) else (a / b, 1.0)
        return complex(m, t), abs(complex(a, b) / complex(m, t))
    v, g = axis(math.cos(beta), math.sin(beta))
    v2, _ = axis(math.cos(2 * beta), math.sin(2 * beta))
    mid = np.longdouble(math.pow(g * g, 4)) * abs(np.clongdouble(v) ** 2 / np.clongdouble(v2))
    return float(np.longdouble(float(mid)) / mid - 1)


def workload(beta):
    n, side = 64, 8.0
    lat = Lattice2D(n, side, periodic_x=True, periodic_y=True)
    X, Y = lat.mesh()
    psi = W.normalise(lat, np.exp(-(X * X + Y * Y) / 4.0) * np.exp(1j * 0.7 * X))
    return W.Workload("drift", lat, psi, np.zeros_like(X), beta * 4 * (side / n) ** 2, STEPS)


def streamed_norm(wl):
    from tsmi.hip import kernel_for
    k = kernel_for(wl, precision=64, sweeps=1)
    try:
        k.evolve(STEPS)
        return k.squared_norm()
    finally:
        k.close()


@pytest.mark.parametrize("beta", ANGLES)
def test_fp64(beta):
    from tsmi.hip import kernel_for
    assert 2 * 4000 * abs(delta(beta)) > 1.5e-13
    wl = workload(beta)
    k = kernel_for(wl, precision=64)
    try:
        k.evolve(STEPS)
        assert abs(k.squared_norm() - streamed_norm(wl)) < 1e-13
    finally:
        k.close()


@pytest.mark.parametrize("beta", ANGLES)
def test_fp64_batch(beta):
    from tsmi.batch import HipBatch
    wl = workload(beta)
    with HipBatch([wl, wl], 64) as b:
        b.evolve(1)         # the other buffer first
        b.set_state(0, wl.psi)
        b.evolve(STEPS)
        norm = W.squared_norm(wl.lattice, b.state(0))
    assert abs(norm - streamed_norm(wl)) < 1e-13


@pytest.mark.parametrize("form,beta", [("B", 2.048), ("A", 0.512)])
def test_fp32(form, beta):
    from tsmi.hip import kernel_for
    n, side = 512, 8.0
    lat = Lattice2D(n, side, periodic_x=True, periodic_y=True)
    X, Y = lat.mesh()
    psi = W.normalise(lat, np.exp(-(X * X + Y * Y) / 4.0) * np.exp(1j * 0.7 * X))
    wl = W.Workload("drift", lat, psi, np.zeros_like(X), beta * 4 * (side / n) ** 2, 1000)
    k = kernel_for(wl, precision=32)
    try:
        n0 = k.squared_norm()
        k.evolve(wl.steps)
        drift = k.squared_norm() / n0 - 1
    finally:
        k.close()
    assert abs(drift) < 1e-7, drift


def test_fp32_two_components():
    from tsmi.pair import HipPair
    lat = Lattice2D(512, 8.0, periodic_x=True, periodic_y=True)
    X, Y = lat.mesh()
    v_a, v_b = 0.5 * 0.64 * (X * X + Y * Y), 0.5 * 0.768 * (X * X + Y * Y)
    amp = np.sqrt(np.maximum(10.0 - v_a, 0.0) / 50.0)
    psi_a = (amp * np.exp(1j * 2.4 * X)).astype(np.complex128)
    psi_b = (0.5 * amp * np.exp(-1j * 1.6 * Y)).astype(np.complex128)
    pw = W.PairWorkload("drift", lat, psi_a, psi_b, v_a, v_b, 5e-4, (400,), g_a=50.0, g_b=50.0, g_ab=40.0, omega_r=1.0)
    n0 = W.squared_norm(lat, psi_a) + W.squared_norm(lat, psi_b)
    with HipPair(pw, precision=32) as h:
        h.evolve(400)
        drift = h.energy()[11] / n0 - 1
    assert abs(drift) < 1e-7, drift
