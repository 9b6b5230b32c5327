"""The reverse sweep on register tiles against the streamed one (sweeps = 1 asks
for one step per pass): sizes at the edges of tiles, closed and even periodic
axes, linear and nonlinear, every scaled form, checkpoints around a pass's
length.  Both run the same arithmetic up to rounding: FP64 1e-11, FP32 5e-5 of
the largest entry (some 40 roundings per cell and step, forward and back)."""
import numpy as np
import pytest

from tsmi import workloads as W
from tsmi.losses import infidelity

pytestmark = pytest.mark.gpu

TOL = {64: 1e-11, 32: 5e-5}


def sweep(wl, target, precision, every, sweeps):
    from tsmi.hip import kernel_for
    k = kernel_for(wl, precision=precision, sweeps=sweeps)
    try:
        k.evolve_checkpointed(wl.steps, every)
        _, g = infidelity(wl.lattice, target, k.sample())
        return k.adjoint(g)
    finally:
        k.close()


def check(wl, precision, every):
    lat = wl.lattice
    target = W.normalise(lat, W.gaussian_packet(lat, 0.4, -0.3, 0.0, 0.0, width=1.5))
    got, ref = sweep(wl, target, precision, every, 0), sweep(wl, target, precision, every, 1)
    for a, r in zip(got, ref):
        assert np.abs(a - r).max() <= TOL[precision] * np.abs(r).max()


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("g,g_lhy", [(0.0, 0.0), (20.0, 3.0)])
@pytest.mark.parametrize("nx,ny,per", [(3, 2, False), (119, 23, False), (120, 24, False), (121, 57, False),
                                       (257, 90, False), (8, 8, True), (112, 16, True), (130, 60, True),
                                       (33, 40, True)])
def test_sizes(nx, ny, per, g, g_lhy, precision):
    check(W.small_case(nx, ny, per, per, steps=11, dt=2e-3, length=12.0, g=g, g_lhy=g_lhy), precision, 4)


@pytest.mark.parametrize("every", [1, 2, 3, 5, 12, 50])
def test_checkpoints(every):
    check(W.small_case(70, 66, False, False, steps=12, dt=2e-3, length=12.0), 64, every)


@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("beta", [0.3, 1.2])
def test_forms(beta, per):
    n, length = 80, 12.0
    check(W.small_case(n, n, per, per, steps=9, dt=4.0 * beta * (length / n) ** 2, length=length), 64, 4)
