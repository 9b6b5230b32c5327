"""Imaginary-time tile passes against the oracle: sizes at the edges of tiles,
every boundary, with and without a norm target, calls of a few steps, single
steps, and a renormalisation left pending across a change of the E form (which
changes the path).  FP64 1e-12, FP32 2e-5, as everywhere."""
import numpy as np
import pytest

from tsmi import workloads as W
from tsmi.hip import kernel_for

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 2e-5}


def close(psi, ref, precision=64):
    err = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
    assert err < TOL[precision], err


def make(nx, ny, px, py, steps, g_lhy=0.0):
    return W.small_case(nx, ny, px, py, steps=steps, g=3.0, g_lhy=g_lhy, imag_time=True)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nx,ny,px,py", [
    (2, 2, False, False), (119, 7, False, False), (120, 8, False, False), (121, 25, False, False),
    (250, 91, False, False), (8, 8, True, True), (112, 16, True, True), (300, 130, True, True), (45, 38, True, True),
    (38, 45, True, False), (90, 61, False, True)])
def test_sizes(oracle, nx, ny, px, py, precision):
    wl = make(nx, ny, px, py, 9, g_lhy=0.4 if nx % 2 else 0.0)
    k = kernel_for(wl, precision=precision, e_planes=oracle.exp_potential(wl.v, wl.dt, True))
    try:
        k.evolve(9)
        close(k.sample(), oracle.evolve(wl), precision)
    finally:
        k.close()


@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("calls", [[1], [2], [3], [4, 1, 2], [5, 0, 6]])
def test_calls(oracle, calls, per):
    wl = make(70, 44, per, per, sum(calls))
    k = kernel_for(wl, e_planes=oracle.exp_potential(wl.v, wl.dt, True))
    ref = wl.psi
    try:
        for n in calls:
            k.evolve(n)
            ref = oracle.evolve(wl, n, ref) if n else ref
            assert abs(k.squared_norm() - oracle.make_desc(wl).norm_target) < 1e-12
        close(k.sample(), ref)
    finally:
        k.close()


@pytest.mark.parametrize("per", [False, True])
def test_pending_across_paths(oracle, per):
    """tile steps, streamed steps (an E table with a zero has no one-plane form),
    tile steps again: each path takes over the other's pending renormalisation."""
    wl = make(70, 44, per, per, 12)
    e = oracle.exp_potential(wl.v, wl.dt, True)
    z = e[0].copy()
    z[0, 0] = 0.0
    a, b = (kernel_for(wl, e_planes=e, sweeps=s) for s in (0, 1))
    try:
        for k in (a, b):
            k.evolve(4)
            k.set_exp_potential(z, None)
            k.evolve(3)
            k.set_exp_potential(e[0], None)
            k.step(exchange=True)
            k.evolve(4)
        close(a.sample(), b.sample())
    finally:
        a.close()
        b.close()
