"""Doubly periodic lattices whose potential on the halo is not a copy of the inner
cells' (a caller may tabulate it as it likes; the reference applies the table of
every tile cell): imaginary time and two components against the oracle, the reverse
sweep against the streamed one.  Tolerances as everywhere: FP64 1e-12, FP32 2e-5; the
sweeps FP64 1e-11, FP32 5e-5 of the largest entry."""
import dataclasses

import numpy as np
import pytest

from tsmi import workloads as W

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 2e-5}


def other_halo(lat, v, seed):
    """v with a halo of its own, the inner cells as they are."""
    out = v + np.random.RandomState(seed).uniform(-30.0, 30.0, v.shape)
    out[lat.inner_y, lat.inner_x] = v[lat.inner_y, lat.inner_x]
    return out


def close(a, r, precision):
    err = float(np.linalg.norm(a - r) / np.linalg.norm(r))
    assert err < TOL[precision], err


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("calls", [[9], [3, 1, 5]])
@pytest.mark.parametrize("nx,ny", [(8, 8), (70, 44), (300, 130), (45, 38)])
def test_imaginary_time(oracle, nx, ny, calls, precision):
    from tsmi.hip import kernel_for
    wl = W.small_case(nx, ny, True, True, steps=sum(calls), g=3.0, imag_time=True)
    wl = dataclasses.replace(wl, v=other_halo(wl.lattice, wl.v, nx))
    ref = wl.psi
    k = kernel_for(wl, precision=precision, e_planes=oracle.exp_potential(wl.v, wl.dt, True))
    try:
        for n in calls:
            k.evolve(n)
            ref = oracle.evolve(wl, n, ref)
        close(k.sample(), ref, precision)
    finally:
        k.close()


@pytest.mark.parametrize("imag,precision", [(False, 64), (True, 64), (True, 32)])
@pytest.mark.parametrize("nx,ny", [(8, 8), (112, 16), (70, 44)])
def test_two_components(oracle, nx, ny, imag, precision):
    from tsmi.pair import HipPair
    pw = W.pair_case(n_x=nx, n_y=ny, periodic_x=True, periodic_y=True, imag_time=imag, omega_r=1.3, omega_i=-0.4, g_a=3.0,
                     g_b=2.0, g_ab=1.5, calls=[7, 2])
    pw = dataclasses.replace(pw, v_a=other_halo(pw.lattice, pw.v_a, 1), v_b=other_halo(pw.lattice, pw.v_b, 2))
    with HipPair(pw, precision=precision, e_planes=oracle.pair_exp_potentials(pw)) as h:
        for n in pw.calls:
            h.evolve(n)
        got = h.state(0), h.state(1)
    for a, r in zip(got, oracle.evolve2(pw)):
        close(a, r, precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("g", [0.0, 20.0])
def test_reverse_sweep(g, precision):
    from tsmi.hip import kernel_for
    from tsmi.losses import infidelity
    wl = W.small_case(70, 44, True, True, steps=11, dt=2e-3, length=12.0, g=g)
    wl = dataclasses.replace(wl, v=other_halo(wl.lattice, wl.v, 3))
    lat = wl.lattice
    target = W.normalise(lat, W.gaussian_packet(lat, 0.4, -0.3, 0.0, 0.0, width=1.5))
    out = []
    for sweeps in (0, 1):
        k = kernel_for(wl, precision=precision, sweeps=sweeps)
        try:
            k.evolve_checkpointed(wl.steps, 4)
            out.append(k.adjoint(infidelity(lat, target, k.sample())[1]))
        finally:
            k.close()
    tol = {64: 1e-11, 32: 5e-5}[precision]
    for a, r in zip(*out):
        assert np.abs(a - r).max() <= tol * np.abs(r).max()


def test_wrapped_tables_keep_their_route():
    """A potential evaluated at wrapped coordinates repeats itself up to rounding: the
    sweep over it runs as tiles, in launches of several steps."""
    import time

    from tsmi.hip import kernel_for
    us = {}
    for wrapped in (True, False):
        wl = W.small_case(300, 300, True, True, steps=60, dt=2e-3, length=12.0)
        if not wrapped:
            wl = dataclasses.replace(wl, v=other_halo(wl.lattice, wl.v, 4))
        k = kernel_for(wl, precision=32)
        try:
            k.evolve_checkpointed(wl.steps, 60)
            g = np.ones_like(wl.psi)
            t = []
            for _ in range(5):
                k.synchronize()
                t0 = time.perf_counter()
                k.adjoint(g)
                t.append(time.perf_counter() - t0)
            us[wrapped] = min(t)
        finally:
            k.close()
    assert us[True] < 0.8 * us[False], us
