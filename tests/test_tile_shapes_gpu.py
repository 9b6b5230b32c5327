"""Every compiled tile shape against the oracle, at sizes where the planner takes it
(asserted through tsmi_tile_geometry): closed and even doubly periodic lattices,
several steps per launch, with and without LHY; mixed axes and odd periodic extents;
single steps; imaginary time.  Two components and the reverse sweep at sizes past
which the planner (two_field_plan.hpp) leaves its small shape, and batches.

Tolerances as in the other tile tests: FP64 1e-12, FP32 5e-6 in real and 2e-5 in
imaginary time and for two components; reverse sweeps against the streamed one, FP32
5e-5 of the largest entry."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from test_tile_gpu import case
from tsmi import workloads as W

pytestmark = pytest.mark.gpu

KINDS = {"closed": (0, 0, 0), "periodic": (1, 1, 0), "mixed": (1, 0, 0), "odd": (1, 1, 0), "imag": (0, 0, 1),
         "imag_mixed": (0, 1, 1), "imag_periodic": (1, 1, 1)}
SHAPES = [   # bits, kind, nx, ny, steps, (rows per wave, waves, steps of the longest launch)
    (32, "closed", 40, 24, 3, (4, 8, 3)), (32, "closed", 632, 372, 8, (4, 16, 4)), (32, "closed", 632, 1500, 8, (12, 8, 4)),
    (32, "closed", 262, 1400, 1, (4, 8, 1)), (32, "closed", 1000, 1400, 1, (4, 16, 1)), (32, "closed", 1600, 1300, 1, (12, 4, 1)),
    (32, "periodic", 40, 24, 4, (4, 8, 2)), (32, "periodic", 2000, 110, 9, (4, 16, 4)),
    (32, "periodic", 668, 1800, 4, (12, 4, 2)), (32, "periodic", 632, 1500, 9, (12, 8, 4)),
    (32, "mixed", 262, 1400, 3, (4, 8, 1)), (32, "mixed", 1000, 1400, 3, (4, 16, 1)), (32, "mixed", 1600, 1300, 3, (12, 4, 1)),
    (32, "odd", 263, 1401, 3, (4, 8, 1)), (32, "odd", 1201, 1101, 3, (4, 16, 1)), (32, "odd", 1601, 1301, 3, (12, 4, 1)),
    (32, "imag", 40, 1500, 3, (4, 8, 1)), (32, "imag", 373, 1600, 3, (4, 16, 1)), (32, "imag_periodic", 372, 1600, 4, (4, 16, 1)),
    (32, "imag_mixed", 372, 1600, 3, (4, 16, 1)), (32, "imag_mixed", 1100, 1400, 3, (12, 4, 1)),
    (64, "closed", 40, 24, 3, (4, 8, 3)), (64, "closed", 336, 517, 3, (6, 4, 2)), (64, "closed", 114, 1100, 5, (6, 8, 3)),
    (64, "closed", 336, 1600, 3, (8, 8, 3)), (64, "closed", 669, 1600, 1, (8, 4, 1)), (64, "closed", 262, 1400, 1, (4, 8, 1)),
    (64, "closed", 484, 1800, 1, (6, 8, 1)), (64, "closed", 1000, 1400, 1, (8, 8, 1)),
    (64, "periodic", 40, 24, 4, (6, 4, 2)), (64, "periodic", 40, 24, 9, (4, 8, 3)), (64, "periodic", 114, 1100, 6, (6, 8, 4)),
    (64, "periodic", 1400, 604, 4, (8, 4, 2)), (64, "periodic", 410, 1300, 6, (8, 8, 4)),
    (64, "mixed", 262, 1400, 3, (4, 8, 1)), (64, "mixed", 114, 1100, 3, (6, 4, 1)), (64, "mixed", 594, 1400, 3, (6, 8, 1)),
    (64, "mixed", 1600, 662, 3, (8, 4, 1)), (64, "odd", 701, 1501, 3, (8, 4, 1)), (64, "odd", 1201, 1101, 3, (8, 8, 1)),
    (64, "imag", 151, 1600, 3, (4, 8, 1)), (64, "imag", 151, 1100, 3, (6, 4, 1)), (64, "imag", 373, 1600, 3, (6, 8, 1)),
    (64, "imag", 632, 1800, 3, (8, 4, 1)), (64, "imag_periodic", 1100, 1000, 4, (8, 4, 1)),
    (64, "imag_mixed", 372, 1600, 3, (6, 8, 1)), (64, "imag_mixed", 1100, 1000, 3, (8, 4, 1)),
]


def rel(a, r):
    return float(np.linalg.norm(a - r) / np.linalg.norm(r))


@pytest.mark.parametrize("g_lhy", [0.0, 0.7])
@pytest.mark.parametrize("bits,kind,nx,ny,steps,shape", SHAPES)
def test_single_lattice(bits, kind, nx, ny, steps, shape, g_lhy, oracle):
    from tsmi import _lib
    from tsmi.batch import desc_of
    from tsmi.hip import kernel_for
    px, py, imag = KINDS[kind]
    if imag:
        wl = W.small_case(nx, ny, bool(px), bool(py), steps=steps, g=3.0, g_lhy=g_lhy, imag_time=True)
    else:
        wl = case(nx, ny, bool(px), bool(py), steps=steps, g_lhy=g_lhy)
    out = (C.c_int32 * 4)()
    d = desc_of(wl, bits)
    assert _lib.load().tsmi_tile_geometry(C.byref(d), steps, out) == 0
    assert tuple(out)[:3] == shape
    k = kernel_for(wl, precision=bits, e_planes=oracle.exp_potential(wl.v, wl.dt, bool(imag)))
    try:
        k.evolve(steps)
        psi = k.sample()
    finally:
        k.close()
    assert rel(psi, oracle.evolve(wl)) < {64: 1e-12, 32: 2e-5 if imag else 5e-6}[bits]


@pytest.mark.parametrize("bits,nx,ny,per,imag,mass_b,steps", [
    (32, 570, 690, False, False, 1.0, 6), (32, 570, 690, False, False, 3.0, 6),      # 8 rows x 8 waves
    (32, 1216, 1216, False, True, 1.0, 3), (32, 1201, 1217, True, True, 1.0, 3),
    (32, 570, 690, True, False, 1.0, 8), (32, 1216, 1216, True, True, 1.0, 4),       # 4 x 16
    (32, 570, 690, True, False, 3.0, 8),                                             # 8 x 8 periodic
    (64, 128, 1216, False, True, 1.4, 3), (64, 128, 1216, True, True, 1.4, 4),       # 4 x 8
    (64, 570, 690, False, False, 1.0, 4), (64, 570, 690, True, False, 1.0, 6)])
def test_two_components(bits, nx, ny, per, imag, mass_b, steps, oracle):
    from tsmi.pair import HipPair
    pw = W.pair_case(n_x=nx, n_y=ny, periodic_x=per, periodic_y=per, imag_time=imag, omega_r=1.3, omega_i=-0.4, mass_b=mass_b,
                     g_a=3.0, g_b=2.0, g_ab=1.5, calls=[steps])
    if mass_b == 3.0:   # one scaled form per component
        pw = dataclasses.replace(pw, dt=4.0 * 1.2 * min(pw.lattice.delta_x, pw.lattice.delta_y) ** 2)
    with HipPair(pw, precision=bits, e_planes=oracle.pair_exp_potentials(pw)) as h:
        h.evolve(steps)
        got = h.state(0), h.state(1)
    for a, r in zip(got, oracle.evolve2(pw)):
        assert rel(a, r) < {64: 1e-12, 32: 2e-5}[bits]


@pytest.mark.parametrize("nx,ny,per,g", [(230, 1000, False, 0.0), (740, 300, True, 0.0),      # 4 rows x 16 waves
                                         (570, 690, False, 20.0), (570, 690, True, 20.0)])    # 8 x 8
def test_reverse_sweep(nx, ny, per, g):
    from tsmi.hip import kernel_for
    from tsmi.losses import infidelity
    wl = W.small_case(nx, ny, per, per, steps=13, dt=2e-3, length=12.0, g=g, g_lhy=0.3 * g)
    lat = wl.lattice
    target = W.normalise(lat, W.gaussian_packet(lat, 0.4, -0.3, 0.0, 0.0, width=1.5))
    out = []
    for sweeps in (0, 1):
        k = kernel_for(wl, precision=32, sweeps=sweeps)
        try:
            k.evolve_checkpointed(wl.steps, 13)
            out.append(k.adjoint(infidelity(lat, target, k.sample())[1]))
        finally:
            k.close()
    for a, r in zip(*out):
        assert np.abs(a - r).max() <= 5e-5 * np.abs(r).max()


@pytest.mark.parametrize("bits,sizes", [
    (32, [(300 + 2 * i, 290 - 4 * i) for i in range(14)]), (32, [(180 + i, 130 + 3 * i) for i in range(30)]),
    (64, [(300 + 2 * i, 290 - 4 * i) for i in range(8)]), (64, [(400, 440), (380, 300), (260, 620)]),
    (64, [(60 + i, 90 - i) for i in range(20)])])
def test_batches(bits, sizes, oracle):
    from tsmi.batch import HipBatch
    wls = [W.small_case(nx, ny, *[(False, False), (True, True), (True, False)][i % 3], g=2.0, seed=W.SEED_BASE + 500 + i)
           for i, (nx, ny) in enumerate(sizes)]
    with HipBatch(wls, bits, e_planes=[oracle.exp_potential(w.v, w.dt, False) for w in wls]) as b:
        b.evolve(9)
        for i, wl in enumerate(wls):
            assert rel(b.state(i), oracle.evolve(wl, steps=9)) < {64: 1e-12, 32: 2e-5}[bits], i
