"""Two-component tile passes against the two-component oracle: sizes at the edges
of tiles, every boundary, every scaled form of the pair updates (and one form per
component), step counts around a pass's own, and a renormalisation left pending
by a single step.  Tolerances as everywhere: FP64 1e-12, FP32 2e-5."""
import dataclasses

import numpy as np
import pytest

from tsmi import workloads as W

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 2e-5}
COUPLED = dict(g_a=3.0, g_b=2.0, g_ab=1.5)


def check(oracle, pw, precision):
    from tsmi.pair import HipPair
    with HipPair(pw, precision=precision, e_planes=oracle.pair_exp_potentials(pw)) as h:
        for n in pw.calls:
            h.evolve(n)
        got = h.state(0), h.state(1)
    for a, r in zip(got, oracle.evolve2(pw)):
        err = float(np.linalg.norm(a - r) / np.linalg.norm(r))
        assert err < TOL[precision], err


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("imag", [False, True])
@pytest.mark.parametrize("nx,ny,px,py", [
    (2, 2, False, False), (119, 7, False, False), (120, 24, False, False), (121, 25, False, False),
    (250, 61, False, False), (8, 8, True, True), (112, 16, True, True), (114, 58, True, True), (300, 130, True, True),
    (45, 38, True, True), (38, 45, True, False), (90, 61, False, True)])
def test_sizes(oracle, nx, ny, px, py, imag, precision):
    check(oracle, W.pair_case(n_x=nx, n_y=ny, periodic_x=px, periodic_y=py, imag_time=imag, omega_r=1.3,
                              omega_i=-0.4 if nx % 2 else 0.0, mass_b=1.4, calls=[9], **COUPLED), precision)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("beta,mass_b", [(0.3, 1.0), (1.2, 1.0), (1.2, 3.0)])
def test_forms(oracle, beta, mass_b, per, precision):
    pw = W.pair_case(n_x=140, n_y=40, periodic_x=per, periodic_y=per, omega_r=1.0, mass_b=mass_b, calls=[7], **COUPLED)
    dt = 4.0 * beta * min(pw.lattice.delta_x, pw.lattice.delta_y) ** 2
    check(oracle, dataclasses.replace(pw, dt=dt), precision)


@pytest.mark.parametrize("imag", [False, True])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("omega", [0.0, 1.1])
@pytest.mark.parametrize("calls", [[1], [2], [3], [1, 4, 2], [5, 0, 6]])
def test_calls(oracle, calls, omega, per, imag):
    check(oracle, W.pair_case(n_x=60, n_y=44, periodic_x=per, periodic_y=per, imag_time=imag, omega_r=omega,
                              calls=calls, **COUPLED), 64)


@pytest.mark.parametrize("omega", [0.0, 1.1])
def test_after_single_step(oracle, omega):
    """evolve after tsmi_pair_step has left a renormalisation pending: the same
    as two evolve calls whose first ends with one step's own."""
    from tsmi import _lib
    from tsmi.pair import HipPair
    pw = W.pair_case(n_x=50, n_y=40, periodic_x=False, periodic_y=False, imag_time=True, omega_r=omega, calls=[1, 5],
                     **COUPLED)
    with HipPair(pw, precision=64, e_planes=oracle.pair_exp_potentials(pw)) as h:
        L = h._L
        _lib.check(L.tsmi_pair_rabi(h._h, 0.5, 0))
        _lib.check(L.tsmi_pair_step(h._h, 0, 0.0))
        _lib.check(L.tsmi_pair_rabi(h._h, 0.5, 1))
        h.evolve(5)
        got = h.state(0), h.state(1)
    for a, r in zip(got, oracle.evolve2(pw)):
        assert float(np.linalg.norm(a - r) / np.linalg.norm(r)) < 1e-12
