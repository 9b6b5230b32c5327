"""Imaginary time with a rotation that cancels a component, fully or nearly: the
component's next norm is then far below the terms it is formed of, and must come out
as the sum of its cells does.  Two components of one shape, the first tanh(r x) of the
second, x the hyperbolic angle of a whole rotation: with r = 1 it vanishes at the
rotation after the first step (against the oracle), with r = 1/2 and no half rotation
before it at the half rotation that ends a call of one step (against the streamed
passes).  FP64, 1e-12 of the two states' norm, as everywhere.

The half rotation that starts a call may not cancel it: the step after it divides the
component to the norm it had before, which scales its rounding errors up to that norm
on every path, the oracle's too."""
import dataclasses

import numpy as np
import pytest

from tsmi import workloads as W

pytestmark = pytest.mark.gpu

COUPLINGS = pytest.mark.parametrize("omega,dt", [(1.3, 1e-3), (10.0, 1e-2), (100.0, 1e-2)])
OFF = pytest.mark.parametrize("off", [0.0, 1e-9, 1e-5])


def make(omega, dt, r, off, calls):
    pw = W.pair_case(n_x=60, n_y=44, periodic_x=False, periodic_y=False, imag_time=True, omega_r=omega, calls=calls,
                     g_a=0.0, g_b=0.0, g_ab=0.0)
    return dataclasses.replace(pw, dt=dt, psi_a=np.tanh(r * 0.5 * omega * dt) * (1.0 + off) * pw.psi_b, v_a=pw.v_b)


def run(oracle, pw, sweeps, initial_half):
    from tsmi.pair import HipPair
    with HipPair(pw, precision=64, e_planes=oracle.pair_exp_potentials(pw), sweeps=sweeps) as h:
        for n in pw.calls:
            h.evolve(n, initial_half=initial_half)
        return h.state(0), h.state(1)


def check(got, ref):
    norm = np.sqrt(sum(np.linalg.norm(z) ** 2 for z in ref))
    for a, z in zip(got, ref):
        assert np.linalg.norm(a - z) < 1e-12 * norm


@pytest.mark.parametrize("calls", [[6], [2, 4]])
@OFF
@COUPLINGS
def test_cancelled_between_steps(oracle, omega, dt, off, calls):
    pw = make(omega, dt, 1.0, off, calls)
    check(run(oracle, pw, 0, True), oracle.evolve2(pw))


@pytest.mark.parametrize("calls", [[1], [1, 5], [1, 1, 3]])
@OFF
@COUPLINGS
def test_cancelled_at_the_end_of_a_call(oracle, omega, dt, off, calls):
    pw = make(omega, dt, 0.5, off, calls)
    check(run(oracle, pw, 0, False), run(oracle, pw, 1, False))
