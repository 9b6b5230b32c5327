"""Batches on register tiles against the oracle: closed, even and odd periodic and
mixed lattices together (several steps per pass and one), step counts around a
pass's own, E tables that leave and regain the phase form between calls, and
batches past the size limit.  FP64 1e-12, FP32 2e-5, as everywhere."""
import numpy as np
import pytest

from tsmi import workloads as W

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 2e-5}
SIZES = [(64, 64, True, True), (120, 24, False, False), (121, 33, False, False), (45, 38, True, True),
         (38, 45, True, True), (30, 61, True, False), (61, 30, False, True), (8, 8, True, True), (250, 140, True, True),
         (37, 1, False, False)]


def make(sizes, g_lhy=0.0):
    return [W.small_case(nx, ny, px, py, g=2.0, g_lhy=g_lhy, seed=W.SEED_BASE + 300 + i)
            for i, (nx, ny, px, py) in enumerate(sizes)]


def ref(oracle, wl, calls):
    psi = wl.psi
    for n in calls:
        psi = oracle.evolve(wl, steps=n, psi=psi)
    return psi


def check(oracle, b, wls, calls, precision):
    for i, wl in enumerate(wls):
        r = ref(oracle, wl, calls)
        err = float(np.linalg.norm(b.state(i) - r) / np.linalg.norm(r))
        assert err < TOL[precision], (i, err)


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("sizes", [SIZES, SIZES[:1], SIZES[1:3], SIZES[3:5]], ids=["all", "even", "closed", "odd"])
@pytest.mark.parametrize("calls", [[1], [2], [3], [13], [4, 1, 6]])
def test_calls(oracle, calls, sizes, precision):
    from tsmi.batch import HipBatch
    wls = make(sizes, g_lhy=0.3 if len(sizes) == 2 else 0.0)
    with HipBatch(wls, precision, e_planes=[oracle.exp_potential(w.v, w.dt, False) for w in wls]) as b:
        for n in calls:
            b.evolve(n)
        check(oracle, b, wls, calls, precision)


def test_e_form_changes(oracle):
    """A table without the phase form moves every lattice to the streaming passes,
    and back, between calls (an odd number of passes leaves the groups' states in
    different buffers)."""
    from tsmi.batch import HipBatch
    wls = make(SIZES[:8])
    es = [oracle.exp_potential(w.v, w.dt, False) for w in wls]
    with HipBatch(wls, 64, e_planes=es) as b:
        b.evolve(5)
        b.set_exp_potential(2, 0.5 * es[2][0], 0.5 * es[2][1])
        b.set_exp_potential(2, *es[2])
        b.evolve(2)
        b.set_exp_potential(0, 2.0 * es[0][0], 2.0 * es[0][1])
        assert np.isfinite(b.state(1)).all()
        b.set_exp_potential(0, *es[0])
        b.tune(2)
        b.evolve(4)
        check(oracle, b, wls, [5, 2, 4], 64)


def test_streaming_after_tiles(oracle):
    from tsmi.batch import HipBatch
    wls = make(SIZES[:8])
    es = [oracle.exp_potential(w.v, w.dt, False) for w in wls]
    with HipBatch(wls, 64, e_planes=es) as b:
        b.evolve(7)
        # half the norm per step on lattice 7: 0.5 E is no phase, so all stream
        b.set_exp_potential(7, 0.5 * es[7][0], 0.5 * es[7][1])
        b.evolve(3)
        check(oracle, b, wls[:7], [7, 3], 64)
