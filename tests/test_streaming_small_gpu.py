"""The streaming passes, which large lattices and batches run, at the sizes that take
register tiles by themselves: small lattices with one or two steps per pass asked for
(mixed axes, LHY, imaginary time), and batches whose descriptors ask for it, the
autotuner among them.  FP64 1e-12 and FP32 2e-5 against the oracle, as everywhere."""
import ctypes as C

import numpy as np
import pytest

from test_hip_parity import CASES, case_id, rel_l2, run_hip
from tsmi import workloads as W

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", CASES, ids=[case_id(c) for c in CASES])
def test_one_step_per_pass(case, oracle):
    wl = W.small_case(**case)
    psi, e, x, _ = run_hip(wl, oracle, sweeps=1)
    ref = oracle.evolve(wl)
    assert rel_l2(psi, ref) < 1e-12
    np.testing.assert_allclose(e, oracle.energy(wl, ref), rtol=1e-12, atol=1e-14)
    np.testing.assert_allclose(x, oracle.expected_values(wl, ref), rtol=1e-11, atol=1e-13)


@pytest.mark.parametrize("case", CASES, ids=[case_id(c) for c in CASES])
def test_one_step_per_pass_fp32(case, oracle):
    wl = W.small_case(**case)
    psi, *_ = run_hip(wl, oracle, precision=32, sweeps=1)
    assert rel_l2(psi, oracle.evolve(wl)) < 2e-5


BATCH = [(64, 64, False, False), (96, 80, True, True), (33, 17, False, False), (300, 40, True, False),
         (40, 130, False, True), (8, 8, True, True), (37, 1, False, False), (520, 70, False, False), (45, 38, True, True)]


@pytest.fixture
def batch_with_sweeps(monkeypatch):
    """HipBatch over descriptors that ask for so many steps per pass."""
    import tsmi.batch as B

    def make(wls, precision, e_planes, sweeps):
        plain = B.desc_of

        def desc(wl, *args):
            d = plain(wl, *args)
            lat = wl.lattice
            d.sweeps = sweeps if sweeps != 2 or lat.periodic_x == lat.periodic_y else 1
            return d
        monkeypatch.setattr(B, "desc_of", desc)
        return B.HipBatch(wls, precision, e_planes=e_planes)
    return make


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("sweeps", [1, 2])
@pytest.mark.parametrize("calls", [[9], [4, 1, 6]])
def test_batch(calls, sweeps, precision, oracle, batch_with_sweeps):
    wls = [W.small_case(nx, ny, px, py, g=2.0, seed=W.SEED_BASE + 700 + i) for i, (nx, ny, px, py) in enumerate(BATCH)]
    es = [oracle.exp_potential(w.v, w.dt, False) for w in wls]
    with batch_with_sweeps(wls, precision, es, sweeps) as b:
        # two where asked for and exact: closed, or both axes periodic and even
        assert all(b.info(i)["steps_per_pass"] == (2 if sweeps == 2 and px == py and (not px or (nx | ny) % 2 == 0) else 1)
                   for i, (nx, ny, px, py) in enumerate(BATCH))
        for n in calls:
            b.evolve(n)
        for i, wl in enumerate(wls):
            ref = wl.psi
            for n in calls:
                ref = oracle.evolve(wl, steps=n, psi=ref)
            assert rel_l2(b.state(i), ref) < {64: 1e-12, 32: 2e-5}[precision], i


def test_autotuner_moves_lattices_and_keeps_states(oracle):
    """Past the tile limit of a batch (1.57M cells in FP64) with the steps per pass left
    open: the autotuner times one and two steps per pass and several segment heights,
    and every state goes on where it was."""
    from tsmi.batch import HipBatch
    sizes = [(640, 600, False, False), (601, 640, True, True), (500, 640, True, False), (520, 500, True, True),
             (400, 640, False, True), (37, 1, False, False)]
    wls = [W.small_case(nx, ny, px, py, g=2.0, seed=W.SEED_BASE + 720 + i) for i, (nx, ny, px, py) in enumerate(sizes)]
    assert sum(w.lattice.W * w.lattice.H for w in wls) > 3 << 19
    es = [oracle.exp_potential(w.v, w.dt, False) for w in wls]
    with HipBatch(wls, 64, e_planes=es) as b:
        b.evolve(3)
        before = [b.info(i) for i in range(len(wls))]
        assert b.tune(steps=2) > 0
        after = [b.info(i) for i in range(len(wls))]
        b.evolve(4)
        for i, wl in enumerate(wls):
            ref = oracle.evolve(wl, steps=4, psi=oracle.evolve(wl, steps=3))
            assert rel_l2(b.state(i), ref) < 1e-12, i
    assert all(r["steps_per_pass"] in (1, 2) and r["rows_per_segment"] % 2 == 0 for r in after[:-1])
    # it did search: with 64-row segments a batch this size leaves most of the chip idle
    assert any(a != r for a, r in zip(before, after))
