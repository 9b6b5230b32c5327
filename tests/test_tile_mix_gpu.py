"""Sizes between the limits of single steps and of several steps per launch, where a
call mixes streamed steps and register tiles: the first and the last step of an even
doubly periodic call, single steps between calls, checkpoints one step apart.  Against
the oracle, FP64 1e-12 and FP32 5e-6 as in the other tile tests."""
import ctypes as C

import numpy as np
import pytest

from test_tile_gpu import case

pytestmark = pytest.mark.gpu


def make(bits, per, oracle):
    from tsmi import _lib
    from tsmi.batch import desc_of
    from tsmi.hip import kernel_for
    nx, ny = (1500, 1400) if bits == 64 else (2100, 2120)
    wl = case(nx, ny, per, per, steps=9)
    out = (C.c_int32 * 4)()
    d, L = desc_of(wl, bits), _lib.load()
    assert L.tsmi_tile_geometry(C.byref(d), 1, out) == 0 and out[0] == 0
    assert L.tsmi_tile_geometry(C.byref(d), 9, out) == 0 and out[2] > 1
    return wl, kernel_for(wl, precision=bits, e_planes=oracle.exp_potential(wl.v, wl.dt, False))


def check(psi, ref, bits):
    assert float(np.linalg.norm(psi - ref) / np.linalg.norm(ref)) < {64: 1e-12, 32: 5e-6}[bits]


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("calls", [[9], [3, 1, 2, 4], [2, 5]])
def test_calls(calls, per, bits, oracle):
    wl, k = make(bits, per, oracle)
    ref = wl.psi
    try:
        for n in calls:
            k.evolve(n)
            ref = oracle.evolve(wl, n, ref)
        check(k.sample(), ref, bits)
    finally:
        k.close()


@pytest.mark.parametrize("bits", [64, 32])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("every", [1, 4, 50])
def test_checkpoints(every, per, bits, oracle):
    wl, k = make(bits, per, oracle)
    try:
        k.evolve_checkpointed(9, every)
        check(k.sample(), oracle.evolve(wl), bits)
    finally:
        k.close()
