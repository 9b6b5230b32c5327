"""Host states through the pinned chunks: planes and complex arrays, windows,
sizes around one and two chunks, both precisions.  Whatever goes in comes out:
FP64 bit for bit, FP32 rounded once."""
import ctypes as C

import numpy as np
import pytest

from tsmi.lattice import Lattice2D

pytestmark = pytest.mark.gpu


# a chunk holds 4 MiB: 262144 complex values, split from 16384 on
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nx,ny,per", [(2, 1, False), (128, 128, False), (128, 129, False), (513, 511, False),
                                       (1031, 517, True), (262145, 3, False)])
def test_state_round_trip(nx, ny, per, precision):
    from tsmi import _lib
    from tsmi.hip import HipKernel
    lat = Lattice2D(nx, 1.0 * nx, ny, 1.0 * ny, per, per)
    rng = np.random.default_rng(nx + ny)
    psi = rng.standard_normal((lat.H, lat.W)) + 1j * rng.standard_normal((lat.H, lat.W))
    ref = psi if precision == 64 else psi.astype(np.complex64).astype(np.complex128)
    with HipKernel(lat, delta_t=1e-3, precision=precision) as k:
        k.set_state(psi)
        assert np.array_equal(k.sample(), ref)
        x, y = lat.W // 3, lat.H // 2
        assert np.array_equal(k.sample(x, y, lat.W - x, lat.H - y), ref[y:, x:])
        re, im = np.ascontiguousarray(psi.imag), np.ascontiguousarray(psi.real)
        _lib.check(k._L.tsmi_set_state(k._h, _lib.dptr(re), _lib.dptr(im)))
        assert np.array_equal(k.sample(), ref.imag + 1j * ref.real)
        out = np.full((2, lat.H, lat.W + 3), 7.0)     # a row stride of the caller's
        p = [o.ctypes.data_as(C.POINTER(C.c_double)) for o in out]
        _lib.check(k._L.tsmi_get_sample(k._h, lat.W + 3, 0, 0, lat.W, lat.H, *p))
        assert np.array_equal(out[0, :, :lat.W], ref.imag) and np.array_equal(out[1, :, :lat.W], ref.real)
        assert np.all(out[:, :, lat.W:] == 7.0)
