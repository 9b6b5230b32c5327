"""Which calls run as register tiles, and in which shape (tsmi_tile_geometry, no
GPU): never beyond the sizes where tiles measured faster, never on lattices whose
shape leaves most of a tile idle, and several steps per launch where the planes'
traffic is what a single one waits for."""
import ctypes as C

import pytest


def tile(nx, ny, steps, bits=32, px=0, py=0, imag=0, sweeps=0, tile_rows=0):
    from tsmi import _lib
    L = _lib.load()
    d = _lib.Desc(nx, ny, px, py, 4, 4, imag, bits, tile_rows, sweeps, 1e-3, 1.0, 1.0, 0.0, 0.1, 0.1, 0.1 * nx, 0.1 * ny,
                  0.0)
    out = (C.c_int32 * 4)()
    assert L.tsmi_tile_geometry(C.byref(d), steps, out) == 0, L.tsmi_last_error()
    return tuple(out)


STREAMED = (0, 0, 0, 0)


@pytest.mark.parametrize("bits", [32, 64])
@pytest.mark.parametrize("nx,ny", [(2, 1000000), (8, 400000), (16, 200000), (1000000, 2), (400000, 3)])
def test_narrow_and_flat_lattices_stream(nx, ny, bits):
    assert tile(nx, ny, 20, bits) == STREAMED and tile(nx, ny, 20, bits, imag=1) == STREAMED


@pytest.mark.parametrize("bits,side", [(32, 1800), (32, 2100), (32, 2160), (64, 1200), (64, 1500), (64, 1600)])
def test_large_lattices_take_several_steps_per_launch(bits, side):
    assert tile(side, side, 40, bits)[2] > 1


@pytest.mark.parametrize("bits,inside,outside", [(32, 2000, 2100), (64, 1400, 1450)])
def test_single_steps_give_out_earlier(bits, inside, outside):
    for px, py, steps in ((0, 0, 1), (1, 1, 1), (1, 1, 2), (1, 0, 9), (0, 1, 9)):
        assert tile(inside - 8 * px, inside - 8 * py, steps, bits, px, py)[2] == 1
        assert tile(outside, outside, steps, bits, px, py) == STREAMED
    assert tile(inside - 9, inside - 8, 9, bits, 1, 1)[2] == 1      # odd periodic
    assert tile(outside + 1, outside, 9, bits, 1, 1) == STREAMED
    assert tile(outside, outside, 9, bits)[2] > 1 and tile(outside, outside, 9, bits, 1, 1)[2] > 1


def test_what_asks_for_streaming_streams():
    assert tile(256, 256, 9, sweeps=1) == tile(256, 256, 9, sweeps=2) == tile(256, 256, 9, tile_rows=16) == STREAMED
    assert tile(256, 1, 9) == tile(256, 256, 0) == STREAMED
    assert tile(2200, 2200, 9) == tile(1300, 1300, 9, imag=1) == tile(1100, 1100, 9, 64, imag=1) == STREAMED


def test_rejects_bad_arguments():
    from tsmi import _lib
    L = _lib.load()
    assert L.tsmi_tile_geometry(None, 3, (C.c_int32 * 4)()) == 1


@pytest.mark.gpu
@pytest.mark.parametrize("nx,ny,px,bits,steps,sweeps", [
    (8, 100000, 0, 32, 20, 2), (2, 100000, 0, 64, 20, 2), (300000, 2, 0, 32, 20, 2), (2100, 2100, 0, 32, 20, 2),
    (1800, 1800, 0, 32, 20, 2), (2101, 2101, 1, 32, 20, 2), (1601, 1601, 1, 64, 20, 2), (2100, 2100, 0, 32, 1, 1),
    (1200, 1200, 0, 64, 1, 1)])
def test_the_chosen_route_is_not_the_slower(nx, ny, px, bits, steps, sweeps):
    """Against the passes that `sweeps` asks for; the margin is for the clock."""
    import time

    import torch
    from tsmi.hip import HipKernel
    from tsmi.lattice import Lattice2D
    lat = Lattice2D(nx, 0.05 * nx, ny, 0.05 * ny, bool(px), bool(px))
    one = torch.ones((lat.H, lat.W), dtype=torch.float64, device="cuda")
    v = 0.1 * one
    e_re, e_im = torch.cos(1e-4 * v), torch.sin(-1e-4 * v)
    ks = [HipKernel(lat, delta_t=1e-4, precision=bits, sweeps=s) for s in (0, sweeps)]
    us = [[], []]
    try:
        for k in ks:
            k.set_stream(torch.cuda.current_stream().cuda_stream)
            k.set_exp_potential_device(e_re.data_ptr(), e_im.data_ptr())
            k.set_state_device(one.data_ptr(), v.data_ptr())
            k.evolve(steps)
        for _ in range(9):
            for k, t in zip(ks, us):
                torch.cuda.synchronize()
                t0 = time.perf_counter()
                for _ in range(max(1, 20 // steps)):
                    k.evolve(steps)
                torch.cuda.synchronize()
                t.append(time.perf_counter() - t0)
    finally:
        for k in ks:
            k.close()
    assert sorted(us[0])[4] < 1.15 * sorted(us[1])[4], us
