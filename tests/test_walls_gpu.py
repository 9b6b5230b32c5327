"""Walls whose phase per step leaves the range of the short reductions: a potential
of up to 1e300 on some cells, tabulated on the device, against the oracle's table
(libm's sine and cosine of the same product).  Tile and streaming passes, FP64 1e-12
and FP32 2e-5 as everywhere."""
import dataclasses

import numpy as np
import pytest

from tsmi import workloads as W

pytestmark = pytest.mark.gpu

TOL = {64: 1e-12, 32: 2e-5}


@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("sweeps", [0, 1, 2])
@pytest.mark.parametrize("per", [False, True])
@pytest.mark.parametrize("height", [2e18, 1e23, -1e33, 1e300])
def test_high_walls(oracle, height, per, sweeps, precision):
    import torch
    from tsmi.hip import HipKernel
    wl = W.small_case(140, 44, per, per, steps=7, g=3.0)
    lat = wl.lattice
    X, Y = lat.mesh()
    wall = (np.abs(X - 0.2 * lat.length_x) < 0.1 * lat.length_x) & (np.abs(Y) < 0.2 * lat.length_y)
    wl = dataclasses.replace(wl, v=np.where(wall, height * (1.0 + 0.01 * np.sin(2 * np.pi * Y / lat.length_y)), wl.v))
    v = torch.from_numpy(np.ascontiguousarray(wl.v)).to("cuda")
    with HipKernel(lat, delta_t=wl.dt, coupling=wl.g, precision=precision, sweeps=sweeps) as k:
        k.set_stream(torch.cuda.current_stream().cuda_stream)
        k.set_potential_exp_device(v.data_ptr())
        k.set_state(wl.psi)
        k.evolve(wl.steps)
        psi = k.sample()
    ref = oracle.evolve(wl)
    assert wall.any() and np.isfinite(ref).all()
    err = float(np.linalg.norm(psi - ref) / np.linalg.norm(ref))
    assert err < TOL[precision], err
