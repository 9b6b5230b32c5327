"""Device-side import and export of states and of E tables: every cell of narrow,
flat and ordinary lattices arrives where it belongs, and the cost follows the cell
count, not the width of the lattice."""
import statistics
import time

import numpy as np
import pytest

from tsmi.lattice import Lattice2D

pytestmark = pytest.mark.gpu


def fields(lat, seed):
    import torch
    g = torch.Generator(device="cpu").manual_seed(seed)
    return [torch.rand((lat.H, lat.W), generator=g, dtype=torch.float64).to("cuda") for _ in range(3)]


# around one workgroup's 256 cells, one stride of the grid (2048 x 256 cells), and
# rows shorter and longer than either
@pytest.mark.parametrize("precision", [64, 32])
@pytest.mark.parametrize("nx,ny,per", [(1, 1, False), (2, 128, False), (3, 85, False), (257, 1, False), (2, 300000, False),
                                       (5, 262147, False), (524287, 3, False), (524289, 2, False), (640, 823, True)])
def test_round_trip(nx, ny, per, precision):
    import torch
    from tsmi.hip import HipKernel
    lat = Lattice2D(nx, 1.0 * nx, ny, 1.0 * ny, per, per)
    re, im, _ = fields(lat, nx + ny)
    a, b = torch.empty_like(re), torch.empty_like(im)
    with HipKernel(lat, delta_t=1e-3, precision=precision) as k:
        k.set_stream(torch.cuda.current_stream().cuda_stream)
        k.set_state_device(re.data_ptr(), im.data_ptr())
        k.get_state_device(a.data_ptr(), b.data_ptr())
        torch.cuda.synchronize()
    keep = (lambda t: t.float().double()) if precision == 32 else (lambda t: t)
    assert torch.equal(a, keep(re)) and torch.equal(b, keep(im))


def test_narrow_lattices_cost_their_cells():
    """2 x 500000 against 1000 x 1000: the same cells.  A row of two cells still
    takes a cache line of the pitched plane, 8 times an ordinary cell's bytes in
    FP64; a mapping by whole rows cost 27 times."""
    import torch
    from tsmi.hip import HipKernel
    us = {}
    for nx, ny in ((1000, 1000), (2, 500000)):
        lat = Lattice2D(nx, 1.0 * nx, ny, 1.0 * ny, False, False)
        re, im, v = fields(lat, 1)
        e_re, e_im = torch.cos(v), torch.sin(v)
        with HipKernel(lat, delta_t=1e-3, precision=64) as k:
            k.set_stream(torch.cuda.current_stream().cuda_stream)
            for name, call in (("state", lambda: k.set_state_device(re.data_ptr(), im.data_ptr())),
                               ("export", lambda: k.get_state_device(re.data_ptr(), im.data_ptr())),
                               ("table", lambda: k.set_potential_exp_device(v.data_ptr()))):
                t = []
                for _ in range(7):
                    torch.cuda.synchronize()
                    t0 = time.perf_counter()
                    for _ in range(20):
                        call()
                    torch.cuda.synchronize()
                    t.append((time.perf_counter() - t0) / 20 * 1e6)
                us[nx, name] = statistics.median(t)
            k.set_exp_potential_device(e_re.data_ptr(), e_im.data_ptr())
    print(us)
    for name in ("state", "export", "table"):
        assert us[2, name] < 12 * us[1000, name], us
