"""The calls a user of this framework makes, as cases that can be timed and
checked: listed() names them, draw() gives more of the same ranges, prepare()
builds what a program holds before the call (lattice, potential, kernel object,
initial state on the GPU), run() is one call through the public entry points
and exact() is the same call in plain torch, 64 bits.

Every pass starts from the initial state of the case (set_state), so it can be
repeated; a 32-bit kernel's results are kept in 32 bits.
"""
from __future__ import annotations

import math
import os
import sys

import numpy as np
import torch
from torch.utils.checkpoint import checkpoint

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "trotter-suzuki-mpi_amd"))

HALO = 4

# What a case says beside its sizes (nx, ny) and boundaries (px, py):
#   kind   evolve    one component, real time, from a state to a state
#          ground    one component, imaginary time, in chunks with the energy read after each
#          pair      two components with Rabi coupling, real or imaginary time
#          batch     many lattices advanced together
#          gradient  evolution and the gradient of its infidelity in V and psi_0
#          timedep   a potential that changes every step
#   bits   32 or 64, the kernel's precision
#   steps  steps of the whole pass
#   system the physical set-up: packet (box of side 20, sum of Gaussians), trap (harmonic),
#          vortices (box of side 64, weak trap, g = 50)


def listed():
    return [
        # the smallest call: a few steps of a small periodic lattice, as an interactive
        # session or a test makes it; launches and latency are all of it
        dict(name="small_64_periodic_fp64", kind="evolve", system="packet", nx=64, ny=64, px=True, py=True, bits=64,
             g=5.0, lhy=0.0, steps=50),
        # the plain method: a wave packet in a harmonic trap in double precision
        dict(name="packet_256_fp64", kind="evolve", system="trap", nx=256, ny=256, px=False, py=False, bits=64,
             g=0.0, lhy=0.0, steps=400),
        # an odd-sized GPE run in single precision with the Lee-Huang-Yang term
        dict(name="trap_1023x769_lhy_fp32", kind="evolve", system="trap", nx=1023, ny=769, px=False, py=False,
             bits=32, g=20.0, lhy=4.0, steps=300),
        # the headline run: vortex dynamics on a large periodic lattice, FP32
        dict(name="vortices_8192_fp32", kind="evolve", system="vortices", nx=8192, ny=8192, px=True, py=True, bits=32,
             g=50.0, lhy=0.0, steps=40),
        # the same in double precision
        dict(name="vortices_8192_fp64", kind="evolve", system="vortices", nx=8192, ny=8192, px=True, py=True, bits=64,
             g=50.0, lhy=0.0, steps=20),
        # ground-state search in imaginary time, the energy watched between chunks
        dict(name="ground_2048_fp32", kind="ground", system="trap", nx=2048, ny=2048, px=False, py=False, bits=32,
             g=100.0, lhy=0.0, steps=300, chunks=3),
        # the same on a small ragged lattice in double precision
        dict(name="ground_700x501_fp64", kind="ground", system="trap", nx=700, ny=501, px=False, py=False, bits=64,
             g=30.0, lhy=0.0, steps=200, chunks=4),
        # two coupled components in real time, FP32
        dict(name="pair_1024_fp32", kind="pair", system="vortices", nx=1024, ny=1024, px=True, py=True, bits=32,
             imag=False, steps=1000),
        # the mixed ground state of two coupled components, FP64
        dict(name="pair_250_imag_fp64", kind="pair", system="trap", nx=250, ny=250, px=False, py=False, bits=64,
             imag=True, steps=1000),
        # a parameter sweep: many small lattices of mixed sizes and boundaries, FP32
        dict(name="batch_32_fp32", kind="batch", system="packet", count=32, side_min=64, side_max=256, bits=32,
             g=0.0, steps=1000),
        # differentiation: the gradient of an infidelity in the potential, forward and backward
        dict(name="gradient_1024_fp32", kind="gradient", system="packet", nx=1024, ny=1024, px=False, py=False,
             bits=32, g=0.0, lhy=0.0, steps=400, every=100),
        # a driven potential, re-tabulated on the device before every step
        dict(name="driven_512_fp64", kind="timedep", system="packet", nx=512, ny=512, px=False, py=False, bits=64,
             g=2.0, lhy=0.0, steps=100),
    ]


def _log(rng, lo, hi):
    return lo * (hi / lo) ** rng.random()


def _sides(rng, lo, hi):
    """Two sides, log-uniform, within a factor of two of each other; odd, even and
    round numbers among them."""
    a = _log(rng, lo, hi)
    b = min(hi, max(lo, a * 2.0 ** rng.uniform(-1.0, 1.0)))
    out = []
    for v in (a, b):
        n = int(round(v))
        how = rng.random()
        if how < 0.3:
            n = max(32, n // 32 * 32)
        elif how < 0.4:
            n |= 1
        out.append(n)
    return out


def _boundaries(rng):
    how = rng.random()
    if how < 0.45:
        return False, False
    if how < 0.85:
        return True, True
    return (True, False) if how < 0.925 else (False, True)


def _steps(rng, sites, most):
    """Steps of a pass: few on large lattices, hundreds on small ones."""
    cap = max(4, min(most, int(1.2e9 / sites)))
    return max(3, int(round(_log(rng, max(3, cap / 8), cap))))


def draw(rng):
    how = rng.random()
    bits = rng.choice((32, 64))
    if how < 0.45:
        system = rng.choice(("packet", "trap", "vortices"))
        nx, ny = _sides(rng, 64, 1600 if system != "vortices" else 6000)
        px, py = _boundaries(rng)
        g = 50.0 if system == "vortices" else rng.choice((0.0, 0.0, 5.0, 20.0))
        return dict(kind="evolve", system=system, nx=nx, ny=ny, px=px, py=py, bits=bits, g=g,
                    lhy=rng.choice((0.0, 0.0, 0.0, 2.0)) if g else 0.0, steps=_steps(rng, nx * ny, 500))
    if how < 0.62:
        nx, ny = _sides(rng, 100, 2200)
        chunks = rng.choice((1, 2, 4))
        px, py = _boundaries(rng)
        return dict(kind="ground", system="trap", nx=nx, ny=ny, px=px, py=py, bits=bits,
                    g=rng.choice((0.0, 10.0, 100.0)), lhy=0.0, steps=chunks * max(3, _steps(rng, nx * ny, 400) // chunks),
                    chunks=chunks)
    if how < 0.76:
        imag = rng.random() < 0.4
        nx, ny = _sides(rng, 80, 1000)
        px, py = rng.choice(((False, False), (True, True)))
        return dict(kind="pair", system="trap" if imag else rng.choice(("trap", "vortices")), nx=nx, ny=ny, px=px,
                    py=py, bits=bits, imag=imag, steps=_steps(rng, 2 * nx * ny, 600))
    if how < 0.84:
        lo = rng.choice((64, 100))
        return dict(kind="batch", system="packet", count=rng.randint(4, 32), side_min=lo, side_max=rng.randint(128, 320),
                    bits=bits, g=rng.choice((0.0, 5.0)), steps=rng.randint(50, 400))
    if how < 0.93:
        nx, ny = _sides(rng, 100, 1100)
        per = rng.random() < 0.3
        steps = max(8, _steps(rng, 4 * nx * ny, 300))
        return dict(kind="gradient", system="packet", nx=nx, ny=ny, px=per, py=per, bits=bits,
                    g=rng.choice((0.0, 0.0, 5.0)), lhy=0.0, steps=steps, every=rng.randint(5, 100))
    nx, ny = _sides(rng, 100, 1100)
    px, py = rng.choice(((False, False), (True, True)))
    return dict(kind="timedep", system="packet", nx=nx, ny=ny, px=px, py=py, bits=bits, g=rng.choice((0.0, 2.0)),
                lhy=0.0, steps=rng.randint(10, 100))


# ---------------------------------------------------------------------------
# inputs, from the seed alone
# ---------------------------------------------------------------------------
class _Box:
    """Lengths, spacing and the tile (halo of 4 on periodic axes) of a case."""

    def __init__(self, nx, ny, px, py, length):
        self.nx, self.ny, self.px, self.py = nx, ny, px, py
        self.lx, self.ly = float(length), float(length) * ny / nx
        self.dx, self.dy = self.lx / nx, self.ly / ny
        self.W, self.H = nx + 2 * HALO * px, ny + 2 * HALO * py
        self.ix = slice(HALO * px, HALO * px + nx)
        self.iy = slice(HALO * py, HALO * py + ny)

    def mesh(self, device):
        def axis(n, d, length, per):
            i = torch.arange(-HALO * per, n + HALO * per, dtype=torch.float64, device=device)
            x = (i + 0.5) * d - 0.5 * length
            x = torch.where(x < -0.5 * length, x + length, x)
            return torch.where(x > 0.5 * length, x - length, x)
        return (axis(self.nx, self.dx, self.lx, self.px)[None, :], axis(self.ny, self.dy, self.ly, self.py)[:, None])

    def norm2(self, psi):
        p = psi[self.iy, self.ix]
        return (p.real ** 2 + p.imag ** 2).sum() * (self.dx * self.dy)

    def normalised(self, psi, norm=1.0):
        return psi * torch.sqrt(norm / self.norm2(psi))

    def lattice(self):
        from tsmi.lattice import Lattice2D
        return Lattice2D(self.nx, self.lx, self.ny, self.ly, self.px, self.py)


LENGTH = {"packet": 20.0, "trap": 24.0, "vortices": 64.0}
DT = {"packet": 1e-3, "trap": 1e-3, "vortices": 5e-4}


def _box(case):
    return _Box(case["nx"], case["ny"], bool(case["px"]), bool(case["py"]), LENGTH[case["system"]])


def _dt(case):
    imag = case["kind"] == "ground" or case.get("imag", False)
    return 1e-4 if imag else DT[case["system"]]


def _uniform(seed, n):
    return np.random.RandomState(seed % (2 ** 31)).uniform(0.0, 1.0, n)


def _gaussians(X, Y, u, box, count):
    v = torch.zeros((box.H, box.W), dtype=torch.float64, device=X.device)
    for k in range(count):
        a, b, w, d = u[4 * k], u[4 * k + 1], 0.5 + 1.5 * u[4 * k + 2], -5.0 + 10.0 * u[4 * k + 3]
        v += d * torch.exp(-((X - (a - 0.5) * box.lx) ** 2 + (Y - (b - 0.5) * box.ly) ** 2) / (2.0 * w * w))
    return v


def _packet(X, Y, u, width=1.0):
    x0, y0, kx, ky = (4.0 * t - 2.0 for t in u[:4])
    r2 = (X - x0) ** 2 + (Y - y0) ** 2
    return torch.exp(-r2 / (2.0 * width * width)) * torch.exp(1j * (kx * X + ky * Y))


def _potential(case, box, seed, device):
    X, Y = box.mesh(device)
    if case["system"] == "packet":
        return _gaussians(X, Y, _uniform(seed + 101, 32), box, 8)
    if case["system"] == "trap":
        w = 0.8 + 0.4 * _uniform(seed + 102, 2)
        return 0.5 * (w[0] * w[0] * X * X + w[1] * w[1] * Y * Y)
    return 0.01 * (X * X + Y * Y)


def _state(case, box, seed, device):
    X, Y = box.mesh(device)
    if case["system"] == "vortices":
        u = _uniform(seed + 103, 48)
        mu = math.sqrt(2.0 * 0.01 * 50.0 / math.pi)
        r_tf = math.sqrt(mu / 0.01)
        psi = torch.sqrt(torch.clamp(mu - 0.01 * (X * X + Y * Y), min=0.0) / 50.0).to(torch.complex128)
        for j in range(16):
            rad, ang = 0.7 * r_tf * math.sqrt(u[3 * j]), 2.0 * math.pi * u[3 * j + 1]
            dx, dy = X - rad * math.cos(ang), Y - rad * math.sin(ang)
            s = 1.0 if u[3 * j + 2] < 0.5 else -1.0
            psi = psi * torch.tanh(torch.sqrt(dx * dx + dy * dy)) * torch.exp(1j * s * torch.atan2(dy, dx))
        return box.normalised(psi)
    if case["kind"] == "ground":
        r = np.random.RandomState((seed + 104) % (2 ** 31))
        noise = torch.from_numpy(r.uniform(-1.0, 1.0, (2, 64, 64))).to(device)
        reps = (1, (box.H + 63) // 64, (box.W + 63) // 64)
        noise = noise.repeat(reps)[:, :box.H, :box.W]
        psi = torch.exp(-(X * X + Y * Y) / 2.0) + 0.01 * torch.complex(noise[0], noise[1])
        return box.normalised(psi)
    return box.normalised(_packet(X, Y, _uniform(seed + 105, 4)))


def _exp_table(v, dt, imag):
    return torch.exp(-dt * v).to(torch.complex128) if imag else torch.exp(-1j * dt * v.to(torch.complex128))


def _batch_cases(case, seed):
    """The lattices of a batch: sides log-uniform, both axes periodic in half of them."""
    u = _uniform(1000 + 7 * case["count"] + case["side_max"], 2 * case["count"])   # shapes belong to the case
    out = []
    for i in range(case["count"]):
        n = int(round(case["side_min"] * (case["side_max"] / case["side_min"]) ** u[2 * i]))
        per = bool(u[2 * i + 1] < 0.5)
        out.append((dict(kind="evolve", system="packet", nx=n, ny=n, px=per, py=per, g=case["g"], lhy=0.0),
                    seed + 1000 * (i + 1)))
    return out


PAIR = dict(g_a=10.0, g_b=8.0, g_ab=4.0, omega_r=1.0, omega_i=0.3)


def _pair_inputs(case, seed, device):
    box = _box(case)
    v_a = _potential(case, box, seed, device)
    v_b = 0.8 * v_a
    X, Y = box.mesh(device)
    if case["system"] == "vortices":
        psi_a = _state(case, box, seed, device)
        psi_b = box.normalised(_state(case, box, seed + 50, device), 1.0 / 3.0)
    else:
        psi_a = box.normalised(_packet(X, Y, _uniform(seed + 106, 4), 1.5))
        psi_b = box.normalised(_packet(X, Y, _uniform(seed + 107, 4), 1.2), 1.0 / 3.0)
    return box, psi_a, psi_b, v_a, v_b


def _timedep_inputs(case, seed, device):
    box = _box(case)
    v0 = _potential(case, box, seed, device)
    X, Y = box.mesh(device)
    v1 = 0.5 * X * torch.ones_like(Y)
    return box, _state(case, box, seed, device), v0.contiguous(), v1.contiguous()


def _drive(v0, v1, t):
    return v0 + math.sin(40.0 * t) * v1


def _target(box, seed, device):
    X, Y = box.mesh(device)
    u = _uniform(seed + 108, 4)
    u[2:] = 0.5     # at rest
    return box.normalised(_packet(X, Y, u))


# ---------------------------------------------------------------------------
# what a user's program holds, and one call
# ---------------------------------------------------------------------------
def _planes(z):
    return z.real.contiguous(), z.imag.contiguous()


def prepare(case, seed):
    dev = torch.device("cuda")
    kind = case["kind"]
    if kind == "batch":
        from tsmi.batch import HipBatch
        from tsmi.workloads import Workload
        wls = []
        for c, s in _batch_cases(case, seed):
            box = _box(c)
            wls.append(Workload("sweep", box.lattice(), _state(c, box, s, dev).cpu().numpy(),
                                _potential(c, box, s, dev).cpu().numpy(), _dt(c), case["steps"], g=c["g"]))
        return dict(case=case, batch=HipBatch(wls, case["bits"]), psi=[w.psi for w in wls])
    if kind == "pair":
        from tsmi.pair import HipPair
        from tsmi.workloads import PairWorkload
        box, pa, pb, va, vb = (t.cpu().numpy() if isinstance(t, torch.Tensor) else t
                               for t in _pair_inputs(case, seed, dev))
        pw = PairWorkload("pair", box.lattice(), pa, pb, va, vb, _dt(case), (case["steps"],), imag_time=case["imag"],
                          **PAIR)
        # in imaginary time the norm targets move with the run: a pass starts from a new object
        return dict(case=case, pw=pw, pair=None if case["imag"] else HipPair(pw, case["bits"]))
    from tsmi.hip import HipKernel
    imag = kind == "ground"
    if kind == "timedep":
        box, psi, v, v1 = _timedep_inputs(case, seed, dev)
    else:
        box, psi, v1 = _box(case), None, None
        psi, v = _state(case, box, seed, dev), _potential(case, box, seed, dev).contiguous()
    kernel = HipKernel(box.lattice(), delta_t=_dt(case), coupling=case["g"], coupling_lhy=case["lhy"], imag_time=imag,
                       precision=case["bits"], norm_target=float(box.norm2(psi)) if imag else 0.0)
    kernel.set_stream(torch.cuda.current_stream().cuda_stream)
    e_re, e_im = _planes(_exp_table(v, _dt(case), imag))
    kernel.set_exp_potential_device(e_re.data_ptr(), None if imag else e_im.data_ptr())
    kernel.set_potential_device(v.data_ptr())
    re, im = _planes(psi)
    s = dict(case=case, kernel=kernel, re=re, im=im, v=v, v1=v1, box=box)
    if kind == "gradient":
        s["t_re"], s["t_im"] = _planes(_target(box, seed, dev))
        for k in ("re", "im", "v"):
            s[k].requires_grad_(True)
    torch.cuda.synchronize()
    return s


def _kept(case, x):
    return x.to(torch.float32) if case["bits"] == 32 else x


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "batch":
        b = state["batch"]
        for i, psi in enumerate(state["psi"]):
            b.set_state(i, psi)
        b.evolve(case["steps"])
        keep = np.complex64 if case["bits"] == 32 else np.complex128
        return [b.state(i).astype(keep) for i in range(case["count"])]
    if kind == "pair":
        pair, pw = state["pair"], state["pw"]
        if pair is None:
            from tsmi.pair import HipPair
            pair = HipPair(pw, case["bits"])
        else:
            pair.set_state(0, pw.psi_a)
            pair.set_state(1, pw.psi_b)
        pair.evolve(case["steps"])
        keep = np.complex64 if case["bits"] == 32 else np.complex128
        out = [pair.state(k).astype(keep) for k in (0, 1)]
        if state["pair"] is None:
            pair.close()
        return out
    kernel = state["kernel"]
    if kind == "gradient":
        from tsmi.autograd import evolve, infidelity
        box = state["box"]
        for k in ("re", "im", "v"):
            state[k].grad = None
        re, im = evolve(kernel, state["v"], state["re"], state["im"], case["steps"], case["every"])
        loss = infidelity(state["t_re"], state["t_im"], re, im, box.dx * box.dy, (box.iy, box.ix))
        loss.backward()
        return [_kept(case, t.detach()) for t in (loss, state["v"].grad, state["re"].grad, state["im"].grad)]
    kernel.set_state_device(state["re"].data_ptr(), state["im"].data_ptr())
    energies = []
    if kind == "timedep":
        from tsmi import timedep
        v0, v1 = state["v"], state["v1"]
        kernel.set_potential_exp_device(v0.data_ptr())
        timedep.evolve(kernel, lambda t: _drive(v0, v1, t), case["steps"])
    elif kind == "ground":
        for _ in range(case["chunks"]):
            kernel.evolve(case["steps"] // case["chunks"])
            energies.append(kernel.energy())
    else:
        kernel.evolve(case["steps"])
    re, im = torch.empty_like(state["re"]), torch.empty_like(state["im"])
    kernel.get_state_device(re.data_ptr(), im.data_ptr())
    out = [_kept(case, re), _kept(case, im)]
    if energies:
        out.append(np.asarray(energies, dtype=np.float32 if case["bits"] == 32 else np.float64))
    return out


def work(case):
    """Bytes: the inputs read once (state and potential in 64 bits) and the results
    written once; flops: 8 pair passes of 4 fused multiply-adds per pair of cells,
    and the potential pass (density, angle, sine and cosine, rotation), 70 per
    cell and step; a reverse step runs both states back and adds the gradient."""
    if case["kind"] == "batch":
        sites = sum((c["nx"] + 2 * HALO * c["px"]) ** 2 for c, _ in _batch_cases(case, 0))
    else:
        b = _box(case)
        sites = b.W * b.H
    comps = 2 if case["kind"] == "pair" else 1
    out = 8 if case["bits"] == 32 else 16
    per_step, extra = 70.0, 0.0
    if case["kind"] == "gradient":
        per_step, extra = 70.0 + 150.0, 1.5 * out
    if case["kind"] == "timedep":
        extra = 8.0
    return {"bytes": comps * sites * (16 + 8 + out + extra), "flops": comps * sites * per_step * case["steps"]}


# ---------------------------------------------------------------------------
# the same in plain torch, 64 bits
# ---------------------------------------------------------------------------
def _pairs(psi, axis, s, a, b):
    """The pair update [[a, b], [b, a]] on cells (x, y), (x+1, y) (axis 1) or (x, y),
    (x, y+1) (axis 0) with x + y + s even; cells without a partner stay."""
    H, W = psi.shape
    out = psi.clone()
    for p in (0, 1):
        o = (p + s) % 2
        n = ((W if axis else H) - o) // 2
        if n <= 0:
            continue
        lo, hi = slice(o, o + 2 * n, 2), slice(o + 1, o + 2 * n, 2)
        i, j = ((slice(p, None, 2), lo), (slice(p, None, 2), hi)) if axis else ((lo, slice(p, None, 2)), (hi, slice(p, None, 2)))
        out[i] = a * psi[i] + b * psi[j]
        out[j] = a * psi[j] + b * psi[i]
    return out


class _Step:
    """One second-order Trotter-Suzuki step of a tile."""

    def __init__(self, box, dt, imag, g, lhy, mass=1.0):
        self.box, self.imag = box, imag
        bx, by = dt / (4.0 * mass * box.dx ** 2), dt / (4.0 * mass * box.dy ** 2)
        self.h = (math.cosh(bx), math.sinh(bx)) if imag else (math.cos(bx), 1j * math.sin(bx))
        self.v = (math.cosh(by), math.sinh(by)) if imag else (math.cos(by), 1j * math.sin(by))
        self.g, self.lhy = g * dt, lhy * dt

    def __call__(self, psi, e, other=None, c_ab=0.0):
        for axis, s in ((0, 0), (1, 0), (0, 1), (1, 1)):
            psi = _pairs(psi, axis, s, *(self.h if axis else self.v))
        x = None
        if self.g or self.lhy:
            n = psi.real ** 2 + psi.imag ** 2
            x = self.g * n
            if self.lhy:
                x = x + self.lhy * n * torch.sqrt(n)
        if other is not None:
            m = c_ab * (other.real ** 2 + other.imag ** 2)
            x = m if x is None else x + m
        psi = psi * e
        if x is not None:
            psi = psi * (torch.exp(-x) if self.imag else torch.exp(-1j * x))
        for axis, s in ((1, 1), (0, 1), (1, 0), (0, 0)):
            psi = _pairs(psi, axis, s, *(self.h if axis else self.v))
        return psi

    def exchange(self, psi):
        b, h = self.box, HALO
        if not (b.px or b.py):
            return psi
        psi = psi.clone()
        if b.px:
            r0 = h if b.py else 0
            rows = slice(r0, r0 + b.H - 2 * h)
            psi[rows, :h], psi[rows, b.W - h:] = psi[rows, b.W - 2 * h:b.W - h].clone(), psi[rows, h:2 * h].clone()
        if b.py:
            psi[:h], psi[b.H - h:] = psi[b.H - 2 * h:b.H - h].clone(), psi[h:2 * h].clone()
        return psi


def _energy(box, psi, v, g):
    """total, kinetic, potential, interaction, LHY (0), squared norm, as the solver defines them."""
    y0, y1, x0, x1 = box.iy.start, box.iy.stop, box.ix.start, box.ix.stop
    my, mx = (0 if box.py else 2), (0 if box.px else 2)
    a0, a1, b0, b1 = y0 + my, y1 - my, x0 + mx, x1 - mx
    c = psi[a0:a1, b0:b1]

    def second(axis):
        def sh(k):
            return psi[a0:a1, b0 + k:b1 + k] if axis else psi[a0 + k:a1 + k, b0:b1]
        return -(sh(2) + sh(-2)) / 12.0 + 4.0 / 3.0 * (sh(1) + sh(-1)) - 2.5 * c
    lap = second(1) / box.dx ** 2 + second(0) / box.dy ** 2
    kin = -0.5 * float((c.conj() * lap).real.sum() / (c.real ** 2 + c.imag ** 2).sum())
    p = psi[box.iy, box.ix]
    n = p.real ** 2 + p.imag ** 2
    s = float(n.sum())
    pot, itr = float((v[box.iy, box.ix] * n).sum()) / s, 0.5 * g * float((n * n).sum()) / s
    return [kin + pot + itr, kin, pot, itr, 0.0, s * box.dx * box.dy]


def _rabi(a, b, var, dt, imag):
    w = complex(0.5 * PAIR["omega_r"], 0.5 * PAIR["omega_i"])
    m, x = abs(w), -dt * var * abs(w)
    if imag:
        c, s = math.cosh(x), w / m * math.sinh(x)
        return c * a + s * b, c * b + s.conjugate() * a
    c, s = math.cos(x), w / m * math.sin(x)
    return c * a + 1j * s * b, c * b + 1j * s.conjugate() * a


def _exact_pair(case, seed, device):
    box, a, b, va, vb = _pair_inputs(case, seed, device)
    dt, imag = _dt(case), case["imag"]
    sa, sb = _Step(box, dt, imag, PAIR["g_a"], 0.0), _Step(box, dt, imag, PAIR["g_b"], 0.0)
    ea, eb = _exp_table(va, dt, imag), _exp_table(vb, dt, imag)
    c_ab = PAIR["g_ab"] * dt
    na, nb = box.norm2(a), box.norm2(b)
    total = na + nb
    a, b = _rabi(a, b, 0.5, dt, imag)
    n = case["steps"]
    for i in range(n):
        last = i == n - 1
        a1, b1 = sa(a, ea, b, c_ab), sb(b, eb, a, c_ab)
        if not last:
            a1, b1 = sa.exchange(a1), sb.exchange(b1)
        if imag:
            a1, b1 = a1 / torch.sqrt(box.norm2(a1) / na), b1 / torch.sqrt(box.norm2(b1) / nb)
        a, b = _rabi(a1, b1, 0.5 if last else 1.0, dt, imag)
        if imag:
            qa, qb = box.norm2(a), box.norm2(b)
            f = torch.sqrt((qa + qb) / total)
            a, b = a / f, b / f
            na, nb = qa / (qa + qb) * total, qb / (qa + qb) * total
    return [a, b]


def _exact_evolve(case, seed, device, steps):
    box = _box(case)
    psi, v = _state(case, box, seed, device), _potential(case, box, seed, device)
    step, e = _Step(box, _dt(case), False, case["g"], case["lhy"]), _exp_table(v, _dt(case), False)
    for i in range(steps):
        psi = step(psi, e)
        if i < steps - 1:
            psi = step.exchange(psi)
    return psi


def _exact_gradient(case, seed, device):
    """Reverse mode through the steps.  On periodic axes a halo cell is a copy of
    the inner cell it mirrors: the derivative is the inner cell's, and zero on the halo."""
    box = _box(case)
    per = box.px or box.py
    psi0, v0 = _state(case, box, seed, device), _potential(case, box, seed, device)
    step = _Step(box, _dt(case), False, case["g"], case["lhy"])
    dt, t = _dt(case), _target(box, seed, device)
    inner = (box.iy, box.ix)

    def wrap(q):
        return torch.nn.functional.pad(q[None, None], (HALO * box.px,) * 2 + (HALO * box.py,) * 2, mode="circular")[0, 0] if per else q

    def wrapc(q):
        return torch.complex(wrap(q.real), wrap(q.imag)) if per else q
    v = v0[inner].clone().requires_grad_(True)
    re, im = (x[inner].clone().requires_grad_(True) for x in (psi0.real, psi0.imag))

    def one(p, vv):
        return step(wrapc(p), _exp_table(wrap(vv), dt, False))[inner]
    psi = torch.complex(re, im)
    for _ in range(case["steps"]):
        psi = checkpoint(one, psi, v, use_reentrant=False)
    c = (t[inner].conj() * psi).sum() * (box.dx * box.dy)
    loss = 1.0 - (c.real ** 2 + c.imag ** 2)
    loss.backward()

    def whole(gr):
        out = torch.zeros((box.H, box.W), dtype=torch.float64, device=device)
        out[inner] = gr
        return out
    return [loss.detach(), whole(v.grad), whole(re.grad), whole(im.grad)]


def exact(case, seed, device="cuda"):
    device = torch.device(device)
    kind = case["kind"]
    if kind == "gradient":
        return _exact_gradient(case, seed, device)
    with torch.no_grad():
        if kind == "batch":
            return [_exact_evolve(c, s, device, case["steps"]) for c, s in _batch_cases(case, seed)]
        if kind == "pair":
            return _exact_pair(case, seed, device)
        if kind == "evolve":
            psi = _exact_evolve(case, seed, device, case["steps"])
            return [psi.real, psi.imag]
        if kind == "timedep":
            box, psi, v0, v1 = _timedep_inputs(case, seed, device)
            dt, t = _dt(case), 0.0
            step = _Step(box, dt, False, case["g"], case["lhy"])
            for i in range(case["steps"]):
                v = v0 if i == 0 else _drive(v0, v1, t)
                psi = step(psi, _exp_table(v, dt, False))
                if i < case["steps"] - 1:
                    psi = step.exchange(psi)
                t += dt
            return [psi.real, psi.imag]
        box = _box(case)
        psi, v = _state(case, box, seed, device), _potential(case, box, seed, device)
        step, e = _Step(box, _dt(case), True, case["g"], case["lhy"]), _exp_table(v, _dt(case), True)
        target, energies = box.norm2(psi), []
        n = case["steps"] // case["chunks"]
        for _ in range(case["chunks"]):
            for i in range(n):
                psi = step(psi, e)
                if i < n - 1:
                    psi = step.exchange(psi)
                psi = psi / torch.sqrt(box.norm2(psi) / target)
            energies.append(_energy(box, psi, v, case["g"]))
        return [psi.real, psi.imag, torch.tensor(energies, dtype=torch.float64)]
