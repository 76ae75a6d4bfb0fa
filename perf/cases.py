"""The work this library is used for, as cases that can be timed and checked.

Every case is one pass of a user's inner loop through the C API: some split-operator steps of
a wavefunction that stays on the GPU and a snapshot of it, a Fourier transform of a field, a
batch of 2-D ground states, or the warm-start network's prediction or gradient.  Sizes are those
of the workloads, the tests and the benchmark of this repository (32^3 .. 512^3, the 3 * 2^k
lengths, 2-D sheets), and draw() spreads over the supported lengths between them.

Cases by kind:
  propagate  grid_wf_propagate with a complex potential, real time (2nd or 4th order, with or
             without k-space cutoff, with or without absorbing boundary), then a snapshot
  gpe        grid_wf_gpe_propagate (Gross-Pitaevskii), real time, or imaginary time with
             renormalisation and the energy a relaxation loop looks at, then a snapshot
  relax      grid_wf_gpe_relax of the linear problem from a start state, a fixed step budget
  fft        cgrid_fft of a field and cgrid_inverse_fft_norm of a spectrum
  batch2d    grid_wf_batch2d_relax of many small 2-D problems, a fixed step budget
  gradient   grid_surrogate_gradient of a minibatch (64^3 potentials and targets)
  predict    grid_surrogate_predict
"""
import ctypes as C
import math

import numpy as np
import torch

import libgrid_amd as LG

STEP = 0.25  # grid spacing (bohr)

# ---- cases -----------------------------------------------------------------------------------


def listed():
    return [
        # the smallest grids in use (a quick look, the smoke run): every launch counts
        dict(name="propagate_32", kind="propagate", nx=32, ny=32, nz=32, prec="fp64", order=2, cutoff=False,
             absorb=False, steps=16),
        # the reference's own wave packet example: 128^3, harmonic trap, energy looked at now and then
        dict(name="propagate_128", kind="propagate", nx=128, ny=128, nz=128, prec="fp64", order=2, cutoff=False,
             absorb=False, steps=20),
        # a scattering run on an oblong box: absorbing layers, lengths that are not powers of two
        dict(name="absorb_96x192x128", kind="propagate", nx=96, ny=192, nz=128, prec="fp64", order=2, cutoff=False,
             absorb=True, steps=8),
        # the benchmark's workload: imaginary-time Gross-Pitaevskii relaxation on 256^3
        dict(name="gpe_256", kind="gpe", nx=256, ny=256, nz=256, prec="fp64", time="imaginary", g=0.1, steps=10),
        # the same step on the largest double-precision grid, which streams from memory
        dict(name="gpe_512", kind="gpe", nx=512, ny=512, nz=512, prec="fp64", time="imaginary", g=0.1, steps=2),
        # vortex dynamics: the largest grid in single precision, real time
        dict(name="vortex_512_fp32", kind="gpe", nx=512, ny=512, nz=512, prec="fp32", time="real", g=0.1, steps=3),
        # training data of the warm-start network: 64^3 single-precision relaxations
        dict(name="relax_64_fp32", kind="relax", nx=64, ny=64, nz=64, prec="fp32", steps=128),
        # a 2-D condensate (one trivial axis), real time
        dict(name="sheet_384x512", kind="gpe", nx=1, ny=384, nz=512, prec="fp64", time="real", g=0.1, steps=20),
        # a convolution's transforms on an oblong grid
        dict(name="fft_192x96x384", kind="fft", nx=192, ny=96, nz=384, prec="fp64"),
        # many small 2-D ground states in one call
        dict(name="batch2d_48", kind="batch2d", count=48, steps=128),
        # one training minibatch of the warm-start network
        dict(name="gradient_8", kind="gradient", batch=8),
        # one warm start
        dict(name="predict_1", kind="predict", batch=1),
    ]


LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512)


def draw(rng):
    kind = rng.choices(("propagate", "gpe", "relax", "fft", "batch2d", "gradient", "predict"),
                       (30, 30, 12, 10, 6, 6, 6))[0]
    if kind == "batch2d":
        return dict(kind=kind, count=round(math.exp(rng.uniform(math.log(8), math.log(128)))), steps=128)
    if kind in ("gradient", "predict"):
        return dict(kind=kind, batch=rng.randint(1, 8))
    # the number of points is spread over its logarithm, the shape around a cube
    flat = kind in ("propagate", "gpe") and rng.random() < 0.2
    lo, hi = (2 ** 12, 2 ** 18) if flat else (2 ** 13, 2 ** 25)
    n = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    shape = []
    for axis in range(2 if flat else 3):
        side = n ** (1.0 / (2 if flat else 3)) * math.exp(rng.uniform(-0.6, 0.6))
        shape.append(min(LENGTHS, key=lambda m: abs(math.log(m / side))))
    nx, ny, nz = ([1] + shape) if flat else shape
    points = nx * ny * nz
    case = dict(kind=kind, nx=nx, ny=ny, nz=nz)
    steps = max(4, min(24, 2 ** 27 // points))
    if kind == "propagate":
        order = rng.choice((2, 2, 4))
        case.update(prec=rng.choice(("fp64", "fp64", "fp32")), order=order, cutoff=rng.random() < 0.3,
                    absorb=order == 2 and not flat and rng.random() < 0.3, steps=steps)
    elif kind == "gpe":
        case.update(prec=rng.choice(("fp64", "fp64", "fp32", "fp32x")), time=rng.choice(("imaginary", "real")),
                    g=rng.choice((0.1, 0.0)), steps=steps)
    elif kind == "relax":
        case.update(prec=rng.choice(("fp64", "fp32")), steps=max(16, min(128, 2 ** 30 // points // 16 * 16)))
    else:
        case.update(prec=rng.choice(("fp64", "fp64", "fp32")))
    if case.get("prec") == "fp32" and kind != "fft":
        case["steps"] = min(case["steps"], 128 if kind == "relax" else 8)
    return case


# ---- grids on the device ---------------------------------------------------------------------

PREC = {"fp64": b"\x00", "fp32": b"\x01", "fp32x": b"\x02"}


class _Device(C.Structure):
    """Leading fields of a grid's device record: the element count and the device array."""

    _fields_ = [("kind", C.c_int), ("prec", C.c_int), ("n", C.c_size_t), ("d", C.c_void_p)]


class _View:
    """A grid's device array as torch sees it; keeps the grid alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=shape, typestr=typestr, data=(ptr, False), version=2)


class State:
    """The grids of one pass, freed with it."""

    def __init__(self, case):
        self.lib, self.case, self.frees = LG.load(), case, []

    def __del__(self):
        for free, handle in reversed(self.frees):
            free(handle)

    def cgrid(self, shape, step, prec, name):
        g = self.lib.cgrid_alloc(*shape, step, LG.boundary("cgrid_value_outside_periodic"), None, name)
        self.frees.append((self.lib.cgrid_free, g))
        self.lib.cgrid_set_precision(g, PREC[prec])
        return g

    def rgrid(self, shape, step, name):
        g = self.lib.rgrid_alloc(*shape, step, LG.boundary("rgrid_value_outside_periodic"), None, name)
        self.frees.append((self.lib.rgrid_free, g))
        return g

    def wf(self, shape, step, propagator, prec, name):
        w = self.lib.grid_wf_alloc(*shape, step, 1.0, LG.WF_PERIODIC_BOUNDARY, propagator, name)
        self.frees.append((self.lib.grid_wf_free, w))
        self.lib.cgrid_set_precision(w.contents.grid, PREC[prec])
        return w

    def view(self, g):
        """The device array of a grid that is current on the device."""
        c = g.contents
        dev = _Device.from_address(c.dev)
        typestr = "<f8" if dev.kind == 1 else "<c16" if dev.prec == 0 else "<c8"
        return torch.as_tensor(_View(self, dev.d, (c.nx, c.ny, c.nz), typestr), device="cuda")

    def fill(self, g, values):
        """Put values on the device: the grid becomes current there."""
        if isinstance(g.contents, LG.cgrid):
            self.lib.cgrid_constant(g, LG.c_complex(0.0, 0.0))
        else:
            self.lib.grid_wf_density(self.w, g)
        self.lib.grid_hip_sync()
        self.view(g).copy_(values)
        torch.cuda.synchronize()


# ---- inputs ----------------------------------------------------------------------------------


def _device():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _axes(shape):
    out = []
    for a, n in enumerate(shape):
        view = [1, 1, 1]
        view[a] = n
        out.append(((torch.arange(n, dtype=torch.float64, device=_device()) - n // 2) * STEP).reshape(view))
    return out


def _shape(case):
    return case["nx"], case["ny"], case["nz"]


def _volume(shape):
    return STEP ** sum(1 for n in shape if n > 1)


def _normalized(psi):
    return psi / torch.sqrt((psi.real ** 2 + psi.imag ** 2).sum() * _volume(psi.shape))


def _fields(case, seed):
    """A moving Gaussian packet and a trap with a few wells, at places that the seed draws."""
    shape = _shape(case)
    rng = np.random.default_rng([seed, 3])
    x = _axes(shape)
    half = [0.5 * n * STEP for n in shape]
    live = [n > 1 for n in shape]
    psi = 1.0
    centre, momentum = rng.uniform(-0.1, 0.1, 3), rng.uniform(-1.0, 1.0, 3)
    for a in range(3):
        if live[a]:
            d = x[a] - centre[a] * half[a]
            w = max(0.3 * half[a], 2 * STEP)
            psi = psi * torch.complex(-d * d / (w * w), momentum[a] * d).exp()
    psi = _normalized(psi.to(torch.complex128))
    v = sum((0.5 * 0.01 * x[a] ** 2 for a in range(3) if live[a]), torch.zeros(1, dtype=torch.float64, device=psi.device))
    for _ in range(4):
        depth, width, at = rng.uniform(0.05, 0.5), rng.uniform(0.1, 0.3), rng.uniform(-0.5, 0.5, 3)
        bump = -depth
        for a in range(3):
            if live[a]:
                bump = bump * torch.exp(-0.5 * ((x[a] - at[a] * half[a]) / (width * half[a])) ** 2)
        v = v + bump
    return psi.contiguous(), v.expand(shape).contiguous()


def _layers(case):
    """Absorbing layers of a quarter of each side."""
    out = []
    for n in _shape(case):
        out += [n // 4, n - 1 - n // 4] if n > 1 else [0, 0]
    return out


def _kmax():
    return 0.5 * math.sqrt(3.0) * math.pi / STEP


def _propagator(case):
    if case.get("order", 2) == 4:
        return LG.WF_4TH_ORDER_CFFT if case["cutoff"] else LG.WF_4TH_ORDER_FFT
    return LG.WF_2ND_ORDER_CFFT if case.get("cutoff") else LG.WF_2ND_ORDER_FFT


SIZES2D = (64, 96, 128, 192, 256)


def _problems2d(case, seed):
    """Small 2-D problems of every size: (start state, potential), wells drawn from the seed."""
    rng = np.random.default_rng([seed, 5])
    out = []
    for i in range(case["count"]):
        n = SIZES2D[i % len(SIZES2D)]
        box = n * 0.2
        x = (np.arange(n) - n // 2) * 0.2
        v = np.zeros((n, n))
        for _ in range(int(rng.integers(3, 9))):
            at, width, depth = rng.uniform(-0.3 * box, 0.3 * box, 2), rng.uniform(0.5, 3.0), rng.uniform(0.05, 0.5)
            e = [np.exp(-0.5 * ((x - c) / width) ** 2) for c in at]
            v -= depth * e[0][:, None] * e[1][None, :]
        e = np.exp(-0.5 * (x / (0.15 * box)) ** 2)
        psi = (e[:, None] * e[None, :]).astype(np.complex128)
        out.append((psi / np.sqrt(np.sum(np.abs(psi) ** 2) * 0.04), v))
    return out


SIDE, SCALE = 64, 2.0
CHANNELS = ((8, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 128), (128, 128), (192, 64), (64, 64), (96, 32),
            (32, 32), (48, 16))


def _network(case, seed):
    """Weights with the spread of a network in training, wells as potentials, amplitudes as targets."""
    rng = np.random.default_rng([seed, 7])
    parts = []
    for cin, cout in CHANNELS:
        parts += [rng.standard_normal(27 * cin * cout) * math.sqrt(2.0 / (27 * cin)), 0.01 * rng.standard_normal(cout)]
    parts.append(0.25 * rng.standard_normal(17))
    params = np.concatenate(parts).astype(np.float32).astype(np.float64)
    x = (np.arange(SIDE) - SIDE // 2) * 0.5
    pot, target = np.zeros((2, case["batch"], SIDE, SIDE, SIDE))
    for b in range(case["batch"]):
        for _ in range(int(rng.integers(4, 11))):
            at, width, depth = rng.uniform(-9.6, 9.6, 3), rng.uniform(0.5, 3.0), rng.uniform(0.05, 0.5)
            e = [np.exp(-0.5 * ((x - c) / width) ** 2) for c in at]
            bump = e[0][:, None, None] * e[1][None, :, None] * e[2][None, None, :]
            pot[b] -= depth * bump
            target[b] += depth * bump
        target[b] /= np.sqrt(np.mean(target[b] ** 2))
    # the interface takes doubles; the network holds 32 bits
    return params, *(a.astype(np.float32).astype(np.float64) for a in (pot, target))


def _doubles(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def prepare(case, seed):
    lib = LG.load()
    lib.grid_hip_enable(b"\x01", 1, None)
    s = State(case)
    kind = case["kind"]
    if kind in ("gradient", "predict"):
        params, s.pot, s.target = _network(case, seed)
        s.net = lib.grid_surrogate_alloc(SIDE, case["batch"], SCALE, 1)
        s.frees.append((lib.grid_surrogate_free, s.net))
        lib.grid_surrogate_set_params(s.net, _doubles(params))
        s.out = np.empty(len(params) if kind == "gradient" else s.pot.size)
        return s
    if kind == "batch2d":
        # the tile that the tuner settles on for this device
        lib.grid_batch2d_set_tile(0, 1024, 1)
        s.starts, wfs, pots = [], [], []
        for psi, v in _problems2d(case, seed):
            n = len(v)
            w = s.wf((1, n, n), 0.2, LG.WF_2ND_ORDER_FFT, "fp64", b"batch")
            r = s.rgrid((1, n, n), 0.2, b"wells")
            LG.set_rgrid(r, v.reshape(1, n, n))
            wfs.append(w)
            pots.append(r)
            s.starts.append(psi.reshape(1, n, n))
        s.wfs, s.pots = (LG.WF * len(wfs))(*wfs), (LG.RG * len(pots))(*pots)
        s.energies, s.taken = (C.c_double * len(wfs))(), (C.c_long * len(wfs))()
        return s
    shape, prec = _shape(case), case["prec"]
    psi, v = _fields(case, seed)
    if kind == "fft":
        s.a, s.b = s.cgrid(shape, STEP, prec, b"field"), s.cgrid(shape, STEP, prec, b"spectrum")
        s.fill(s.a, psi)
        s.fill(s.b, torch.fft.fftn(psi))
        s.fa, s.fb = s.cgrid(shape, STEP, prec, b"transformed"), s.cgrid(shape, STEP, prec, b"back")
        return s
    s.w = s.wf(shape, STEP, _propagator(case), prec, b"psi")
    s.w.contents.kmax = _kmax()
    s.fill(s.w.contents.grid, psi)
    s.out = s.cgrid(shape, STEP, prec, b"snapshot")
    if kind == "propagate":
        s.pot = s.cgrid(shape, STEP, "fp64", b"potential")
        s.fill(s.pot, v)
        if case["absorb"]:
            lib.grid_wf_boundary(s.w, None, *_layers(case))
    else:
        s.pot = s.rgrid(shape, STEP, b"vext")
        s.fill(s.pot, v)
    if kind == "relax":
        s.start = s.cgrid(shape, STEP, prec, b"start")
        s.fill(s.start, psi)
    return s


# ---- one pass --------------------------------------------------------------------------------

DT, DTAU = 0.05, 0.05


def run(s):
    lib, case = s.lib, s.case
    kind = case["kind"]
    if kind == "propagate":
        for _ in range(case["steps"]):
            lib.grid_wf_propagate(s.w, s.pot, LG.c_complex(DT, 0.0))
        lib.cgrid_copy(s.out, s.w.contents.grid)
        return s.view(s.out)
    if kind == "gpe":
        imaginary = case["time"] == "imaginary"
        t = LG.c_complex(0.0, -DTAU) if imaginary else LG.c_complex(DT, 0.0)
        for _ in range(case["steps"]):
            lib.grid_wf_gpe_propagate(s.w, s.pot, case["g"], t, b"\x01" if imaginary else b"\x00")
        lib.cgrid_copy(s.out, s.w.contents.grid)
        if imaginary and case["prec"] == "fp64":  # what a relaxation loop looks at
            return s.view(s.out), lib.grid_wf_gpe_last_energy(s.w)
        return s.view(s.out)
    if kind == "relax":
        lib.cgrid_copy(s.w.contents.grid, s.start)
        n = lib.grid_wf_gpe_relax(s.w, s.pot, 0.0, DTAU, 1e-14, case["steps"], None)
        lib.cgrid_copy(s.out, s.w.contents.grid)
        return s.view(s.out), n
    if kind == "fft":
        lib.cgrid_copy(s.fa, s.a)
        lib.cgrid_fft(s.fa)
        lib.cgrid_copy(s.fb, s.b)
        lib.cgrid_inverse_fft_norm(s.fb)
        return s.view(s.fa), s.view(s.fb)
    if kind == "batch2d":
        for w, psi in zip(s.wfs, s.starts):
            LG.set_cgrid(w.contents.grid, psi)
        lib.grid_wf_batch2d_relax(len(s.wfs), s.wfs, s.pots, 0.1, 1e-14, case["steps"], s.energies, s.taken)
        # the states are held in 32 bits; the interface widens them
        return np.concatenate([LG.get_cgrid(w.contents.grid).ravel() for w in s.wfs]).astype(np.complex64)
    n = case["batch"]
    if kind == "gradient":
        loss = lib.grid_surrogate_gradient(s.net, n, _doubles(s.pot), _doubles(s.target), _doubles(s.out))
        # gradients and loss are held in 32 bits; the interface widens them
        return s.out.astype(np.float32), np.float32(loss)
    lib.grid_surrogate_predict(s.net, n, _doubles(s.pot), _doubles(s.out))
    return s.out.astype(np.float32)


# ---- what a pass cannot do without -------------------------------------------------------------


def _points(case):
    return case["nx"] * case["ny"] * case["nz"]


def work(case):
    """Bytes: a step reads the state and the potential once and writes the state once.  Flops: two
    forward and two inverse transforms a step (5 N log2 N each) and the factors."""
    kind = case["kind"]
    if kind in ("propagate", "gpe", "relax", "fft"):
        n = _points(case)
        c = 16 if case["prec"] == "fp64" else 8
        fft = 5.0 * n * math.log2(n)
        if kind == "fft":
            return {"bytes": 4.0 * c * n, "flops": 2 * fft}
        per_bytes, per_flops = 2.0 * c * n + (c if kind == "propagate" else 8) * n, 4 * fft + 40.0 * n
        if case.get("absorb"):
            per_flops *= 2
        return {"bytes": case["steps"] * per_bytes, "flops": case["steps"] * per_flops}
    if kind == "batch2d":
        n = case["count"] * float(np.mean([m * m for m in SIZES2D]))
        # a state, its factors and its potential fit on the chip: read and written once
        return {"bytes": n * 36.0, "flops": case["steps"] * n * (2 * 5 * math.log2(n / case["count"]) + 20)}
    level = (0, 1, 1, 2, 2, 3, 3, 2, 2, 1, 1, 0)
    fwd = sum(2.0 * 27 * ci * co * SIDE ** 3 / 8 ** lv for (ci, co), lv in zip(CHANNELS, level)) * case["batch"]
    io = SIDE ** 3 * case["batch"]
    if kind == "predict":
        return {"bytes": 8.0 * 2 * io, "flops": fwd}
    return {"bytes": 8.0 * 2 * io + 8.0 * 1.45e6, "flops": 3 * fwd}


# ---- the same in 64 bits, without this library -------------------------------------------------


def _k2(shape, step):
    out = 0.0
    for a, n in enumerate(shape):
        if n == 1:
            continue
        k = torch.fft.fftfreq(n, d=step, dtype=torch.float64, device=_device()) * 2 * math.pi
        view = [1, 1, 1]
        view[a] = n
        out = out + (k * k).reshape(view)
    return out


def _kinetic(psi, t, k2, kmax=None):
    f = torch.fft.fftn(psi)
    f *= torch.exp(torch.complex(torch.zeros_like(k2), -0.5 * k2) * t)
    if kmax is not None:
        f[k2 >= kmax * kmax] = 0.0
    return torch.fft.ifftn(f)


def _split(psi, v, t, k2, order=2, kmax=None):
    def pot(t):
        return torch.exp(v * (-1j * t))

    if order == 4:
        psi = _kinetic(psi * pot(t / 6), t / 2, k2, kmax)
        return _kinetic(psi * pot(2 * t / 3), t / 2, k2, kmax) * pot(t / 6)
    psi = _kinetic(psi, t / 2, k2, kmax)
    return _kinetic(psi * pot(t), t / 2, k2, kmax)


def _absorption(shape, layers):
    t = torch.zeros(shape, dtype=torch.float64, device=_device())
    for a, n in enumerate(shape):
        lo, hi = layers[2 * a], layers[2 * a + 1]
        if not lo:
            continue
        i = torch.arange(n, dtype=torch.float64, device=t.device)
        s = torch.where(i < lo, (lo - i) / lo, torch.where(i > hi, (i - hi) / lo, torch.zeros_like(i)))
        view = [1, 1, 1]
        view[a] = n
        t = t + s.reshape(view)
    return torch.clamp(t * 2 / 3, max=1.0)


def _exact_network(case, seed):
    """The network by shifted products over channels, in 64 bits."""
    dev = _device()
    params, pot, target = _network(case, seed)
    p = torch.tensor(params, device=dev, requires_grad=case["kind"] == "gradient")
    x = torch.zeros(*pot.shape, 8, dtype=torch.float64, device=dev)
    x[..., 0] = SCALE * torch.tensor(pot, device=dev)
    layers, at = [], 0
    for cin, cout in CHANNELS:
        w = p[at:at + 27 * cin * cout].reshape(cout, 27, cin)
        at += 27 * cin * cout
        layers.append((w, p[at:at + cout]))
        at += cout

    def conv(x, layer):
        w, bias = layers[layer]
        y = bias
        for t in range(27):
            d = (t // 9 - 1, t // 3 % 3 - 1, t % 3 - 1)
            y = y + torch.roll(x, [-k for k in d], (1, 2, 3)) @ w[:, t].T
        return torch.relu(y)

    def pool(x):
        b, z, y, w, c = x.shape
        return x.reshape(b, z // 2, 2, y // 2, 2, w // 2, 2, c).mean((2, 4, 6))

    def up(x):
        return x.repeat_interleave(2, 1).repeat_interleave(2, 2).repeat_interleave(2, 3)

    e1 = conv(x, 0)
    e2 = conv(conv(pool(e1), 1), 2)
    e3 = conv(conv(pool(e2), 3), 4)
    y = conv(conv(pool(e3), 5), 6)
    y = conv(conv(torch.cat([up(y), e3], -1), 7), 8)
    y = conv(conv(torch.cat([up(y), e2], -1), 9), 10)
    y = conv(torch.cat([up(y), e1], -1), 11)
    out = y @ p[at:at + 16] + p[at + 16]
    if case["kind"] == "predict":
        return out.reshape(-1)
    loss = ((out - torch.tensor(target, device=dev)) ** 2).mean()
    loss.backward()
    return p.grad, loss.detach()


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gradient", "predict"):
        return _exact_network(case, seed)
    if kind == "batch2d":
        out = []
        for psi, v in _problems2d(case, seed):
            n = len(v)
            psi, v = (torch.tensor(a, device=_device()).reshape(1, n, n) for a in (psi, v))
            k2 = _k2((1, n, n), 0.2)
            kh, pv = torch.exp(-0.5 * 0.1 * k2 / 2), torch.exp(-0.1 * v)
            for _ in range(case["steps"]):
                psi = torch.fft.ifftn(kh * torch.fft.fftn(psi))
                psi = torch.fft.ifftn(kh * torch.fft.fftn(pv * psi))
                psi = psi / torch.sqrt((psi.abs() ** 2).sum() * 0.04)
            out.append(psi.reshape(-1))
        return torch.cat(out)
    psi, v = _fields(case, seed)
    if case["prec"] != "fp64":  # the inputs as they are held
        psi = psi.to(torch.complex64).to(torch.complex128)
    if kind == "fft":
        spectrum = torch.fft.fftn(_fields(case, seed)[0])
        if case["prec"] != "fp64":
            spectrum = spectrum.to(torch.complex64).to(torch.complex128)
        return torch.fft.fftn(psi), torch.fft.ifftn(spectrum)
    k2 = _k2(_shape(case), STEP)
    kmax = _kmax() if case.get("cutoff") else None
    dv = _volume(_shape(case))
    if kind == "propagate":
        if case["prec"] != "fp64":
            v = v.to(torch.float32).to(torch.float64)
        alpha = _absorption(_shape(case), _layers(case)) if case["absorb"] else None
        for _ in range(case["steps"]):
            forward = _split(psi, v, DT, k2, case["order"], kmax)
            if alpha is not None:
                forward = (1 - alpha) * forward + alpha * _split(psi, v, -1j * DT, k2, 2, kmax)
            psi = forward
        return psi
    imaginary = kind == "relax" or case["time"] == "imaginary"
    g = case.get("g", 0.0)
    energy = None
    for i in range(case["steps"]):
        rho = psi.real ** 2 + psi.imag ** 2
        if kind == "gpe" and imaginary and i == case["steps"] - 1:
            f = torch.fft.fftn(psi)
            kinetic = 0.5 * float((k2 * (f.real ** 2 + f.imag ** 2)).sum()) * dv / rho.numel()
            energy = kinetic + float((v * rho).sum()) * dv + 0.5 * g * float((rho * rho).sum()) * dv
            del f
        psi = _split(psi, v + g * rho, -1j * DTAU if imaginary else DT, k2)
        if imaginary:
            psi = _normalized(psi)
    if kind == "relax":
        return psi, None
    return (psi, energy) if imaginary and case["prec"] == "fp64" else psi
