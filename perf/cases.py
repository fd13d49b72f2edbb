"""What a user of this framework has it do, as cases that can be timed.

Each case is one pass through the public Python interface (``Spectral2D``,
``FilteredSampler``, ``Ensemble``, ``ClosureNet``) of a program that keeps its
simulation, ensemble or network between passes:

- ``steps``     device-resident RK3 steps with the CFL step, then the w and
                psi fields brought up to date for the program's own device code
- ``dropin``    one step of the Fortran drop-in's default mode: w from a host
                buffer, the step, w and psi back into host buffers
- ``literal``   the reference's IntegrateOneStep routine by routine
- ``rhs``       ComputePsi and ComputeRHS on a (rectangular) grid
- ``output``    what a write of a restart and of the statistics needs: w, psi,
                u and v in physical space, the diagnostics, the shell spectrum
- ``snapshot``  one filtered sample (w, psi and the subgrid flux) of a DNS
- ``ensemble``  a batch of independent runs of mixed sizes, and its diagnostics
- ``closure``   coarse runs with the learned closure, one network call for all
- ``gradient``  loss and gradient of the closure network on a batch
- ``forward``   the network's output on a batch

``exact`` states the same in 64 bits with torch alone.
"""
import json
import math
import os

import numpy as np
import torch

from spectral2d_amd import NO_DEALIASING, _lib
from spectral2d_amd.closure import FilteredSampler
from spectral2d_amd.cnn import ClosureNet, param_count
from spectral2d_amd.ensemble import Ensemble
from spectral2d_amd.spectral import FP32, FP64, Spectral2D

NU = 1.0e-4
CFL = 0.5
DATA = os.path.join(os.path.dirname(os.path.abspath(_lib.__file__)), "data")


def listed():
    return [
        # a small run driven by an unchanged Fortran program: host buffers in and out
        {"name": "dropin_64_fp64", "kind": "dropin", "n": 64},
        # a size between the powers of two (padded 144), where launches count
        {"name": "steps_96_fp64", "kind": "steps", "n": 96, "fp64": True, "steps": 8},
        # the same at an ordinary size (padded 1152)
        {"name": "steps_768_fp64", "kind": "steps", "n": 768, "fp64": True, "steps": 4},
        # the headline run: decaying turbulence, 1024^2 FP64
        {"name": "steps_1024_fp64", "kind": "steps", "n": 1024, "fp64": True, "steps": 10},
        # the DNS that the closure's data comes from
        {"name": "steps_2048_fp32", "kind": "steps", "n": 2048, "fp64": False, "steps": 4},
        # a program that composes the step from the reference's routines
        {"name": "literal_1024_fp64", "kind": "literal", "n": 1024, "fp64": True},
        # the same routines on a small rectangular grid
        {"name": "rhs_96x64_fp64", "kind": "rhs", "nx": 96, "ny": 64, "fp64": True},
        # one write of fields and statistics of the headline run
        {"name": "output_1024_fp64", "kind": "output", "n": 1024, "fp64": True},
        # one training sample of the closure network
        {"name": "snapshot_2048_256", "kind": "snapshot", "n": 2048, "nc": 256},
        # the ensemble of decaying-turbulence runs, with its statistics read
        {"name": "ensemble_256_fp32", "kind": "ensemble", "runs": 256, "small": 128, "large": 512,
         "fp64": False, "steps": 20},
        # evaluation of the learned closure: sixteen members, two refreshes
        {"name": "closure_16x256", "kind": "closure", "n": 256, "runs": 16, "steps": 16,
         "every": 8},
        # one training step's loss and gradient at the training batch
        {"name": "gradient_256x16", "kind": "gradient", "h": 256, "w": 256, "batch": 16},
    ]


def _size(rng, lo, hi):
    """A resolved size 2^a 3^b (b <= 2) in [lo, hi], even over the logarithm."""
    ok = sorted({2 ** a * 3 ** b for a in range(3, 12) for b in range(3)})
    ok = [n for n in ok if lo <= n <= hi]
    x = math.exp(rng.uniform(math.log(lo), math.log(hi)))
    return min(ok, key=lambda n: abs(math.log(n / x)))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "dropin", "literal", "rhs", "output", "snapshot",
                       "ensemble", "closure", "gradient", "forward"])
    c = {"kind": kind}
    if kind not in ("ensemble", "gradient", "forward"):
        c["k0"] = round(rng.uniform(4.0, 16.0), 2)  # where the flow's energy peaks
    if kind == "steps":
        c["n"] = _size(rng, 32, 2048)
        c["fp64"] = rng.random() < 0.6 and c["n"] <= 1536
        c["steps"] = rng.randint(1, max(1, min(12, 3 * 2048 ** 2 // c["n"] ** 2)))
    elif kind == "dropin":
        c["n"] = _size(rng, 32, 768)
    elif kind == "literal":
        c["n"] = _size(rng, 32, 1152)
        c["fp64"] = rng.random() < 0.7
    elif kind == "rhs":
        c["nx"], c["ny"] = _size(rng, 32, 1024), _size(rng, 32, 1024)
        c["fp64"] = rng.random() < 0.7
    elif kind == "output":
        c["n"] = _size(rng, 64, 1536)
        c["fp64"] = rng.random() < 0.7
    elif kind == "snapshot":
        c["n"] = _size(rng, 256, 2048)
        c["nc"] = rng.choice([n for n in (32, 64, 96, 128, 192, 256) if 2 * n <= c["n"]])
    elif kind == "ensemble":
        c["fp64"] = rng.random() < 0.25
        c["runs"] = int(math.exp(rng.uniform(math.log(2), math.log(128 if c["fp64"] else 256))))
        c["small"] = rng.choice([64, 128])
        c["large"] = rng.choice([128, 256, 512])
        c["steps"] = rng.randint(4, 20)
    elif kind == "closure":
        c["n"] = 256
        c["runs"] = rng.randint(1, 24)
        c["every"] = rng.choice([4, 8, 12])
        c["steps"] = rng.randint(4, 16)
    else:
        c["h"], c["w"] = 8 * rng.randint(4, 32), rng.choice([128, 256, 384])
        c["batch"] = rng.randint(1, 10)
    return c


# ------------------------------------------------- flows and networks in 64 bits

class _Grid:
    """Wavenumbers, masks and the RK3 step of the (padded) grid, FP64 on the
    GPU, fields as half spectra [..., nyG, nxG / 2 + 1]."""

    def __init__(self, nx, ny=None, pad=True):
        ny = nx if ny is None else ny
        self.nx, self.ny = nx, ny
        self.nxG, self.nyG = (3 * nx // 2, 3 * ny // 2) if pad else (nx, ny)
        kx = torch.arange(self.nxG // 2 + 1, device="cuda", dtype=torch.float64)
        ky = torch.arange(self.nyG, device="cuda", dtype=torch.float64)
        ky = torch.where(ky > self.nyG // 2, ky - self.nyG, ky)[:, None]
        self.k2 = kx * kx + ky * ky
        self.inv_k2 = torch.where(self.k2 > 0, 1.0 / self.k2.clamp(min=1.0), 0.0)
        self.kept = (self.k2 <= (nx // 2) ** 2).double()
        # derivatives drop the Nyquist column and row
        self.ikx = 1j * torch.where(kx == self.nxG // 2, 0.0, kx)
        self.iky = 1j * torch.where(ky == self.nyG // 2, 0.0, ky)
        self.weight = torch.where((kx == 0) | (kx == self.nxG // 2), 0.5, 1.0)  # half the mode count
        self.shell = torch.floor(torch.sqrt(self.k2) + 0.5).long()

    def phys(self, f):
        return torch.fft.irfft2(f, s=(self.nyG, self.nxG), norm="forward")

    def spec(self, f):
        return torch.fft.rfft2(f, norm="forward")

    def turbulence(self, seed, k0, developed=False, ke=0.5):
        """Decaying-turbulence vorticity, one field per entry of k0, scaled to
        kinetic energy ke: E ~ k^4 exp(-(k / k0)^2) as a run starts, or with
        the k^-3 range of a developed flow."""
        k0 = torch.as_tensor(k0, dtype=torch.float64, device="cuda").reshape(-1, 1, 1)
        gen = torch.Generator(device="cuda").manual_seed(int(seed))
        noise = torch.randn(k0.shape[0], self.nyG, self.nxG, generator=gen, device="cuda",
                            dtype=torch.float64)
        k = torch.sqrt(self.k2)
        cut = (self.k2 < (min(self.nx, self.ny) // 2) ** 2) & (self.k2 > 0)
        if developed:
            shape = torch.exp(-(2.0 * k / self.nx) ** 2) / torch.sqrt(1.0 + (k / k0) ** 7)
        else:
            shape = torch.exp(-0.5 * (k / k0) ** 2)
        w = self.spec(noise) * cut * k ** 2.5 * shape
        tke = (self.weight * w.abs() ** 2 * self.inv_k2).sum((-2, -1), keepdim=True)
        return w * torch.sqrt(ke / tke)

    def velocity(self, psi):
        return self.iky * psi, -self.ikx * psi

    def rhs(self, w, nu, forcing=0.0):
        u, v = (self.phys(f) for f in self.velocity(w * self.inv_k2))
        om = self.phys(w)
        n = self.ikx * self.spec(u * om) * self.kept + self.iky * self.spec(v * om) * self.kept
        return -n - nu * self.k2 * w - forcing

    def cfl_dt(self, w):
        u, v = (self.phys(f) for f in self.velocity(w * self.inv_k2))
        top = (u.abs() + v.abs()).amax((-2, -1), keepdim=True)
        return CFL * (2.0 * math.pi / self.nx) / top

    def step(self, w, nu, dt, forcing=0.0):
        a = (w + dt * self.rhs(w, nu, forcing)) * self.kept
        a = (0.75 * w + 0.25 * a + 0.25 * dt * self.rhs(a, nu, forcing)) * self.kept
        return (w / 3 + 2 * a / 3 + 2 * dt / 3 * self.rhs(a, nu, forcing)) * self.kept

    def steps(self, w, nu, n):
        for _ in range(n):
            w = self.step(w, nu, self.cfl_dt(w))
        return w

    def diagnostics(self, w):
        """tke, enstrophy, palinstrophy and the largest mode of each field."""
        e = self.weight * w.abs() ** 2
        return torch.stack([(e * self.inv_k2).sum((-2, -1)), e.sum((-2, -1)),
                            (e * self.k2).sum((-2, -1)), w.abs().amax((-2, -1))], -1)

    def spectrum(self, psi, nu):
        nb = int(math.hypot(self.nxG // 2, self.nyG // 2) + 1.0) + 1
        u, v = self.velocity(psi)
        e = self.weight * (u.abs() ** 2 + v.abs() ** 2)
        sh = self.shell.reshape(-1)
        ek = torch.zeros(nb, dtype=torch.float64, device="cuda").index_add_(0, sh, e.reshape(-1))
        cnt = torch.bincount(sh, (2 * self.weight).expand_as(self.k2).reshape(-1), minlength=nb)
        b = torch.arange(nb, dtype=torch.float64, device="cuda")
        return [ek, cnt.to(torch.int32), ek.sum().item(), 2 * nu * (b ** 2 * ek).sum().item(),
                2 * nu * (b ** 4 * ek).sum().item()]

    def coarse(self, w, n):
        """The n x n samples of the modes |k| <= n / 2 of w."""
        return _sampled(w * (self.k2 <= (n // 2) ** 2), self.nyG, n)


def _sampled(w, nyG, n):
    h = n // 2
    s = torch.zeros(*w.shape[:-2], n, h + 1, dtype=w.dtype, device=w.device)
    s[..., : h + 1, :] = w[..., : h + 1, : h + 1]
    s[..., h + 1:, :] = w[..., nyG - h + 1: nyG, : h + 1]
    s[..., h, :] += w[..., nyG - h, : h + 1]  # +n/2 and -n/2 are one row, and one column
    s[..., h] *= 2.0
    return torch.fft.irfft2(s, s=(n, n), norm="forward")


def _network(p, x):
    """The closure network on x [batch, h, w, 2] with parameters p, 64 bits."""
    def conv(x, taps, b):  # taps [9][ci][co]
        y = b
        for t in range(9):
            y = y + torch.roll(x, (1 - t // 3, 1 - t % 3), (1, 2)) @ taps[t]
        return y
    at = 0

    def take(*shape):
        nonlocal at
        n = math.prod(shape)
        at += n
        return p[at - n: at].reshape(shape)
    gelu = torch.nn.functional.gelu
    x = gelu(conv(x, take(9, 2, 64), take(64)))
    for _ in range(4):
        taps = take(9, 64, 64).transpose(1, 2)
        x = gelu(conv(x, taps, take(64)))
    taps = take(9, 64, 1)
    return conv(x, taps, take(1))[..., 0]


def _random_params(gen):
    """Weights as the training run starts from."""
    p = []
    for ci, co in [(2, 64)] + 4 * [(64, 64)] + [(64, 1)]:
        p.append(torch.randn(9 * ci * co, generator=gen, device="cuda") * math.sqrt(2.0 / (9 * ci)))
        p.append(0.1 * torch.randn(co, generator=gen, device="cuda"))
    p = torch.cat(p)
    assert p.numel() == param_count()
    return p


def _batch(case, seed):
    """Smooth unit-variance planes (inputs w, psi and a target), FP32, dense."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    b, h, w = case["batch"], case["h"], case["w"]
    ky = torch.fft.fftfreq(h, 1.0 / h, device="cuda")[:, None]
    kx = torch.fft.rfftfreq(w, 1.0 / w, device="cuda")
    amp = torch.exp(-0.5 * (kx * kx + ky * ky) / 400.0)
    f = torch.fft.irfft2(torch.fft.rfft2(torch.randn(3, b, h, w, generator=gen, device="cuda")) * amp,
                         s=(h, w))
    f = (f / f.std((1, 2, 3), keepdim=True)).contiguous()
    return f, _random_params(gen)


def _shipped():
    """The committed closure network: parameters and scales."""
    with np.load(os.path.join(DATA, "closure_cnn_256.npz")) as z:
        return z["params"].astype(np.float32), tuple(float(s) for s in z["scales"])


def _host(w):
    """A half spectrum as the host buffer of set_field / set_vorticity."""
    return torch.view_as_real(w).cpu().numpy().reshape(-1)


def _members(case, seed):
    """Sizes, viscosities and initial vorticity {size: (runs, field)} of an ensemble."""
    rng = np.random.RandomState(seed % (1 << 32))
    sizes = [n for n in (64, 128, 256, 512) if case["small"] <= n <= max(case["small"], case["large"])]
    n = rng.choice(sizes, case["runs"])
    k0 = rng.uniform(4.0, 16.0, case["runs"])
    nu = 10.0 ** rng.uniform(-4.0, -3.0, case["runs"])
    fields = {}
    for size in sizes:
        at = np.flatnonzero(n == size)
        if at.size:
            fields[size] = at, _Grid(size).turbulence(seed + size, k0[at])
    return n, nu, fields


class _Slot:
    """A device slot as an array that torch can take without a copy."""

    def __init__(self, sim, f):
        self.sim = sim  # keeps the memory
        self.__cuda_array_interface__ = {
            "shape": (sim.nyG, sim.rISize), "strides": None, "version": 2,
            "typestr": "<f8" if sim.precision == FP64 else "<f4",
            "data": (sim.device_ptr(f), False)}


def _slot(sim, f):
    return torch.as_tensor(_Slot(sim, f), device="cuda")


def _precision(case):
    return FP64 if case["fp64"] else FP32


# --------------------------------------------------------------- the passes

def prepare(case, seed):
    kind = case["kind"]
    s = {"case": case}
    if kind in ("steps", "dropin", "literal", "output", "snapshot", "rhs"):
        nx, ny = case.get("nx", case.get("n")), case.get("ny", case.get("n"))
        prec = FP64 if kind == "dropin" else FP32 if kind == "snapshot" else _precision(case)
        sim = s["sim"] = Spectral2D(nx, ny, precision=prec)
        w = _Grid(nx, ny).turbulence(seed, case.get("k0", 10.0), kind == "snapshot")[0]
        s["w"] = _host(w)
        sim.set_field("w", s["w"])
        sim.ComputePsi()
        s["dt"] = 0.1 * 2.0 * math.pi / nx
        if kind == "dropin":
            s["psi"] = sim.get_field("psi")
        elif kind == "snapshot":
            s["sampler"] = FilteredSampler(sim, case["nc"])
        else:
            s["slots"] = {f: _slot(sim, f) for f in ("w", "psi", "u", "v", "wS", "psiS", "dW")}
    elif kind in ("ensemble", "closure"):
        runs = case["runs"]
        if kind == "ensemble":
            n, nu, fields = _members(case, seed)
            prec = _precision(case)
        else:
            n, nu, prec = np.full(runs, case["n"]), np.full(runs, 2.0e-5), FP32
            w = _Grid(case["n"]).turbulence(seed, runs * [case.get("k0", 12.0)], True)
            fields = {case["n"]: (np.arange(runs), w)}
            params, scales = _shipped()
            s["grid"] = Spectral2D(case["n"], dealias=NO_DEALIASING, precision=FP32)
            s["net"] = ClosureNet(case["n"], case["n"], runs)
            s["net"].set_params(params)
            s["net"].set_scales(*scales)
        s["ens"] = ens = Ensemble(n, prec)
        ens.set_viscosity(nu)
        for at, w in fields.values():
            for r, f in zip(at, w.cpu()):
                ens.set_vorticity(int(r), _host(f))
        # the members whose fields the program looks at: the first of each size
        s["look"] = [int(at[0]) for at, _ in fields.values()]
    else:
        s["planes"], params = _batch(case, seed)
        s["net"] = ClosureNet(case["h"], case["w"], case["batch"])
        s["net"].set_params(params.cpu().numpy())
        s["tau"] = torch.empty_like(s["planes"][0])
    return s


def run(s):
    case = s["case"]
    kind, sim = case["kind"], s.get("sim")
    if kind == "steps":
        sim.rk3_steps(case["steps"], NU, 0.0, CFL)
        sim.sync_fields()
        return s["slots"]["w"], s["slots"]["psi"]
    if kind == "dropin":
        sim.set_field("w", s["w"])
        sim.rk3_step(NU, s["dt"])
        return sim.get_field("w", s["w"]), sim.get_field("psi", s["psi"])
    if kind == "literal":
        sim.IntegrateOneStep(NU, s["dt"])
        return s["slots"]["w"], s["slots"]["psi"]
    if kind == "rhs":
        sim.copy_field("w", "wS")
        sim.ComputePsi("wS", "psiS")
        sim.ComputeRHS(NU, "u", "v", "wS", "psiS", "dW")
        return s["slots"]["dW"], s["slots"]["psiS"], s["slots"]["wS"]
    if kind == "output":
        sim.copy_field("w", "wS")
        sim.copy_field("psi", "psiS")
        sim.ComputeVelocity("u", "v", "psi", trans=True)
        sim.TransformC2R("wS")
        sim.TransformC2R("psiS")
        d = sim.diagnostics()
        ek, cnt, *sums = sim.ComputeSpectrum(NU)
        stats = np.array([d["tke"], d["enstrophy"], d["palinstrophy"], d["max_abs_w"]] + sums)
        if not case["fp64"]:  # sums of FP32 modes are good to 32 bits
            stats, ek = stats.astype(np.float32), ek.astype(np.float32)
        n = sim.nxG
        return [s["slots"][f][:, :n] for f in ("wS", "psiS", "u", "v")], stats, ek, cnt
    if kind == "snapshot":
        return s["sampler"].snapshot()
    if kind in ("ensemble", "closure"):
        ens = s["ens"]
        if kind == "ensemble":
            ens.steps(case["steps"], cfl=CFL, graph=True)
        else:
            ens.closure_steps(s["grid"], s["net"], case["steps"], cfl=CFL, every=case["every"])
        d = ens.diagnostics()
        keys = ("tke", "enstrophy", "palinstrophy", "max_abs_w")
        # the members' values are good to their precision
        to = np.float64 if case.get("fp64") else np.float32
        return (np.array([[x[k] for k in keys] for x in d]).astype(to),
                [ens.get_field(r).astype(to) for r in s["look"]])
    x, b = s["planes"], case["batch"]
    plane, ld = case["h"] * case["w"], case["w"]
    if kind == "gradient":
        loss, g = s["net"].gradient(b, x[0].data_ptr(), x[1].data_ptr(), plane, ld,
                                    x[2].data_ptr(), plane, ld)
        return np.float32(loss), g
    s["net"].forward(b, x[0].data_ptr(), x[1].data_ptr(), plane, ld, s["tau"].data_ptr(), plane, ld)
    return s["tau"]


# ------------------------------------------------------------- what is needed

def _step_work(n, steps, size):
    """Bytes and operations of RK3 steps: the mixed fields of each stage once
    each way (3 + 2 padded fields), the kept modes; 5 n log2 n a transform."""
    k, p = n // 2 + 1, 3 * n // 2
    lg = math.log2(p)
    return {"bytes": steps * 3 * 2 * size * k * (10 * p + 4 * n),
            "flops": steps * 3 * (5 * k * 5 * p * lg + 2.5 * p * 5 * p * lg)}


def _net_flops(case, times):
    return times * 2.0 * (9 * 2 * 64 + 4 * 9 * 64 * 64 + 9 * 64) * case["batch"] * case["h"] * case["w"]


def work(case):
    kind = case["kind"]
    size = 8 if case.get("fp64", kind == "dropin") else 4
    if kind == "steps":
        w = _step_work(case["n"], case["steps"], size)
        out = 2 * 2 * size * (3 * case["n"] // 2) * (3 * case["n"] // 4 + 1)
        return {"bytes": w["bytes"] + out, "flops": w["flops"]}
    if kind == "dropin":
        w = _step_work(case["n"], 1, 8)
        return {"bytes": w["bytes"] + 3 * 16 * (3 * case["n"] // 2) * (3 * case["n"] // 4 + 1),
                "flops": w["flops"]}
    if kind in ("literal", "rhs", "output", "snapshot"):
        nx, ny = case.get("nx", case.get("n")), case.get("ny", case.get("n"))
        x, y = 3 * nx // 2, 3 * ny // 2
        field = 2 * size * (x // 2 + 1) * y  # bytes
        lg = math.log2(x * y)
        # a 2D transform is two passes over its field, each read and written
        transforms, others = {"literal": (18, 12), "rhs": (6, 5), "output": (4, 5),
                              "snapshot": (6, 3)}[kind]
        return {"bytes": field * (4 * transforms + others), "flops": transforms * 2.5 * x * y * lg}
    if kind == "ensemble":
        sizes = [n for n in (64, 128, 256, 512) if case["small"] <= n <= max(case["small"], case["large"])]
        per = [_step_work(n, case["steps"], size) for n in sizes]
        return {k: case["runs"] * sum(p[k] for p in per) / len(per) for k in ("bytes", "flops")}
    if kind == "closure":
        w = _step_work(case["n"], case["steps"], 4)
        net = {"h": case["n"], "w": case["n"], "batch": 1}
        calls = -(-case["steps"] // case["every"])
        act = 2 * 64 * case["n"] ** 2
        return {"bytes": case["runs"] * (w["bytes"] + calls * 10 * act),
                "flops": case["runs"] * (w["flops"] + _net_flops(net, calls))}
    # activations (BF16, 64 channels) of five layers written and read: z and
    # gelu(z) forward, both and the gradient of each backward
    act = 2 * 64 * case["batch"] * case["h"] * case["w"]
    if kind == "gradient":
        return {"bytes": 35 * act, "flops": _net_flops(case, 3)}
    return {"bytes": 10 * act, "flops": _net_flops(case, 1)}


# ------------------------------------------------------- the same in 64 bits

def _real(w):
    """A half spectrum in the layout of a device slot."""
    return torch.view_as_real(w.contiguous()).reshape(w.shape[-2], -1)


def _closure_forcing(g, w, params, scales, guard=True):
    """Kept modes of the network's output for fields w on grid g."""
    n, h = g.nx, g.nx // 2
    x = torch.stack([g.coarse(w, n) * scales[0], g.coarse(w * g.inv_k2, n) * scales[1]], -1)
    with torch.no_grad():
        tau = torch.fft.rfft2(scales[2] * _network(params, x), norm="forward")
    f = torch.zeros_like(w)
    tau[..., h] *= 0.5
    f[..., : h + 1, : h + 1] = tau[..., : h + 1, :]
    f[..., g.nyG - h:, : h + 1] = tau[..., h:, :]
    f[..., h, : h + 1] *= 0.5
    f[..., g.nyG - h, : h + 1] *= 0.5
    f = f * g.kept
    col = f[..., :, 0]
    f[..., :, 0] = 0.5 * (col + torch.roll(col.flip(-1), 1, -1).conj())
    if guard:  # shells that the forcing would feed keep none of it
        e = (g.weight * (w.conj() * f).real).reshape(w.shape[0], -1)
        nb = int(g.shell.max()) + 1
        sums = torch.zeros(w.shape[0], nb, dtype=torch.float64, device="cuda")
        sums.index_add_(1, g.shell.reshape(-1), e)
        f = f * (sums >= 0.0)[:, g.shell]
    return f


def exact(case, seed):
    kind = case["kind"]
    if kind in ("gradient", "forward"):
        planes, params = _batch(case, seed)
        x = torch.stack([planes[0], planes[1]], -1).double()
        p = params.double().requires_grad_(kind == "gradient")
        y = _network(p, x)
        if kind == "forward":
            return y
        loss = ((y - planes[2].double()) ** 2).mean()
        loss.backward()
        return loss.item(), p.grad
    if kind == "ensemble":
        n, nu, fields = _members(case, seed)
        stats = torch.zeros(case["runs"], 4, dtype=torch.float64, device="cuda")
        look = []
        for size, (at, w) in fields.items():
            g = _Grid(size)
            w = g.steps(w, torch.as_tensor(nu[at], device="cuda").reshape(-1, 1, 1), case["steps"])
            stats[torch.as_tensor(at, device="cuda")] = g.diagnostics(w)
            look.append(_real(w[0]).reshape(-1))
        return stats, look
    if kind == "closure":
        g = _Grid(case["n"])
        w = g.turbulence(seed, case["runs"] * [case.get("k0", 12.0)], True)
        params, scales = _shipped()
        params = torch.as_tensor(params, device="cuda").double()
        for k in range(case["steps"]):
            if k % case["every"] == 0:
                f = _closure_forcing(g, w, params, scales)
            w = g.step(w, 2.0e-5, g.cfl_dt(w), f)
        return g.diagnostics(w), [_real(w[0]).reshape(-1)]
    nx, ny = case.get("nx", case.get("n")), case.get("ny", case.get("n"))
    g = _Grid(nx, ny)
    w = g.turbulence(seed, case.get("k0", 10.0), kind == "snapshot")[0]
    dt = 0.1 * 2.0 * math.pi / nx
    if kind == "steps":
        w = g.steps(w, NU, case["steps"])
        return _real(w), _real(w * g.inv_k2)
    if kind in ("dropin", "literal"):
        w = g.step(w, NU, dt)
        out = _real(w), _real(w * g.inv_k2)
        return tuple(x.reshape(-1) for x in out) if kind == "dropin" else out
    if kind == "rhs":
        return _real(g.rhs(w, NU)), _real(w * g.inv_k2), _real(w)
    if kind == "output":
        psi = w * g.inv_k2
        u, v = g.velocity(psi)
        ek, cnt, *sums = g.spectrum(psi, NU)
        stats = torch.cat([g.diagnostics(w), torch.tensor(sums, device="cuda", dtype=torch.float64)])
        return [g.phys(f) for f in (w, psi, u, v)], stats, ek, cnt
    nc = case["nc"]
    c, h = _Grid(nc), nc // 2

    def cut(f):  # the modes |k| <= nc / 2 on the coarse padded grid
        z = torch.zeros(c.nyG, c.nxG // 2 + 1, dtype=f.dtype, device="cuda")
        z[: h + 1, : h + 1] = f[: h + 1, : h + 1]
        z[c.nyG - h:, : h + 1] = f[g.nyG - h:, : h + 1]
        return z * c.kept
    wb = cut(w)
    tau = c.rhs(wb, 0.0) - cut(g.rhs(w, 0.0))
    return tuple(c.coarse(f, nc) for f in (wb, wb * c.inv_k2, tau))
