"""Timed workloads of the framework, through its public entry points (``Solver`` and ``Batch``).

A case is one stretch of a simulation as the driver runs it: ``steps`` time steps in calls of
``check`` steps with the L1 test after each (the reference's loop tests L1 every 100 steps), a
surfTrack scan after each call where the case asks for one, and at the end the energy and the
field psi on the host.  The adjoint cases are one gradient, the batch cases one stretch of an
ensemble.  A state is a handle with its field loaded and its tile schedules tuned; a pass
continues the simulation from where the handle is.  Fields of FP32-mixed handles are taken as
float32, the precision they carry.

Physical parameters are those of the bench workloads and of the driver's presets: the cubic model at
8 points per wavelength (time steps 0.1, 0.05 and 0.02), or the reference's quintic constants at 16.
"""
import math

import numpy as np
import torch

from smectic3d_amd import Batch, Solver
from smectic3d_amd import _abi as A

LENGTHS = (16, 24, 32, 48, 64, 96, 128, 192, 256, 384, 512)


def _case(name, kind, nx, ny, nz, prec, steps, check, model="cubic", eps=0.3, dt=0.05, start="layers", **more):
    case = {"name": name, "kind": kind, "nx": nx, "ny": ny, "nz": nz, "prec": prec, "steps": steps, "check": check,
            "model": model, "eps": eps, "dt": dt, "start": start, "force": "mu", "w_mid": 0.0, "boxes": 1, "surf": False}
    case.update(more)
    return case


def listed():
    return [
        # a small box, the shortest kernels: parameter studies and the reference's constants at low resolution
        _case("periodic_48x32x64_f64_quintic", "periodic", 48, 32, 64, "f64", 500, 100, "quintic", -0.7, 1e-3),
        # the plain 64^3 preset from noise
        _case("periodic_64_f32", "periodic", 64, 64, 64, "f32", 200, 100, eps=0.5, dt=0.02, start="noise"),
        # an oblong box with the mid-plane penalty of the morphology runs
        _case("periodic_192x96x384_f64_penalty", "periodic", 192, 96, 384, "f64", 200, 100, "quintic", -0.7, 5e-4,
              w_mid=1.0),
        # the headline box, in the reference's arithmetic and in the mixed one
        _case("periodic_256_f64", "periodic", 256, 256, 256, "f64", 500, 100, dt=0.1),
        _case("periodic_256_f32", "periodic", 256, 256, 256, "f32", 300, 100, dt=0.02),
        # the reference's production size
        _case("periodic_512_f64", "periodic", 512, 512, 512, "f64", 100, 100),
        # Stokes advection: the reference's psiSH force in a small box, the mu force in the 256^3 workload
        _case("advected_96x64x128_f64_sh", "advected", 96, 64, 128, "f64", 200, 100, "quintic", -0.7, 1e-3, force="sh",
              start="noise"),
        _case("advected_256_f32_mu", "advected", 256, 256, 256, "f32", 100, 100, eps=0.5, dt=0.02, start="noise"),
        # DCT box of the surface runs: the plain steps in FP32, and with surfTrack every 20 steps in FP64
        _case("neumann_256x256x384_f32", "neumann", 256, 256, 384, "f32", 200, 100, eps=0.5, dt=0.02),
        _case("neumann_128x96x192_f64_surf", "neumann", 128, 96, 192, "f64", 200, 20, eps=0.5, surf=True),
        # an ensemble of uneven boxes in one graph, and the gradient of one box
        _case("batch_24_f32", "batch", 64, 96, 128, "f32", 200, 200, eps=0.4, dt=0.02, start="noise", boxes=24),
        _case("adjoint_128_f64", "adjoint", 128, 128, 128, "f64", 200, 50, start="noise"),
    ]


def draw(rng):
    kind = rng.choice(["periodic"] * 4 + ["advected", "advected", "neumann", "neumann", "neumann_advected", "batch", "adjoint"])
    prec = "f64" if kind == "adjoint" else rng.choice(["f64", "f32"])
    model = rng.choice(["cubic", "cubic", "quintic"])
    most = {"batch": 8 * 128 ** 3, "adjoint": 128 ** 3, "neumann_advected": 2.6e7}.get(kind, 5e7)
    while True:
        nx, nz = rng.choice(LENGTHS), rng.choice(LENGTHS)
        ny = rng.choice([n for n in LENGTHS if n % 16 == 0])
        boxes = rng.randint(2, 12) if kind == "batch" else 1
        if 2e4 <= nx * ny * nz <= most / boxes and nz >= 32:
            break
    steps = {"periodic": 200, "neumann": 200, "batch": 100, "adjoint": 100}.get(kind, 60)
    check = {"batch": steps, "adjoint": 50}.get(kind, rng.choice([20, steps]))
    eps, dt = (-0.7, 1e-3) if model == "quintic" else (round(rng.uniform(0.2, 0.6), 3), 0.02 if "advected" in kind or prec == "f32" else 0.05)
    start = "noise" if kind != "periodic" and kind != "neumann" else rng.choice(["noise", "layers"])
    case = _case("", kind, nx, ny, nz, prec, steps, check, model, eps, dt, start, boxes=boxes, force=rng.choice(["sh", "mu"]),
                 w_mid=1.0 if kind == "periodic" and model == "quintic" and rng.random() < 0.5 else 0.0,
                 surf=kind == "neumann" and prec == "f64" and rng.random() < 0.5)
    del case["name"]
    return case


def _shapes(case):
    if case["boxes"] == 1:
        return [(case["nx"], case["ny"], case["nz"])]
    if case["nx"] == 64 and case["ny"] == 96 and case["nz"] == 128:  # the uneven cubes of the ensemble workload
        return [(n, n, n) for n in [64] * 11 + [96] * 9 + [128] * 4][:case["boxes"]]
    return [(case["nx"], case["ny"], case["nz"]) if i % 3 else (case["nx"], case["ny"], case["nx"])
            for i in range(case["boxes"])]


def _configs(case):
    quintic = case["model"] == "quintic"
    out = []
    for i, (nx, ny, nz) in enumerate(_shapes(case)):
        out.append(A.make_config(
            nx, ny, nz, nw=16 if quintic else 8, q0=1.0, dt=case["dt"],
            eps=case["eps"] + (0.2 * i / case["boxes"] if case["boxes"] > 1 else 0.0),
            beta=2.0 if quintic else 0.0, gamma=1.0, nl_model=A.SMX_NL_QUINTIC if quintic else A.SMX_NL_CUBIC,
            bc=A.SMX_BC_NEUMANN if "neumann" in case["kind"] else A.SMX_BC_PERIODIC,
            precision=A.SMX_FP64 if case["prec"] == "f64" else A.SMX_FP32_MIXED,
            advect=1 if "advected" in case["kind"] else 0,
            force_form=A.SMX_FORCE_SH if case["force"] == "sh" else A.SMX_FORCE_MU,
            w_mid=case["w_mid"], mid_plane=nz // 2 if case["w_mid"] else -1))
    return out


def _fields(case, seed):
    """Initial fields: curved layers with a little noise, or noise alone."""
    rng = np.random.default_rng(seed)
    out = []
    for shape, cfg in zip(_shapes(case), _configs(case)):
        psi = rng.uniform(-1.0, 1.0, shape)
        if case["start"] == "noise":
            psi *= 0.05
        else:
            psi *= 0.01
            x, y, z = ((np.arange(n) - n // 2 + rng.uniform(-2, 2)) * (l / n)
                       for n, l in zip(shape, (cfg.lx, cfg.ly, cfg.lz)))
            amp = 1.0 if case["model"] == "quintic" else 0.4
            r2 = np.maximum((x * x)[:, None, None] + (y * y)[None, :, None] - (z * z)[None, None, :], 0.0)
            psi += amp * np.cos(np.sqrt(r2 + 4.0))
        out.append(psi)
    return out


def prepare(case, seed):
    cfgs, fields = _configs(case), _fields(case, seed)
    state = {"case": case}
    if case["kind"] == "batch":
        b = Batch(cfgs)
        b.autotune(5)
        for box, psi in zip(b.boxes, fields):
            box.set_psi(psi)
        state["batch"] = b
        return state
    s = Solver(cfgs[0])
    s.autotune(5)
    if case["kind"] == "adjoint":
        # a workspace of the full records, kept between calls
        nx, ny, nz = s.shape
        w = 8 if case["prec"] == "f64" else 4
        segments = -(-case["steps"] // case["check"])
        s.set_adjoint_budget(segments * (w * nx * ny * nz * case["check"] + 2 * w * nx * ny * (nz // 2 + 1) * (case["check"] + 1)))
        state["psi0"] = fields[0]
    else:
        s.set_psi(fields[0])
        s.set_l1_tracking(True)
    state["solver"] = s
    if case["surf"]:
        state["surf"] = [np.zeros(s.shape[0] * s.shape[1]) for _ in range(4)]
    return state


def _as_carried(psi, case):
    psi = torch.from_numpy(psi)
    return psi if case["prec"] == "f64" else psi.to(torch.float32)


def run(state):
    case = state["case"]
    if case["kind"] == "batch":
        b = state["batch"]
        b.run(case["steps"], graph_steps=10)
        return {"psi": [_as_carried(box.get_psi(), case) for box in b.boxes]}
    s = state["solver"]
    if case["kind"] == "adjoint":
        loss, dpsi0, deps, dq0 = s.adjoint_grad(state["psi0"], case["steps"], case["check"], 0.5)
        return {"loss": loss, "dpsi0": _as_carried(dpsi0, case), "deps": deps, "dq0": dq0}
    out = {"l1": []}
    for _ in range(case["steps"] // case["check"]):
        s.step(case["check"])
        out["l1"].append(s.l1())
        if case["surf"]:
            out["surf"] = s.surftrack(0.1, -1.0, out=state["surf"])
    out["energy"] = s.energy()
    out["psi"] = _as_carried(s.get_psi(), case)
    return out


def work(case):
    """One field in, one field out; per step the state in and out of the two points where the whole field has to
    meet (the nonlinearity in real space, the update in k-space), with the transforms between them."""
    total_bytes = total_flops = 0.0
    w = 8 if case["prec"] == "f64" else 4
    for nx, ny, nz in _shapes(case):
        n = float(nx * ny * nz)
        fft = 2.5 * n * math.log2(n)
        step_bytes, step_flops = 6 * w * n, 2 * fft + 30 * n
        if "advected" in case["kind"]:
            step_bytes, step_flops = 20 * w * n, 13 * fft + 150 * n
        if case["kind"] == "adjoint":
            step_bytes, step_flops = 16 * w * n, 4 * fft + 80 * n
        total_bytes += case["steps"] * step_bytes + 2 * w * n
        total_flops += case["steps"] * step_flops
        total_bytes += 2 * w * n * (case["steps"] // case["check"])  # the two fields of each L1 test
    return {"bytes": total_bytes, "flops": total_flops}


class _Plain:
    """The same time loop in 64 bits with torch.fft.  A Neumann box is the evenly mirrored periodic one."""

    def __init__(self, cfg, psi, dev):
        self.c, self.neumann = cfg, cfg.bc == A.SMX_BC_NEUMANN
        psi = torch.as_tensor(psi, dtype=torch.float64, device=dev)
        if self.neumann:
            for ax in range(3):
                psi = torch.cat([psi, psi.flip(ax)], ax)
        self.psi, self.shape = psi, psi.shape
        d = (cfg.lx / cfg.nx, cfg.ly / cfg.ny, cfg.lz / cfg.nz)
        self.dv, self.dz = d[0] * d[1] * d[2], d[2]
        self.k = []
        for ax, n in enumerate(self.shape):
            k = 2 * math.pi * torch.fft.fftfreq(n, d=d[ax], dtype=torch.float64, device=dev)
            k[n // 2] = math.pi / d[ax]
            k = k[:n // 2 + 1] if ax == 2 else k
            self.k.append(k.reshape([-1 if a == ax else 1 for a in range(3)]))
        self.k2 = self.k[0] ** 2 + self.k[1] ** 2 + self.k[2] ** 2
        self.npast = None

    def _back(self, f):
        f = torch.fft.ifft2(f, dim=(0, 1))
        f[..., 0].imag.zero_()
        f[..., -1].imag.zero_()
        return torch.fft.irfft(f, n=self.shape[2], dim=2)

    def local(self, p):
        b, g = self.c.beta, self.c.gamma
        n = b * p * p - g * p ** 3 if self.c.nl_model == A.SMX_NL_CUBIC else b * p ** 3 - g * p ** 5
        if self.c.w_mid:
            m, n = self.c.mid_plane, n.clone()
            n[..., m] += 2 * self.c.w_mid / self.dz ** 2 * (p[..., m - 1] - 2 * p[..., m] + p[..., m + 1])
        return n

    def linear(self, eps=None, q0=None):
        c = self.c
        lin = (c.eps if eps is None else eps) - c.alpha * (self.k2 - (c.q0 if q0 is None else q0) ** 2) ** 2
        return 1 + 0.5 * c.dt * lin, 1 - 0.5 * c.dt * lin

    def advection(self, ph, p, n):
        c = self.c
        f = self._back(c.alpha * (self.k2 - c.q0 ** 2) ** 2 * ph)
        if c.force_form == A.SMX_FORCE_MU:
            f = f - c.eps * p - self.local(p)
        grad = [self._back(1j * k * ph) for k in self.k]
        s = [torch.fft.rfftn(f * g) for g in grad]
        k2 = self.k2.clone()
        k2[0, 0, 0] = 1.0
        dot = sum(k * a for k, a in zip(self.k, s)) / k2
        for k, a, g in zip(self.k, s, grad):
            u = (a - k * dot) / (c.rho * c.eta * k2)
            u[0, 0, 0] = 0
            n = n - self._back(u) * g
        if self.neumann:
            for ax in range(3):
                n = 0.5 * (n + n.flip(ax))
        return n

    def steps(self, count):
        c1, c2 = self.linear()
        for _ in range(count):
            p = self.psi
            n = self.local(p)
            if self.npast is None:
                self.npast = torch.fft.rfftn(n)
            ph = torch.fft.rfftn(p)
            if self.c.advect:
                n = self.advection(ph, p, n)
            nq = torch.fft.rfftn(n)
            self.psi = self._back((c1 * ph + 0.5 * self.c.dt * (3 * nq - self.npast)) / c2)
            self.npast, self.last = nq, p

    def l1(self):
        return float((self.psi - self.last).abs().sum() / (self.c.dt * self.psi.abs().sum()))

    def energy(self):
        c, p = self.c, self.psi
        w = torch.full_like(self.k[2], 2.0)
        w[..., 0] = w[..., -1] = 1.0
        q = torch.fft.rfftn(p)
        quad = float((w * (0.5 * c.alpha * (c.q0 ** 2 - self.k2) ** 2 - 0.5 * c.eps) * (q.real ** 2 + q.imag ** 2)).sum())
        if c.nl_model == A.SMX_NL_CUBIC:
            loc = float((-c.beta / 3 * p ** 3 + c.gamma / 4 * p ** 4).sum())
        else:
            loc = float((-c.beta / 4 * p ** 4 + c.gamma / 6 * p ** 6).sum())
        return (quad / p.numel() + loc) * self.dv / (8 if self.neumann else 1)

    def field(self):
        c = self.c
        return self.psi[:c.nx, :c.ny, :c.nz].cpu()


def _exact_gradient(case, cfg, psi, dev):
    ref = _Plain(cfg, psi, dev)
    psi0 = ref.psi.clone().requires_grad_(True)
    eps = torch.tensor(cfg.eps, dtype=torch.float64, device=dev, requires_grad=True)
    q0 = torch.tensor(cfg.q0, dtype=torch.float64, device=dev, requires_grad=True)
    c1, c2 = ref.linear(eps, q0)
    p, npast = psi0, torch.fft.rfftn(ref.local(psi0))
    for _ in range(case["steps"]):
        nq = torch.fft.rfftn(ref.local(p))
        p = torch.fft.irfftn((c1 * torch.fft.rfftn(p) + 0.5 * cfg.dt * (3 * nq - npast)) / c2, s=ref.shape)
        npast = nq
    z = torch.arange(cfg.nz, dtype=torch.float64, device=dev) * ref.dz
    loss = 0.5 * ((p - 0.5 * torch.cos(q0.detach() * z)) ** 2).sum()
    loss.backward()
    return {"loss": float(loss), "dpsi0": psi0.grad.cpu(), "deps": float(eps.grad), "dq0": None}


def exact(case, seed):
    dev = torch.device("cuda:0" if torch.cuda.is_available() else "cpu")
    cfgs, fields = _configs(case), _fields(case, seed)
    if case["kind"] == "adjoint":
        return _exact_gradient(case, cfgs[0], fields[0], dev)
    if case["kind"] == "batch":
        psi = []
        for cfg, f in zip(cfgs, fields):
            ref = _Plain(cfg, f, dev)
            ref.steps(case["steps"])
            psi.append(ref.field())
        return {"psi": psi}
    ref, out = _Plain(cfgs[0], fields[0], dev), {"l1": []}
    for _ in range(case["steps"] // case["check"]):
        ref.steps(case["check"])
        out["l1"].append(ref.l1())
        if case["surf"]:
            out["surf"] = None
    out["energy"] = ref.energy()
    out["psi"] = ref.field()
    return out
