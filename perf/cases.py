"""The work that programs built on this library have it do, as cases that can be timed.

A case is a dict of plain values.  Kinds:

* ``steps``: a lattice advanced many steps in one call, rho and u then handed over on the
  device (``Lattice.step`` and ``macro_device``); cavities, the channel past a sphere and
  periodic Taylor-Green vortices (these with the conserved sums, as the precision study reads);
* ``driver``: the time loop of an ASL flow driver, one ``execute()`` and one ``executeAll(bc)``
  per step, rho and u read on the host at the end (an output step);
* ``body``: a tunnel with a body (resting or turning) run by ``LBGKTurbulence`` in such a loop,
  the surface force and u read at the end;
* ``batch``: cavities of uneven sizes advanced together;
* ``closure``: periodic decaying turbulence with the learned closure in the collision;
* ``train``: Adam steps of the closure's network;
* ``restart``: populations written from the host, some steps, populations read back.
"""
import math

import numpy as np
import torch

import asl_amd
from asl_amd import _lib

ELEM = {"f32": 4, "f64": 8, "f16": 2, "bf16": 2}


def listed():
    return [
        # the smallest call: a driver's loop on the cavity that the smoke run uses, all launches and host work
        {"name": "driver_cavity_16", "kind": "driver", "geo": "cavity", "q": 19, "dtype": "f32", "nx": 16, "ny": 16,
         "nz": 16, "steps": 10, "tau": 0.6},
        # ASL's flow driver: a D3Q15 duct of 300 x 50 x 50, a hundred steps between two outputs
        {"name": "driver_duct_q15", "kind": "driver", "geo": "duct", "q": 15, "dtype": "f32", "nx": 300, "ny": 50,
         "nz": 50, "steps": 100, "tau": 0.55},
        # the 64^3 lid-driven cavity, in the replayed chunks of a long run
        {"name": "cavity_64", "kind": "steps", "geo": "cavity", "q": 19, "dtype": "f32", "nx": 64, "ny": 64, "nz": 64,
         "steps": 100, "tau": 0.6, "graph": True},
        # the headline workload: channel past a sphere, FP32, the benchmark's 20 steps
        {"name": "channel_f32", "kind": "steps", "geo": "channel", "q": 19, "dtype": "f32", "nx": 256, "ny": 128,
         "nz": 128, "steps": 20, "tau": 0.56, "graph": True},
        # the same with 16-bit storage, the option for larger lattices
        {"name": "channel_f16", "kind": "steps", "geo": "channel", "q": 19, "dtype": "f16", "nx": 256, "ny": 128,
         "nz": 128, "steps": 20, "tau": 0.56, "graph": True},
        # the precision study's vortex: D3Q27, periodic, the largest state here
        {"name": "vortex_q27_f32", "kind": "steps", "geo": "vortex", "q": 27, "dtype": "f32", "nx": 224, "ny": 224,
         "nz": 224, "steps": 10, "tau": 0.5005, "graph": False},
        # its FP64 reference run, at an odd and ragged size
        {"name": "vortex_q27_f64", "kind": "steps", "geo": "vortex", "q": 27, "dtype": "f64", "nx": 97, "ny": 89,
         "nz": 101, "steps": 20, "tau": 0.5005, "graph": False},
        # many small cavities of uneven sizes in one launch a step
        {"name": "batch_cavities", "kind": "batch", "q": 19, "dtype": "f32", "count": 16, "lmin": 32, "lmax": 96,
         "sizes": 1, "steps": 100, "graph": True},
        # the coarse lattice of the closure study, one chunk between two energies
        {"name": "closure_128", "kind": "closure", "nx": 128, "ny": 128, "nz": 128, "steps": 50},
        # the training of its network: the study's batch
        {"name": "closure_train", "kind": "train", "samples": 262144, "batch": 16384, "steps": 20},
        # a vehicle-like run: turbulence model, body in a tunnel, surface force on output steps
        {"name": "body_force", "kind": "body", "q": 19, "dtype": "f32", "nx": 160, "ny": 72, "nz": 60, "steps": 20,
         "tau": 0.52, "turning": False},
        # checkpoint and restart of a duct through host memory
        {"name": "restart_duct", "kind": "restart", "q": 19, "dtype": "f32", "nx": 120, "ny": 70, "nz": 66,
         "steps": 10, "tau": 0.56},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["steps", "steps", "steps", "driver", "driver", "body", "batch", "closure", "train", "restart"])
    if kind == "train":
        return {"kind": kind, "samples": _log_int(rng, 30000, 300000), "batch": _log_int(rng, 500, 20000),
                "steps": rng.randint(5, 20)}
    if kind == "closure":
        n = [rng.randint(40, 136) for _ in range(3)]
        return {"kind": kind, "nx": n[0], "ny": n[1], "nz": n[2], "steps": rng.randint(10, 50)}
    if kind == "batch":
        return {"kind": kind, "q": rng.choice([15, 19, 27]), "dtype": rng.choice(["f32", "f32", "f16"]),
                "count": rng.randint(3, 16), "lmin": rng.randint(16, 32), "lmax": rng.randint(40, 80),
                "sizes": rng.randint(2, 1 << 20), "steps": rng.randint(20, 100), "graph": rng.random() < 0.5}
    q, dtype = rng.choice([15, 19, 19, 27]), rng.choice(["f32", "f32", "f32", "f64", "f16", "bf16"])
    tau = round(rng.uniform(0.51, 0.9), 3)
    if kind == "steps":
        geo = rng.choice(["cavity", "channel", "vortex"])
        cells = math.exp(rng.uniform(math.log(2e4), math.log(2.5e6)))
        a, b = rng.uniform(0.6, 1.6), rng.uniform(0.8, 1.25)
        side = cells ** (1.0 / 3.0)
        return {"kind": kind, "geo": geo, "q": q, "dtype": dtype, "nx": max(20, int(side * a)),
                "ny": max(20, int(side * b / math.sqrt(a))), "nz": max(20, int(side / b / math.sqrt(a))),
                "steps": rng.randint(4, 40), "tau": tau, "graph": rng.random() < 0.5}
    n = {"nx": _log_int(rng, 40, 200), "ny": _log_int(rng, 30, 80), "nz": _log_int(rng, 30, 80)}
    if kind == "body":
        return dict({"kind": kind, "q": rng.choice([15, 19]), "dtype": "f32", "steps": rng.randint(5, 30),
                     "tau": round(rng.uniform(0.51, 0.6), 3), "turning": rng.random() < 0.5}, **n)
    if kind == "restart":
        return dict({"kind": kind, "q": q, "dtype": dtype, "steps": rng.randint(2, 20), "tau": tau}, **n)
    geo = rng.choice(["cavity", "duct"])
    if rng.random() < 0.5:  # the small lattices of a first look at a flow
        n = {k: max(12, v // 3) for k, v in n.items()}
    return dict({"kind": kind, "geo": geo, "q": q, "dtype": dtype, "steps": rng.randint(5, 100), "tau": tau}, **n)


# ---------------------------------------------------------------------------
# Inputs: plain torch and numpy, from the case and the seed
# ---------------------------------------------------------------------------
def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _generator(seed):
    g = torch.Generator(device=_device())
    g.manual_seed(int(seed))
    return g


def _size(case):
    return (case["nx"], case["ny"], case["nz"])


def _sphere_map(size, radius, centre):
    """Level set of a sphere on the ghost-inclusive block, clamp(d / 1.8, -1, 1)."""
    p = [(torch.arange(s + 2, device=_device(), dtype=torch.float32) - 1.0) - c for s, c in zip(size, centre)]
    d = torch.sqrt(p[0][:, None, None] ** 2 + p[1][None, :, None] ** 2 + p[2][None, None, :] ** 2) - radius
    return (d / 1.8).clamp(-1.0, 1.0)


def _noise(size, seed, amp):
    s = tuple(n + 2 for n in size)
    return (torch.rand((3,) + s, generator=_generator(seed), device=_device()) * 2.0 - 1.0) * amp


def _wrap(a):
    """The periodic ghost layer around the last three axes."""
    for d in (-3, -2, -1):
        n = a.shape[d]
        a = torch.cat([a.narrow(d, n - 1, 1), a, a.narrow(d, 0, 1)], dim=d)
    return a


def _vortex(size, seed):
    """Taylor-Green vortex of random phase with its pressure; rho, u with the ghost layer."""
    ph = torch.rand(3, generator=_generator(seed), device=_device(), dtype=torch.float64) * 2.0 * math.pi
    x = [(torch.arange(n, device=_device(), dtype=torch.float64) * (2.0 * math.pi / n) + ph[d]) for d, n in
         enumerate(size)]
    sx, cx, sy, cy = x[0].sin()[:, None, None], x[0].cos()[:, None, None], x[1].sin()[:, None], x[1].cos()[:, None]
    cz = x[2].cos()
    u0 = 0.04
    u = torch.stack([u0 * sx * cy * cz, -u0 * cx * sy * cz, torch.zeros(size, device=_device(), dtype=torch.float64)])
    c2 = [(2.0 * v).cos() for v in x]
    rho = 1.0 + 3.0 * (u0 * u0 / 16.0) * (c2[0][:, None, None] + c2[1][:, None]) * (c2[2] + 2.0)
    return _wrap(rho), _wrap(u)


def _turbulence(size, seed):
    """Random-phase solenoidal field, E(k) ~ k^4 exp(-2 (k/4)^2), u_rms 0.03."""
    k = [torch.fft.fftfreq(n, 1.0 / n, device=_device()) for n in size[:2]]
    k.append(torch.fft.rfftfreq(size[2], 1.0 / size[2], device=_device()))
    K = torch.meshgrid(*k, indexing="ij")
    k2 = K[0] ** 2 + K[1] ** 2 + K[2] ** 2
    amp = k2.sqrt() * torch.exp(-k2 / 16.0)
    w = torch.randn((3,) + tuple(size), generator=_generator(seed), device=_device())
    uh = torch.fft.rfftn(w, dim=(1, 2, 3)) * amp
    k2[0, 0, 0] = 1.0
    div = (K[0] * uh[0] + K[1] * uh[1] + K[2] * uh[2]) / k2
    u = torch.fft.irfftn(torch.stack([uh[d] - K[d] * div for d in range(3)]), s=tuple(size), dim=(1, 2, 3))
    u = u - u.mean(dim=(1, 2, 3), keepdim=True)
    u = u * (0.03 / torch.sqrt((u * u).sum(0).mean() / 3.0))
    return torch.ones(tuple(n + 2 for n in size), device=_device()), _wrap(u)


def _network(seed):
    """Parameters, input shift and scale and output scale of a closure network (the moments are about 2e-3)."""
    return _parameters(seed), np.zeros(7, np.float32), np.full(7, 500.0, np.float32), 0.002


def _parameters(seed):
    """He-style random weights W1 (32 x 7), b1, W2 (32 x 32), b2, w3, b3 with zero biases."""
    rng = np.random.default_rng(int(seed))
    w = [rng.uniform(-1.0, 1.0, n) * math.sqrt(b / fan) for n, b, fan in ((224, 6, 7), (1024, 6, 32), (32, 3, 32))]
    return np.concatenate([w[0], np.zeros(32), w[1], np.zeros(32), w[2], [0.0]]).astype(np.float32)


def _lid():
    return [("velocity", ["ZE"], {"u": (0.05, 0.0, 0.0)}), ("noslip", ["X0", "XE", "Y0", "YE", "Z0"], {})]


def _through(inlet):
    return [(inlet, ["X0"], {"u": (0.04, 0.0, 0.0), "p": 1.0}), ("pressure", ["XE"], {"p": 1.0}),
            ("noslip", ["Y0", "YE", "Z0", "ZE"], {})]


def _setting(case, seed):
    """What defines a flow: size, viscosity, rho (None: 1), u, boundary conditions in their order, map, periodicity."""
    size = _size(case)
    kind = case["kind"]
    geo = case.get("geo", {"closure": "turbulence", "body": "body", "restart": "duct"}.get(kind))
    nu = (case.get("tau", 0.5 + 0.005 / 4.0) - 0.5) / 3.0
    s = {"q": case.get("q", 19), "size": size, "nu": nu, "rho": None, "bcs": [], "map": None, "periodic": False}
    if geo == "cavity":
        s.update(u=_noise(size, seed, 1e-3), bcs=_lid())
    elif geo in ("duct", "channel", "body"):
        u = _noise(size, seed, 1e-3)
        u[0] += 0.04
        s.update(u=u, bcs=_through("velocity"))
        if geo != "duct":
            r = min(size) / 8.0 if geo == "channel" else min(size) / 6.0
            m = _sphere_map(size, r, tuple(0.25 * n if d == 0 else 0.5 * n for d, n in enumerate(size)))
            u *= (m > 0)
            turning = case.get("turning", False)
            centre = tuple(0.25 * n if d == 0 else 0.5 * n for d, n in enumerate(size))
            s.update(map=m, bcs=s["bcs"] + [("turning", None, {"omega": (0.0, 0.0, 0.02 / r), "centre": centre})
                                            if turning else ("noslip", None, {})])
    elif geo == "vortex":
        rho, u = _vortex(size, seed)
        s.update(rho=rho, u=u, periodic=True)
    else:
        rho, u = _turbulence(size, seed)
        s.update(rho=rho, u=u, periodic=True)
    host = torch.float64 if case.get("dtype") == "f64" else torch.float32
    s["u"] = s["u"].to(host)
    s["rho"] = None if s["rho"] is None else s["rho"].to(host)
    return s


def _batch_settings(case, seed):
    rng = np.random.default_rng(case["sizes"])  # sizes and viscosities belong to the case, fields to the seed
    out = []
    for i in range(case["count"]):
        n = int(round(case["lmin"] * (case["lmax"] / case["lmin"]) ** rng.random()))
        tau = float(rng.uniform(0.51, 1.0))
        out.append(_setting({"kind": "steps", "geo": "cavity", "q": case["q"], "dtype": case["dtype"], "nx": n,
                             "ny": n, "nz": n, "tau": tau}, 1000 * int(seed) + i))
    return out


def _samples(case, seed):
    """Normalised network inputs and targets."""
    g = _generator(seed)
    x = torch.randn((case["samples"], 7), generator=g, device=_device())
    t = torch.tanh(x[:, 0] - 0.5 * x[:, 3]) + 0.5 * x[:, 6] * x[:, 1] + 0.3 * torch.randn(
        case["samples"], generator=g, device=_device())
    return x, t / t.std()


# ---------------------------------------------------------------------------
# The library's side
# ---------------------------------------------------------------------------
_FACES = {"X0": _lib.X0, "XE": _lib.XE, "Y0": _lib.Y0, "YE": _lib.YE, "Z0": _lib.Z0, "ZE": _lib.ZE}
_KINDS = {"velocity": _lib.BC_CONSTANT_VELOCITY, "pressure": _lib.BC_CONSTANT_PRESSURE, "noslip": _lib.BC_NOSLIP}


def _lattice(s, dtype):
    L = asl_amd.Lattice(s["size"], s["q"], dtype=dtype, periodic=s["periodic"], nu=s["nu"])
    L.init_equilibrium(1.0 if s["rho"] is None else s["rho"].cpu().numpy(), s["u"].cpu().numpy())
    ids = []
    for kind, faces, p in s["bcs"]:
        if faces is None:
            ids.append(L.add_map_bc(_lib.BC_NOSLIP_MAP, s["map"].cpu().numpy()))
        else:
            ids.append(L.add_slice_bc(_KINDS[kind], sum(_FACES[f] for f in faces), p=p.get("p", 0.0), u=p.get("u")))
    for b in ids:
        L.execute_bc(b)
    L.finalize()
    return L, ids


def _driver(s, dtype, turbulence):
    """The objects of an ASL driver: the method and its boundary conditions, executed once before the loop."""
    block = asl_amd.Block(s["size"])
    vt = {15: asl_amd.d3q15, 19: asl_amd.d3q19, 27: asl_amd.d3q27}[s["q"]]()
    num = (asl_amd.LBGKTurbulence if turbulence else asl_amd.LBGK)(block, s["nu"], vt, dtype=dtype)
    num.init()
    asl_amd.LBGKUtilities(num).initF(s["u"].cpu().numpy())
    bcs = []
    for kind, faces, p in s["bcs"]:
        where = s["map"].cpu().numpy() if faces is None else faces
        if kind == "velocity":
            bcs.append(asl_amd.generateBCConstantVelocity(num, p["u"], where))
        elif kind == "pressure":
            bcs.append(asl_amd.generateBCConstantPressure(num, p["p"], where))
        elif kind == "turning":
            bcs.append(asl_amd.generateBCVelocity(num, None, where, rotation=tuple(p["omega"]) + tuple(p["centre"])))
        else:
            bcs.append(asl_amd.generateBCNoSlip(num, where))
    asl_amd.initAll(bcs)
    asl_amd.executeAll(bcs)
    num.lattice.finalize()
    return num, bcs


class _Field:
    """A device field of a lattice as torch takes it (it keeps the lattice)."""

    def __init__(self, lattice, address, shape):
        self.lattice = lattice
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8" if lattice.host_dtype == np.float64
                                         else "<f4", "data": (address, False), "version": 2}


def _macro(L, stream):
    """rho and u on the device, ordered on the program's stream."""
    r, u = L.macro_device(stream.cuda_stream)
    return {"rho": torch.as_tensor(_Field(L, r, L.S), device="cuda"),
            "u": torch.as_tensor(_Field(L, u, (3,) + L.S), device="cuda")}


def prepare(case, seed):
    kind = case["kind"]
    st = {"case": case, "stream": torch.cuda.Stream()}
    if kind == "train":
        x, t = _samples(case, seed)
        st["mlp"] = asl_amd.Mlp(_parameters(seed))
        st["mlp"].set_data(x.cpu().numpy(), t.cpu().numpy())
        st["seed"] = int(seed)
    elif kind == "batch":
        st["lattices"] = [_lattice(s, case["dtype"])[0] for s in _batch_settings(case, seed)]
        st["batch"] = asl_amd.Batch(st["lattices"])
    elif kind in ("driver", "body"):
        s = _setting(case, seed)
        st["num"], st["bcs"] = _driver(s, case["dtype"], kind == "body")
        if kind == "body":
            st["force"] = asl_amd.generateComputeSurfaceForce(st["num"], s["map"].cpu().numpy())
    else:
        s = _setting(case, seed)
        st["lattice"], st["ids"] = _lattice(s, case.get("dtype", "f32"))
        if kind == "closure":
            st["lattice"].set_closure(*_network(seed))
        if kind == "restart":
            st["f"] = st["lattice"].f()
    return st


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "train":
        losses = state["mlp"].train(case["steps"], case["batch"], 2e-3, state["seed"] + 1)
        return {"losses": losses.astype(np.float32), "params": state["mlp"].params()}  # FP32 sums
    if kind == "batch":
        state["batch"].step(case["steps"], graph=case["graph"])
        return [_macro(L, state["stream"]) for L in state["lattices"]]
    if kind in ("driver", "body"):
        num, bcs = state["num"], state["bcs"]
        for _ in range(case["steps"]):
            num.execute()
            asl_amd.executeAll(bcs)
        if kind == "driver":
            return {"rho": num.getRho(), "u": num.getVelocity()}
        state["force"].execute()
        return {"force": state["force"].field, "u": num.getVelocity()}
    L = state["lattice"]
    if kind == "restart":
        L.write_f(state["f"])
        for b in state["ids"]:
            L.execute_bc(b)
        L.step(case["steps"])
        return {"f": L.f(), "rho": L.rho(), "u": L.velocity()}
    L.step(case["steps"], graph=case.get("graph", False))
    out = _macro(L, state["stream"])
    if kind == "closure" or case.get("geo") == "vortex":
        out["sums"] = L.conservation()
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without
# ---------------------------------------------------------------------------
def _flops(q):
    """Moments (8 per direction), equilibrium and relaxation (10 per direction)."""
    return 18 * q


def work(case):
    """Populations in and out once a pass whatever the number of steps, rho and u out once; arithmetic of every step."""
    kind = case["kind"]
    if kind == "train":
        per = 2 * (7 * 32 + 32 * 32 + 32)  # forward; backward twice that
        return {"bytes": case["steps"] * case["batch"] * 32 + 2 * 1345 * 4, "flops": case["steps"] * case["batch"] * 3 * per}
    if kind == "batch":
        rng = np.random.default_rng(case["sizes"])
        cells = 0
        for _ in range(case["count"]):
            cells += int(round(case["lmin"] * (case["lmax"] / case["lmin"]) ** rng.random())) ** 3
            rng.uniform(0.51, 1.0)
    else:
        cells = case["nx"] * case["ny"] * case["nz"]
    q, dtype = case.get("q", 19), case.get("dtype", "f32")
    macro = 16 if dtype != "f64" else 32
    nbytes = cells * (2 * q * ELEM[dtype] + macro)
    flops = cells * case["steps"] * _flops(q)
    if kind == "closure":
        flops += cells * case["steps"] * 2 * (8 * 32 + 32 * 32 + 32)
    if kind == "body":
        nbytes += cells * 12
    if kind == "restart":
        nbytes += cells * q * macro // 2
    return {"bytes": nbytes, "flops": flops}


# ---------------------------------------------------------------------------
# The same flows in 64 bits, plain torch
# ---------------------------------------------------------------------------
def _template(q):
    if q == 15:
        e = [(a, b, c) for a in (1, -1) for b in (1, -1) for c in (1, -1)]
        return [(0, 0, 0)] + _axes() + e, [2 / 9] + [1 / 9] * 6 + [1 / 72] * 8
    edges = [(1, 1, 0), (1, -1, 0), (-1, -1, 0), (-1, 1, 0), (0, 1, 1), (0, 1, -1), (0, -1, -1), (0, -1, 1),
             (1, 0, 1), (1, 0, -1), (-1, 0, -1), (-1, 0, 1)]
    if q == 19:
        return [(0, 0, 0)] + _axes() + edges, [1 / 3] + [1 / 18] * 6 + [1 / 36] * 12
    corners = [(a, b, c) for a in (1, -1) for b in (1, -1) for c in (1, -1)]
    return [(0, 0, 0)] + _axes() + edges + corners, [8 / 27] + [2 / 27] * 6 + [1 / 54] * 12 + [1 / 216] * 8


def _axes():
    return [(1, 0, 0), (0, 1, 0), (0, 0, 1), (-1, 0, 0), (0, -1, 0), (0, 0, -1)]


def _dot(m, c):
    return sum(m[d] if c[d] > 0 else -m[d] for d in range(3) if c[d]) if any(c) else torch.zeros_like(m[0])


class _Reference:
    """Populations f_i / w_i of the interior in FP64, pulled, links replaced by the boundary conditions, relaxed."""

    def __init__(self, s, turbulence=False, network=None):
        self.s, self.c, self.w = s, *_template(s["q"])
        self.inv = [self.c.index(tuple(-x for x in v)) for v in self.c]
        self.turbulence, self.network = turbulence, network
        inner = (slice(1, -1),) * 3
        u = s["u"].double()[(slice(None),) + inner]
        rho = torch.ones(s["size"], dtype=torch.float64, device=u.device) if s["rho"] is None else s["rho"].double()[inner]
        uu = (u * u).sum(0)
        self.f = [rho * (1 + 3 * _dot(u, c) + 4.5 * _dot(u, c) ** 2 - 1.5 * uu) for c in self.c]
        self._links(u.device)

    def _links(self, dev):
        """Per direction and boundary condition, in order: the cells whose incoming population it gives."""
        s, size = self.s, self.s["size"]
        self.links = []
        m = s["map"]
        self.fluid = torch.ones(size, dtype=torch.bool, device=dev) if m is None else m[1:-1, 1:-1, 1:-1] > 0
        guard = None if m is None else (m <= 0) & (m > -0.9999)
        solved = [torch.zeros(size, dtype=torch.bool, device=dev) for _ in self.c]
        for kind, faces, p in s["bcs"]:
            for k, c in enumerate(self.c):
                if not any(c):
                    continue
                at = torch.zeros(size, dtype=torch.bool, device=dev)
                if faces is None:
                    at = self.fluid & guard[1 - c[0]:size[0] + 1 - c[0], 1 - c[1]:size[1] + 1 - c[1],
                                            1 - c[2]:size[2] + 1 - c[2]]
                else:
                    for face in faces:
                        d = "XYZ".index(face[0])
                        if c[d] == (1 if face[1] == "0" else -1):
                            at.select(d, 0 if face[1] == "0" else size[d] - 1).fill_(True)
                if bool(at.any()):
                    self.links.append((kind, k, at.nonzero(as_tuple=True), p))
                    solved[k] |= at
        # cells the library computes: the fluid, and solid cells that feed it through a link nobody gives
        self.computed = self.fluid.clone()
        if m is not None:
            while True:
                before = int(self.computed.sum())
                for k, c in enumerate(self.c):
                    if any(c):
                        self.computed |= torch.roll(self.computed & ~solved[k], [-x for x in c], (0, 1, 2))
                if int(self.computed.sum()) == before:
                    break

    def incoming(self):
        f = self.f
        new = [torch.roll(f[k], c, (0, 1, 2)) if any(c) else f[k].clone() for k, c in enumerate(self.c)]
        dens = None
        for kind, k, at, p in self.links:
            if kind == "noslip":
                new[k][at] = f[self.inv[k]][at]
            elif kind == "velocity":
                new[k][at] = f[self.inv[k]][at] + 6.0 * sum(a * b for a, b in zip(p["u"], self.c[k]))
            elif kind == "pressure":
                new[k][at] = p["p"]
            else:  # turning body: density at the ghost node from what the fluid around it sent there
                if dens is None:
                    num, den = torch.zeros_like(f[0]), torch.zeros_like(f[0])
                    for i, c in enumerate(self.c):
                        if any(c):
                            back = [-x for x in c]
                            num += self.w[i] * torch.roll(f[self.inv[i]] * self.fluid, back, (0, 1, 2))
                            den += self.w[i] * torch.roll(self.fluid.double(), back, (0, 1, 2))
                    dens = num / den
                g = [x - d for x, d in zip(at, self.c[k])]
                r = dens[g[0], g[1], g[2]]
                x = [a.double() - o for a, o in zip(g, p["centre"])]
                o = p["omega"]
                uw = (o[1] * x[2] - o[2] * x[1], o[2] * x[0] - o[0] * x[2], o[0] * x[1] - o[1] * x[0])
                new[k][at] = r + 3.0 * r * sum(a * b for a, b in zip(uw, self.c[k]))
        return new

    def step(self):
        self.f = self.incoming()
        f = self.f
        rho = sum(w * x for w, x in zip(self.w, f))
        m = torch.stack([sum(w * c[d] * x for w, c, x in zip(self.w, self.c, f) if c[d]) for d in range(3)])
        mm = 1.5 * (m * m).sum(0) / rho
        eq = []
        for c in self.c:
            a = _dot(m, c)
            eq.append(rho + 3 * a + 4.5 * a * a / rho - mm)
        omega = 1.0 / (3.0 * self.s["nu"] + 0.5)
        if self.turbulence:
            r = 4.0 * sum((x - e) ** 2 for x, e in zip(f, eq)) / sum(x * x for x in f)
            omega = torch.where(r > 1, 1.0 / (3.0 * torch.clamp(self.s["nu"] * r, max=0.5) + 0.5), omega)
        if self.network is not None:
            omega = self._relaxation(f, rho, m)
        for k in range(len(f)):
            f[k] = f[k] + omega * (eq[k] - f[k])
        self.rho, self.u = rho, m / rho

    def _relaxation(self, f, rho, m):
        p, mu, sc, out = self.network
        p = torch.tensor(p, device=rho.device).to(torch.bfloat16).double()
        x = []
        for a, b in ((0, 0), (1, 1), (2, 2), (0, 1), (0, 2), (1, 2)):
            t = sum(w * c[a] * c[b] * v for w, c, v in zip(self.w, self.c, f) if c[a] * c[b])
            x.append(t - m[a] * m[b] / rho - (rho / 3.0 if a == b else 0.0))
        x.append(rho - 1.0)
        x = torch.stack([(v - float(s0)) * float(s1) for v, s0, s1 in zip(x, mu, sc)], dim=-1)
        h = torch.relu(x @ p[:224].view(32, 7).T + p[224:256])
        h = torch.relu(h @ p[256:1280].view(32, 32).T + p[1280:1312])
        tau0 = 3.0 * self.s["nu"] + 0.5
        y = h @ p[1312:1344] + p[1344]
        return 1.0 / torch.clamp(tau0 + y * out, min=0.5 + (tau0 - 0.5) / 2.0)

    def fields(self):
        """rho and u of the whole block: cells that are not computed keep their initial values."""
        rho = torch.ones_like(self.s["u"][0], dtype=torch.float64) if self.s["rho"] is None else self.s["rho"].double().clone()
        u = self.s["u"].double().clone()
        inner = (slice(1, -1),) * 3
        rho[inner] = torch.where(self.computed, self.rho, rho[inner])
        u[(slice(None),) + inner] = torch.where(self.computed, self.u, u[(slice(None),) + inner])
        return {"rho": rho, "u": u}

    def sums(self):
        rho = sum(w * x for w, x in zip(self.w, self.f))
        m = torch.stack([sum(w * c[d] * x for w, c, x in zip(self.w, self.c, self.f) if c[d]) for d in range(3)])
        return torch.stack([rho.sum(), m[0].sum(), m[1].sum(), m[2].sum(), ((m * m).sum(0) / (2.0 * rho)).sum()]).cpu()

    def force(self):
        """Momentum exchanged over the links between solid and fluid, at both of their ends."""
        new, f, m = self.incoming(), self.f, self.s["map"]
        size = self.s["size"]
        out = torch.zeros((3,) + tuple(n + 2 for n in size), dtype=torch.float64, device=m.device)
        active = (m.abs() < 0.9999)[1:-1, 1:-1, 1:-1]
        for k, c in enumerate(self.c):
            if not any(c):
                continue
            there = self.fluid if not any(c) else torch.roll(self.fluid, [-x for x in c], (0, 1, 2))
            solid_here = active & ~self.fluid & there
            fluid_here = active & self.fluid & ~there
            for d in range(3):
                if c[d]:
                    back = [-x for x in c]
                    a = torch.roll(new[k] + f[self.inv[k]], back, (0, 1, 2)) - 2.0
                    b = 2.0 - f[k] - new[self.inv[k]]
                    out[d, 1:-1, 1:-1, 1:-1] += self.w[k] * c[d] * (torch.where(solid_here, a, 0.0) + torch.where(
                        fluid_here, b, 0.0))
        return out


def _exact_flow(s, steps, turbulence=False, network=None):
    r = _Reference(s, turbulence, network)
    for _ in range(steps):
        r.step()
    return r


def _mix(z):
    z = (z ^ (z >> np.uint64(30))) * np.uint64(0xBF58476D1CE4E5B9)
    z = (z ^ (z >> np.uint64(27))) * np.uint64(0x94D049BB133111EB)
    return z ^ (z >> np.uint64(31))


def _exact_training(case, seed):
    """Adam on the same batches (splitmix64 of the seed, the step and the sample) in FP64."""
    x, t = (v.double() for v in _samples(case, seed))
    p = torch.tensor(_parameters(seed), device=x.device).double()
    m, v, losses = torch.zeros_like(p), torch.zeros_like(p), []
    golden = np.uint64(0x9E3779B97F4A7C15)
    with np.errstate(over="ignore"):
        for s in range(case["steps"]):
            sd = _mix(np.array([int(seed) + 1], dtype=np.uint64) + golden * np.uint64(s + 1))
            pick = _mix(sd + (np.arange(case["batch"], dtype=np.uint64) + np.uint64(1)) * golden) % np.uint64(case["samples"])
            at = torch.from_numpy(pick.astype(np.int64)).to(x.device)
            q = p.clone().requires_grad_(True)
            h = torch.relu(x[at] @ q[:224].view(32, 7).T + q[224:256])
            h = torch.relu(h @ q[256:1280].view(32, 32).T + q[1280:1312])
            loss = 0.5 * ((h @ q[1312:1344] + q[1344] - t[at]) ** 2).mean()
            g, = torch.autograd.grad(loss, q)
            losses.append(loss.detach())
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            p = p - 2e-3 * (m / (1 - 0.9 ** (s + 1))) / (torch.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
    return {"losses": torch.stack(losses), "params": p}


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _exact_training(case, seed)
    if kind == "batch":
        return [_exact_flow(s, case["steps"]).fields() for s in _batch_settings(case, seed)]
    s = _setting(case, seed)
    r = _exact_flow(s, case["steps"], kind == "body", _network(seed) if kind == "closure" else None)
    out = r.fields()
    if kind == "body":
        return {"force": r.force(), "u": out["u"]}
    if kind == "restart":
        return dict(out, f=None)  # the view's ghost cells hold no defined values
    if kind == "closure" or case.get("geo") == "vortex":
        out["sums"] = r.sums()
    return out
