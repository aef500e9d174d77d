"""Performance cases of the dynamical core, through the entry points a host
program calls (``dcm_amd.hip``): whole time steps on resident state, the
pressure solve, and the advection routines, over the sizes this repository's
own configurations use and odd ones between them.

``listed()`` names the cases, ``draw(rng)`` gives another one of the same
ranges, ``prepare(case, seed)`` builds what a program holds before the call
(inputs on the GPU, context, model), ``run(state)`` is one call, ``work(case)``
the bytes and operations it cannot do without, ``tolerance(case)`` how far two
correct implementations may differ, and ``exact(case, seed)`` the same call in
64-bit torch without the library.
"""
import ctypes
import math
import os
import random
import sys
import types

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "dynamical-cloud-model_amd"))  # the package
from dcm_amd import hip as H  # noqa: E402
from dcm_amd import workloads as W  # noqa: E402

DEV = "cuda"


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------
def listed():
    return [
        # the reference's shipped namelists: a y-z slice of a few thousand
        # cells, kord 3, every option of sources, FP64; all launches
        dict(name="step_slice_fp64", op="step", ip=1, jp=101, kp=120, delta=100.0, dt=2.5, nq=3,
             kord=3, ptol=1e-8, mixed=False, mg=False, physics=True, flow="shear"),
        # the reference's warm bubble on the default settings (FP64, Jacobi)
        dict(name="step_bubble_fp64", op="step", ip=64, jp=64, kp=64, delta=50.0, dt=1.0, nq=0,
             kord=2, ptol=1e-10, mixed=False, mg=False, physics=False, flow="bubble"),
        # a ragged domain with the subgrid model and the relaxation terms,
        # mixed precision with the default (Chebyshev) preconditioner
        dict(name="step_physics_mixed", op="step", ip=150, jp=91, kp=70, delta=50.0, dt=0.5, nq=3,
             kord=2, ptol=1e-10, mixed=True, mg=False, physics=True, flow="shear"),
        # a quasi-2-D shear layer, mixed precision, multigrid
        dict(name="step_layer_mixed", op="step", ip=512, jp=4, kp=256, delta=10.0, dt=0.2, nq=0,
             kord=2, ptol=1e-10, mixed=True, mg=True, physics=False, flow="layer"),
        # the moist bubble with eight tracers, the production settings
        dict(name="step_moist_mixed", op="step", ip=256, jp=256, kp=128, delta=50.0, dt=0.5, nq=9,
             kord=2, ptol=1e-10, mixed=True, mg=True, physics=False, flow="bubble"),
        # the largest domain
        dict(name="step_large_mixed", op="step", ip=512, jp=512, kp=256, delta=25.0, dt=0.25, nq=5,
             kord=2, ptol=1e-10, mixed=True, mg=True, physics=False, flow="bubble"),
        # twelve uneven domains stepped together
        dict(name="ensemble_mixed", op="ensemble", members=12, shapes=404, delta=50.0, dt=1.0,
             kord=2, ptol=1e-10, mixed=True, mg=True),
        # the pressure solve alone: the reference's FP64 BiCGSTAB, as the
        # Fortran host calls it once per step, and the mixed one
        dict(name="solve_fp64", op="solve", ip=192, jp=192, kp=96, delta=50.0, mixed=False,
             mg=False),
        dict(name="solve_mixed", op="solve", ip=128, jp=96, kp=64, delta=50.0, mixed=True, mg=True),
        # advection of one scalar and of a category of three, FP64
        dict(name="mpdata_scalar", op="mpdata", ip=256, jp=256, kp=128, nf=1, kord=2,
             monotone=True),
        dict(name="mpdata_category", op="mpdata", ip=201, jp=119, kp=77, nf=3, kord=3,
             monotone=True),
        # sedimentation of a category of three, as the microphysics calls it
        dict(name="sedimentation", op="sediment", ip=256, jp=256, kp=128, nf=3, kord=1,
             monotone=False),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _odd_part(n):
    while n % 2 == 0:
        n //= 2
    return n


def _multigrid_takes(ip, jp, kp):
    """The V-cycle halves every even dimension; it needs a coarsest level."""
    return ip * jp * kp > 2048 and _odd_part(ip) * _odd_part(jp) * _odd_part(kp) <= 512


def draw(rng):
    op = rng.choice(["step", "step", "step", "solve", "mpdata", "sediment", "ensemble"])
    if op == "ensemble":
        mixed = rng.random() < 0.7
        return dict(op=op, members=rng.randint(4, 12 if mixed else 8),
                    shapes=rng.randrange(1 << 20), delta=50.0, dt=1.0, kord=2, ptol=1e-10,
                    mixed=mixed, mg=True)
    if op == "step":
        flow = rng.choice(["bubble", "bubble", "shear", "layer"])
        mixed = rng.random() < 0.6
        if flow == "layer":
            ip, jp, kp, delta, dt = 16 * _log(rng, 8, 48), 4, 16 * rng.randint(6, 20), 10.0, 0.2
        elif rng.random() < 0.2:  # a slice
            ip, jp, kp, delta, dt = 1, _log(rng, 61, 501), rng.randint(60, 130), 100.0, 1.0
        else:
            hi = 288 if mixed else 96
            ip, jp = (_log(rng, 20, hi) for _ in range(2))
            kp, delta, dt = _log(rng, 20, 160 if mixed else 80), 50.0, 0.5
            if rng.random() < 0.6:
                ip, jp, kp = (max(16, 16 * round(n / 16)) for n in (ip, jp, kp))
        physics = flow == "shear" or rng.random() < 0.2
        nq = 0 if flow == "layer" else rng.choice([0, 1, 3, 9])
        return dict(op=op, ip=ip, jp=jp, kp=kp, delta=delta, dt=dt, nq=nq,
                    kord=rng.choice([2, 2, 3]), ptol=1e-10, mixed=mixed,
                    mg=_multigrid_takes(ip, jp, kp) and (mixed or rng.random() < 0.3),
                    physics=physics, flow=flow)
    if op == "solve":
        mixed = rng.random() < 0.6
        hi = 256 if mixed else 192
        ip, jp, kp = _log(rng, 24, hi), _log(rng, 24, hi), _log(rng, 24, 128)
        if mixed:
            ip, jp, kp = (16 * round(n / 16) for n in (ip, jp, kp))
        return dict(op=op, ip=ip, jp=jp, kp=kp, delta=50.0, mixed=mixed,
                    mg=mixed and _multigrid_takes(ip, jp, kp))
    ip, jp, kp = _log(rng, 16, 256), _log(rng, 16, 256), _log(rng, 16, 160)
    if op == "mpdata":
        return dict(op=op, ip=ip, jp=jp, kp=kp, nf=rng.choice([1, 1, 2, 3, 4]),
                    kord=rng.choice([1, 2, 2, 3]), monotone=rng.random() < 0.8)
    return dict(op=op, ip=ip, jp=jp, kp=kp, nf=rng.choice([1, 2, 3, 4]),
                kord=rng.choice([1, 1, 2, 3]), monotone=rng.random() < 0.5)


def _shapes(case):
    """Uneven member domains, as the 64-member ensemble of the benchmark."""
    rng = random.Random(case["shapes"])
    return [(rng.choice((32, 48, 64, 96, 128)), rng.choice((32, 48, 64, 96, 128)),
             rng.choice((32, 64, 96))) for _ in range(case["members"])]


def _member(case, shape):
    return dict(op="step", ip=shape[0], jp=shape[1], kp=shape[2], delta=case["delta"],
                dt=case["dt"], nq=0, kord=case["kord"], ptol=case["ptol"], mixed=case["mixed"],
                mg=case["mg"], physics=False, flow="bubble")


# ---------------------------------------------------------------------------
# domains and initial fields
# ---------------------------------------------------------------------------
def _domain(case):
    delta = case.get("delta", 50.0)
    theta = None
    if case.get("flow") == "layer":
        mid = case["kp"] * delta / 2.0

        def theta(z):
            z = np.asarray(z, dtype=np.float64)
            return 300.0 + 0.003 * z + 0.25 * (1.0 + np.tanh((z - mid) / 50.0))
    elif case.get("flow") == "shear":
        def theta(z):
            return 291.0 + 0.004 * np.asarray(z, dtype=np.float64)
    return W.make_domain(case["ip"], case["jp"], case["kp"], delta, delta, delta, theta)


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) * 7919 + 17)
    return g


def _rand(g, *shape):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float64)


def _axes(dom):
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV)
    return t(dom.xn)[:, None, None], t(dom.yn)[None, :, None], t(dom.zn)[None, None, :]


def _blob(dom, x0, y0, z0, radius):
    X, Y, Z = _axes(dom)
    r = ((X - x0) ** 2 + (Y - y0) ** 2 + (Z - z0) ** 2).sqrt_()
    return torch.where(r <= radius, torch.cos(r * (math.pi / (2.0 * radius))) ** 2, 0.0)


def _inner(a):
    return a[..., 1:-1, 1:-1, 1:-1]


def _step_fields(case, dom, seed):
    """u, v, w, th and q as the program has them before its first step."""
    g = _gen(seed)
    z = torch.zeros
    f = {n: z(dom.shape, device=DEV, dtype=torch.float64) for n in ("u", "v", "w", "th")}
    q = z((case["nq"],) + dom.shape, device=DEV, dtype=torch.float64)
    r = _rand(g, 8 + 4 * max(case["nq"], 1)).tolist()
    lx, ly, lz = (n * case["delta"] for n in (dom.ip, dom.jp, dom.kp))
    zn = torch.from_numpy(dom.zn).to(DEV)
    side = min(lx if dom.ip > 1 else ly, ly)
    if case["flow"] == "layer":
        _inner(f["u"])[:] = (10.0 + 0.5 * r[0]) * torch.tanh((zn[1:-1] - 0.5 * lz) / 50.0)
        _inner(f["w"])[:] = 1e-3 * (2.0 * _rand(g, dom.ip, dom.jp, dom.kp) - 1.0)
    else:
        rad = min(500.0, 0.35 * side, 0.35 * lz)
        x0 = 0.2 * lx * (r[0] - 0.5) if dom.ip > 1 else float(dom.xn[1])
        f["th"] += (1.0 + r[1]) * _blob(dom, x0, 0.2 * ly * (r[2] - 0.5),
                                        min(500.0, 0.4 * lz), rad)
        _inner(f["th"])[:] += 0.01 * (2.0 * _rand(g, dom.ip, dom.jp, dom.kp) - 1.0)
        # a background wind: the bubble's uniform, or sheared
        wind = 2.0 + (0.003 + 0.002 * r[3]) * zn if case["flow"] == "shear" else 2.0 + r[3]
        if dom.ip > 1:
            f["u"] += wind
        f["v"] -= 0.5 * wind
    for n in range(case["nq"]):
        a = r[8 + 4 * n:12 + 4 * n]
        if n == 0:
            _inner(q[0])[:] = 0.014 * torch.exp(-zn[1:-1] / 2000.0)
            _inner(q[0])[:] *= 1.0 + 0.01 * _rand(g, dom.ip, dom.jp, dom.kp)
        else:
            x0 = lx * (a[0] - 0.5) if dom.ip > 1 else float(dom.xn[1])
            q[n] = 0.2 + a[3] * _blob(dom, x0, ly * (a[1] - 0.5), lz * a[2],
                                      max(4.0 * case["delta"], 0.2 * side))
            _halo_zero(q[n])
    f["q"] = q
    return f


def _halo_zero(a):
    a[0], a[-1], a[:, 0], a[:, -1], a[:, :, 0], a[:, :, -1] = 0, 0, 0, 0, 0, 0


def _physics(case, dom):
    if not case["physics"]:
        return None
    prof = np.zeros((3, 3, dom.kp + 2)) + 2.0 + 0.004 * dom.zn
    return W.physics_profiles(dom, u=prof if dom.ip > 1 else 0.0 * prof, v=-0.5 * prof, z0=0.05,
                              z0th=0.01, damping_layer=True, damping_tau=300.0, forcing=True,
                              forcing_tau=600.0, divergence=True, divergence_val=2e-5,
                              divergence_hgt=0.5 * float(dom.z[dom.kp]))


# ---------------------------------------------------------------------------
# what a program holds: contexts, models, device buffers
# ---------------------------------------------------------------------------
class Buffer:
    """A torch tensor handed to the library by its device pointer."""

    def __init__(self, t):
        self.t = t.contiguous()
        self.ptr = ctypes.c_void_p(self.t.data_ptr())


class Owned:
    """Library objects, closed in order when the last user lets go of them."""

    def __init__(self, *objects, keep=None):
        self.objects, self.keep = objects, keep

    def __del__(self):
        for o in self.objects:
            o.close()


class _Memory:
    """Device memory of a model as torch imports it; a view holds the model."""

    def __init__(self, ptr, shape, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8",
                                         "data": (ptr, False), "version": 2}


class ResidentModel:
    """A model with zero-copy views of its fields."""

    def __init__(self, case, seed):
        self.case = case
        dom = self.dom = _domain(case)
        self.ctx = H.Context(dom)
        if case["mg"]:
            self.ctx.set_precond_multigrid(True)
        nq = case["nq"]
        cats = tuple(range(1, nq + 1))
        mc = W.Case("case", dom, case["dt"], 1, kord=case["kord"], monotone=True,
                    ptol=case["ptol"], nq=nq, c_s=cats, c_e=cats, physics=_physics(case, dom))
        # the fields start at zero on the GPU and are then written in place
        cfg = H.InitConfig(ip=dom.ip, jp=dom.jp, kp=dom.kp)
        zero = {n: np.zeros(dom.kp + 2) for n in ("u", "v")}
        axes = {n: np.ascontiguousarray(getattr(dom, n)) for n in ("z", "zn", "xn", "yn")}
        prof = H.InitProfiles(**{n: a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))
                                 for n, a in {**zero, **axes}.items()})
        mc.init = (types.SimpleNamespace(cfg=cfg), {"_struct": prof})
        self.model = H.Model(self.ctx, mc, H.MIXED if case["mixed"] else H.FP64)
        self.owner = Owned(self.model, self.ctx)
        self._views = {}
        f = _step_fields(case, dom, seed)
        for name, field in (("u", H.F_U), ("v", H.F_V), ("w", H.F_W), ("th", H.F_TH)):
            self.view(field).copy_(f[name])
        if nq:
            self.view(H.F_Q).copy_(f["q"])
        torch.cuda.synchronize()
        if H.load().dcm_model_init(self.model.h) != 0:
            raise RuntimeError(H.load().dcm_last_error().decode())

    def view(self, field):
        p = ctypes.c_void_p()
        if H.load().dcm_model_field(self.model.h, field, 0, ctypes.byref(p)) != 0:
            raise RuntimeError(H.load().dcm_last_error().decode())
        v = self._views.get(p.value)
        if v is None:
            shape = self.dom.shape if field != H.F_Q else (self.case["nq"],) + self.dom.shape
            v = self._views[p.value] = torch.as_tensor(_Memory(p.value, shape, self.owner),
                                                      device=DEV)
        return v

    def fields(self, previous=True):
        names = [("u", H.F_U), ("v", H.F_V), ("w", H.F_W), ("th", H.F_TH), ("p", H.F_P)]
        if previous:
            names += [("zu", H.F_ZU), ("zv", H.F_ZV), ("zw", H.F_ZW)]
        if self.case["nq"]:
            names.append(("q", H.F_Q))
        return {n: self.view(f) for n, f in names}


def _solve_fields(case, dom, seed):
    """Right-hand sides of four successive steps (divergences of smooth
    momentum sources with some noise, so of zero mean), and the pressure of
    the step before."""
    g = _gen(seed)
    out = []
    X, Y, Z = _axes(dom)
    lx, ly, lz = (n * case["delta"] for n in (dom.ip, dom.jp, dom.kp))
    a = _rand(g, 6).tolist()
    noise = [_rand(g, *dom.shape) - 0.5 for _ in range(3)]
    for n in range(4):
        ph = 2.0 * math.pi * a[0] + 0.05 * n
        s = [torch.sin(2.0 * math.pi * X / lx + ph) * torch.cos(math.pi * Z / lz) + 0.0 * Y,
             torch.cos(2.0 * math.pi * (1 + int(2 * a[1])) * Y / ly + ph) * torch.sin(
                 2.0 * math.pi * X / lx) + 0.0 * Z,
             torch.sin(math.pi * Z / lz) * torch.sin(2.0 * math.pi * (X / lx + Y / ly) + ph)]
        s = [0.02 * (f + 0.02 * e) for f, e in zip(s, noise)]
        s[2][:, :, 0] = 0
        s[2][:, :, dom.kp] = 0
        for f in s[:2]:
            f[0], f[:, 0] = f[dom.ip].clone(), f[:, dom.jp].clone()
        b = torch.zeros(dom.shape, device=DEV, dtype=torch.float64)
        b[1:-1, 1:-1, 1:-1] = ((s[0][1:-1] - s[0][:-2])[:, 1:-1, 1:-1] +
                               (s[1][:, 1:-1] - s[1][:, :-2])[1:-1, :, 1:-1] +
                               (s[2][:, :, 1:-1] - s[2][:, :, :-2])[1:-1, 1:-1, :]) / case["delta"]
        out.append(b)
    return out, torch.zeros(dom.shape, device=DEV, dtype=torch.float64)


def _advect_fields(case, dom, seed):
    """A non-divergent wind (a stream function in x-z, a wind in y that is
    constant along y), Courant numbers up to 0.3, and the category's fields."""
    g = _gen(seed)
    X, Y, Z = _axes(dom)
    a = _rand(g, 8).tolist()
    lx, ly, lz = (n * 50.0 for n in (dom.ip, dom.jp, dom.kp))
    t = lambda b: torch.from_numpy(np.ascontiguousarray(b)).to(DEV)
    x, zw = t(dom.x)[:, None], t(dom.z)[None, :]
    ra, rn = t(dom.rhoa)[None, None, :], t(dom.rhoan)[None, None, :]
    wave = 2.0 * math.pi
    psi = torch.sin(wave * (x / lx + a[0])) * torch.sin(math.pi * zw / lz)
    amp = 1.0 + 0.3 * torch.sin(wave * (Y / ly + a[1]))
    dpz = psi - torch.roll(psi, 1, 1)
    dpx = psi - torch.roll(psi, 1, 0)
    dpx[0] = dpx[dom.ip]
    u = -amp * dpz[:, None, :] / rn
    w = amp * dpx[:, None, :] / ra
    scale = 10.0 / float(max(u.abs()[1:, :, 1:-1].max(), w.abs().max()))
    u, w = u * scale + 3.0, w * scale
    v = 6.0 * torch.sin(wave * (X / lx + a[2])) * torch.cos(math.pi * Z / lz) + 0.0 * Y
    for f in (u, v, w):
        f[0], f[-1] = f[dom.ip].clone(), f[1].clone()
        f[:, 0], f[:, -1] = f[:, dom.jp].clone(), f[:, 1].clone()
        f[:, :, 0], f[:, :, -1] = 0, 0
    w[:, :, dom.kp] = 0
    q = torch.zeros((case["nf"],) + dom.shape, device=DEV, dtype=torch.float64)
    for n in range(case["nf"]):
        b = _rand(g, 4).tolist()
        q[n] = 0.3 * torch.exp(-Z / (0.5 * lz)) + b[3] * _blob(
            dom, lx * (b[0] - 0.5), ly * (b[1] - 0.5), lz * b[2], 0.3 * min(lx, ly, lz))
        _inner(q[n])[:] += 0.01 * _rand(g, dom.ip, dom.jp, dom.kp)
    return u.contiguous(), v.contiguous(), w.contiguous(), q


def _sediment_fields(case, dom, seed):
    """Fall speeds up to 8 m/s (none through the lid) and mixing ratios."""
    g = _gen(seed)
    w = torch.zeros(dom.shape, device=DEV, dtype=torch.float64)
    w[1:-1, 1:-1, :-1] = -8.0 * _rand(g, dom.ip, dom.jp, dom.kp + 1)
    w[:, :, dom.kp] = 0
    q = torch.zeros((case["nf"],) + dom.shape, device=DEV, dtype=torch.float64)
    _inner(q)[:] = 1e-3 * _rand(g, case["nf"], dom.ip, dom.jp, dom.kp)
    return w, q


def prepare(case, seed):
    if case["op"] == "step":
        m = ResidentModel(case, seed)
        return types.SimpleNamespace(case=case, model=m)
    if case["op"] == "ensemble":
        ms = [ResidentModel(_member(case, s), 1000 * seed + n)
              for n, s in enumerate(_shapes(case))]
        e = H.Ensemble([m.model for m in ms])
        return types.SimpleNamespace(case=case, models=ms, ensemble=e,
                                     owner=Owned(e, keep=[m.owner for m in ms]))
    dom = _domain(case)
    ctx = H.Context(dom)
    s = types.SimpleNamespace(case=case, dom=dom, ctx=ctx, owner=Owned(ctx))
    if case["op"] == "solve":
        if case["mg"]:
            ctx.set_precond_multigrid(True)
        b, x = _solve_fields(case, dom, seed)
        s.sw = Buffer(torch.zeros(dom.shape, device=DEV, dtype=torch.float64))
        s.b, s.x, s.n = [Buffer(a) for a in b], Buffer(x), 0
    elif case["op"] == "mpdata":
        u, v, w, q = _advect_fields(case, dom, seed)
        s.u, s.v, s.w, s.q = Buffer(u), Buffer(v), Buffer(w), Buffer(q)
    else:
        w, q = _sediment_fields(case, dom, seed)
        s.w, s.q = Buffer(w), Buffer(q)
    torch.cuda.synchronize()
    return s


def run(s):
    c = s.case
    if c["op"] == "step":
        s.model.model.step(1)
        return s.model.fields()
    if c["op"] == "ensemble":
        s.ensemble.step(1)
        return [m.fields(previous=False) for m in s.models]
    if c["op"] == "solve":
        # the next step's right-hand side, from the pressure the last one left
        b = s.b[s.n % len(s.b)]
        s.n += 1
        if c["mixed"]:
            s.ctx.bicgstab_mixed(s.sw, s.x, b, 1e-10)
        else:
            s.ctx.bicgstab(s.sw, s.x, b, 1e-10)
        return s.x.t
    if c["op"] == "mpdata":
        if c["nf"] == 1:
            s.ctx.mpdata3d(1.0, s.u, s.v, s.w, s.q, 0.0, 0.0, c["kord"], c["monotone"], 0)
        else:
            s.ctx.mpdata_vec3d(1.0, s.u, s.v, s.w, s.q, c["nf"], None, None, c["kord"],
                               c["monotone"], 0)
        return s.q.t
    s.ctx.mpdata_vec_vert3d(0.1, s.w, s.q, c["nf"], None, None, c["kord"], c["monotone"], 2)
    return s.q.t


# ---------------------------------------------------------------------------
# bytes and operations that cannot be avoided
# ---------------------------------------------------------------------------
def work(case):
    """Each input read once, each output written once (FP64 fields; a solve's
    pressure, right-hand side and result), and about 40 operations a cell for
    an operator application, 150 for MPDATA of a field and pass."""
    if case["op"] == "ensemble":
        ws = [work(_member(case, s)) for s in _shapes(case)]
        return {k: sum(w[k] for w in ws) for k in ("bytes", "flops")}
    cells = case["ip"] * case["jp"] * case["kp"]
    if case["op"] == "step":
        # u, v, w at two levels, theta, p and q: read and written
        words = 2 * (8 + case["nq"])
        return {"bytes": 8.0 * words * cells,
                "flops": cells * (200.0 + 150.0 * case["kord"] * (1 + case["nq"]))}
    if case["op"] == "solve":
        return {"bytes": 8.0 * 3 * cells, "flops": 40.0 * cells}
    if case["op"] == "mpdata":
        return {"bytes": 8.0 * (3 + 2 * case["nf"]) * cells,
                "flops": 150.0 * case["kord"] * case["nf"] * cells}
    return {"bytes": 8.0 * (1 + 2 * case["nf"]) * cells,
            "flops": 40.0 * case["kord"] * case["nf"] * cells}


def tolerance(case):
    """About four times what a change of summation order, or FP64 in place of
    the mixed path, was measured to move the outputs by."""
    if case["op"] in ("mpdata", "sediment"):
        return {"rel": 1e-13, "max": 1e-11}
    if case["mixed"]:
        # FP32 MPDATA (4e-7 after four steps); a solve's pressure 6e-8
        return {"rel": 2e-6, "max": 2e-5} if case["op"] != "solve" else {"rel": 3e-7, "max": 3e-6}
    if case["op"] == "solve":
        return {"rel": 5e-10, "max": 5e-9}
    # FP64: where BiCGSTAB stops within ptol depends on the order of its
    # sums (w of the sheared slice at ptol 1e-8 moves by 6e-6 in four steps)
    rel = 3e-7 if case.get("flow") == "shear" or case.get("ip") == 1 else 1e-8
    rel *= case["ptol"] / 1e-10
    return {"rel": rel, "max": 10.0 * rel}


# ---------------------------------------------------------------------------
# the same calls in 64-bit torch
# ---------------------------------------------------------------------------
class Grid:
    """Metrics on the GPU, shaped to multiply padded (i, j, k) arrays; m()
    is the value one index below, p() one above."""

    def __init__(self, dom):
        self.dom = dom
        self.ip, self.jp, self.kp = dom.ip, dom.jp, dom.kp
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a, dtype=np.float64)).to(DEV)
        ax = {"dx": 0, "dxn": 0, "dy": 1, "dyn": 1}
        for n in ("dx", "dy", "dz", "dxn", "dyn", "dzn", "rhoa", "rhoan", "theta", "thetan"):
            shape = [1, 1, 1]
            shape[ax.get(n, 2)] = -1
            setattr(self, n, t(getattr(dom, n)).reshape(shape))

    @staticmethod
    def m(a):
        return a.roll([1 if n > 1 else 0 for n in a.shape], [0, 1, 2])

    @staticmethod
    def p(a):
        return a.roll([-1 if n > 1 else 0 for n in a.shape], [0, 1, 2])


def _sh(a):
    """a(k+dk, j+dj, i+di) as a function of the offsets."""
    def at(dk=0, dj=0, di=0):
        if not (dk or dj or di):
            return a
        return a.roll((-di, -dj, -dk), (0, 1, 2))
    return at


def _fill(a, lbc=0.0, ubc=0.0):
    """exchange_full on one rank: periodic sides; z planes the given values
    over the interior columns, the z-wrapped interior over the side halos."""
    a[0], a[-1] = a[-2].clone(), a[1].clone()
    a[:, 0], a[:, -1] = a[:, -2].clone(), a[:, 1].clone()
    lo, hi = a[:, :, -2].clone(), a[:, :, 1].clone()
    lo[1:-1, 1:-1], hi[1:-1, 1:-1] = lbc, ubc
    a[:, :, 0], a[:, :, -1] = lo, hi
    return a


def _fill_faces(a):
    """exchange_along_dim: periodic faces, z planes zero."""
    a[0, 1:-1, 1:-1], a[-1, 1:-1, 1:-1] = a[-2, 1:-1, 1:-1].clone(), a[1, 1:-1, 1:-1].clone()
    a[1:-1, 0, 1:-1], a[1:-1, -1, 1:-1] = a[1:-1, -2, 1:-1].clone(), a[1:-1, 1, 1:-1].clone()
    a[:, :, 0], a[:, :, -1] = 0, 0
    return a


def _only_inner(new, old):
    out = old.clone()
    out[1:-1, 1:-1, 1:-1] = new[1:-1, 1:-1, 1:-1]
    return out


def _pos(x):
    return x.clamp(min=0.0)


def _neg(x):
    return x.clamp(max=0.0)


def _donor(G, dt, u, v, w, p):
    U, V, Wv, P = _sh(u), _sh(v), _sh(w), _sh(p)
    ra, rn = G.rhoa, G.rhoan
    fx = (_pos(u) * p + _neg(u) * P(0, 0, 1)) * dt / G.dxn
    fxl = (_pos(U(0, 0, -1)) * P(0, 0, -1) + _neg(U(0, 0, -1)) * p) * dt / G.dxn
    fy = (_pos(v) * p + _neg(v) * P(0, 1, 0)) * dt / G.dyn
    fyl = (_pos(V(0, -1, 0)) * P(0, -1, 0) + _neg(V(0, -1, 0)) * p) * dt / G.dyn
    fz = (_pos(w) * p + _neg(w) * P(1)) * ra * dt / (G.dzn * rn)
    fzl = (_pos(Wv(-1)) * P(-1) + _neg(Wv(-1)) * p) * G.m(ra) * dt / (G.dzn * rn)
    return p - (fx - fxl) - (fy - fyl) - (fz - fzl)


def _antidiff(G, dt, u, v, w, p):
    """The density-weighted antidiffusive velocities (mpdata_3d, kord > 1)."""
    sm = 1e-60
    U, V, Wv, P = _sh(u), _sh(v), _sh(w), _sh(p)
    ra, rn, ram, rnp = G.rhoa, G.rhoan, G.m(G.rhoa), G.p(G.rhoan)
    g3 = 0.5 * (rn + rnp)
    dxm, dym, dzm = G.m(G.dx), G.m(G.dy), G.m(G.dz)
    hx, hy, hz = (0.5 * (G.m(d) + d) for d in (G.dxn, G.dyn, G.dzn))
    fr = lambda a, b, c, d: (a + b - c - d) / (a + b + c + d + sm)
    d1 = (ra * (w + Wv(0, 0, 1)) - ram * (Wv(-1) + Wv(-1, 0, 1))) / (dzm * rn) + (
        v + V(0, 0, 1) - V(0, -1, 0) - V(0, -1, 1)) / dym
    d2 = (ra * (w + Wv(0, 1)) - ram * (Wv(-1) + Wv(-1, 1))) / (dzm * rn) + (
        u + U(0, 1) - U(0, 0, -1) - U(0, 1, -1)) / dxm
    d3 = (rn * (u - U(0, 0, -1)) + rnp * (U(1) - U(1, 0, -1))) / (dxm * g3) + (
        rn * (v - V(0, -1)) + rnp * (V(1) - V(1, -1))) / (dym * g3)
    tz1 = 0.25 * (ra * (Wv(0, 0, 1) + w) + ram * (Wv(-1, 0, 1) + Wv(-1))) / rn * fr(
        P(1, 0, 1), P(1), P(-1, 0, 1), P(-1)) / hz
    ty1 = 0.25 * (V(0, 0, 1) + v + V(0, -1, 1) + V(0, -1)) * fr(
        P(0, 1, 1), P(0, 1), P(0, -1, 1), P(0, -1)) / hy
    tz2 = 0.25 * (ra * (Wv(0, 1) + w) + ram * (Wv(-1, 1) + Wv(-1))) / rn * fr(
        P(1, 1), P(1), P(-1, 1), P(-1)) / hz
    tx2 = 0.25 * (U(0, 1) + u + U(0, 1, -1) + U(0, 0, -1)) * fr(
        P(0, 1, 1), P(0, 0, 1), P(0, 1, -1), P(0, 0, -1)) / hx
    ty3 = 0.25 * (rnp * (V(1) + V(1, -1)) + rn * (v + V(0, -1))) / g3 * fr(
        P(1, 1), P(0, 1), P(1, -1), P(0, -1)) / hy
    tx3 = 0.25 * (rnp * (U(1) + U(1, 0, -1)) + rn * (u + U(0, 0, -1))) / g3 * fr(
        P(1, 0, 1), P(0, 0, 1), P(1, 0, -1), P(0, 0, -1)) / hx
    one = lambda c, d, dn, a, s: (c.abs() * d - dt * a * c * c) * (s - p) / (s + p + sm) / dn
    us = one(u, G.dx, G.dxn, 1.0, P(0, 0, 1)) - 0.5 * dt * u * (tz1 + ty1)
    us = us - 0.25 * dt * u * ((U(0, 0, 1) - U(0, 0, -1)) / dxm + d1)
    vs = one(v, G.dy, G.dyn, 1.0, P(0, 1)) - 0.5 * dt * v * (tz2 + tx2)
    vs = vs - 0.25 * dt * v * ((V(0, 1) - V(0, -1)) / dym + d2)
    ws = one(w, G.dz, G.dzn, ra / g3, P(1)) - 0.5 * dt * w * (ty3 + tx3)
    ws = ws - 0.25 * dt * w * ((G.p(ra) * Wv(1) - ram * Wv(-1)) / (dzm * g3) + d3)
    return [_fill(_only_inner(a, torch.zeros_like(a))) for a in (us, vs, ws)]


def _betas(G, dt, u, v, w, p, old):
    sm = 1e-60
    U, V, Wv, P = _sh(u), _sh(v), _sh(w), _sh(p)
    ra, rn, ram = G.rhoa, G.rhoan, G.m(G.rhoa)
    near = [(0, 0, 0), (0, 0, -1), (0, 0, 1), (0, -1, 0), (0, 1, 0), (-1, 0, 0), (1, 0, 0)]
    mx, mn = old.clone(), old.clone()
    for f in (_sh(old), P):
        for o in near:
            mx, mn = torch.maximum(mx, f(*o)), torch.minimum(mn, f(*o))
    d1 = dt * ((_pos(U(0, 0, -1)) * P(0, 0, -1) - _neg(u) * P(0, 0, 1)) * rn / G.dxn +
               (_pos(V(0, -1)) * P(0, -1) - _neg(v) * P(0, 1)) * rn / G.dyn +
               (_pos(Wv(-1)) * ram * P(-1) - _neg(w) * ra * P(1)) / G.dzn) + sm
    d2 = dt * ((_pos(u) - _neg(U(0, 0, -1))) * rn * p / G.dxn +
               (_pos(v) - _neg(V(0, -1))) * rn * p / G.dyn +
               (_pos(w) * ra - _neg(Wv(-1)) * ram) * p / G.dzn + sm)
    zero = torch.zeros_like(p)
    return (_fill_faces(_only_inner(rn * (mx - p) / d1, zero)),
            _fill_faces(_only_inner(rn * (p - mn) / d2, zero)))


def _limit(x, up, dn, *o):
    one = torch.ones((), device=DEV, dtype=torch.float64)
    return (torch.minimum(one, torch.minimum(dn, _sh(up)(*o))) * _pos(x) +
            torch.minimum(one, torch.minimum(up, _sh(dn)(*o))) * _neg(x))


def _mpdata(G, dt, u, v, w, fields, kord, monotone, whole_min):
    """mpdata_3d / mpdata_vec_3d with zero boundary values: the fields share
    the first one's antidiffusive velocities and limiter."""
    m = [min(0.0, float((f if whole_min else _inner(f)).min())) for f in fields]
    old = [f - s for f, s in zip(fields, m)]
    cur = [_fill(_only_inner(_donor(G, dt, u, v, w, f), f), -s, -s) for f, s in zip(old, m)]
    vel = (u, v, w)
    for _ in range(1, kord):
        vel = _antidiff(G, dt, *vel, cur[0])
        if monotone:
            up, dn = _betas(G, dt, *vel, cur[0], old[0])
            z = torch.zeros_like(up)
            vel = [_fill(_only_inner(_limit(a, up, dn, *o), z))
                   for a, o in zip(vel, ((0, 0, 1), (0, 1, 0), (1, 0, 0)))]
        cur = [_fill(_only_inner(_donor(G, dt, *vel, f), f), -s, -s) for f, s in zip(cur, m)]
    return [f + s for f, s in zip(cur, m)]


def _sediment(G, dt, w, fields, kord, monotone):
    """mpdata_vec_vert_3d with outflow through the floor (neumann 2)."""
    sm = 1e-60
    ra, rn, ram, rnp = G.rhoa, G.rhoan, G.m(G.rhoa), G.p(G.rhoan)
    g3 = 0.5 * (rn + rnp)
    den = G.dzn * rn

    def zfill(a, bc):
        a[:, :, 0], a[:, :, -1] = bc, bc
        return a

    def upwind(w, p):
        wm, P = _sh(w)(-1).clone(), _sh(p)
        wm[:, :, 1] = w[:, :, 1]
        fr = (_pos(w) * p + _neg(w) * P(1)) * ra * dt / den
        fl = (_pos(wm) * P(-1) + _neg(wm) * p) * ram * dt / den
        return p - (fr - fl)

    m = [min(0.0, float(_inner(f).min())) for f in fields]
    old = [f - s for f, s in zip(fields, m)]
    cur = [zfill(_only_inner(upwind(w, f), f), -s) for f, s in zip(old, m)]
    for _ in range(1, kord):
        p, P, Wv = cur[0], _sh(cur[0]), _sh(w)
        ws = (w.abs() * G.dz - dt * (ra / g3) * w * w) * (P(1) - p) / (P(1) + p + sm) / G.dzn
        ws = ws - 0.25 * dt * w * ((G.p(ra) * Wv(1) - ram * Wv(-1)) / (G.m(G.dz) * g3))
        w = zfill(_only_inner(ws, torch.zeros_like(w)), 0.0)
        if monotone:
            O, Wv = _sh(old[0]), _sh(w)
            mx, mn = old[0], old[0]
            for a in (O(-1), O(1), P(-1), p, P(1)):
                mx, mn = torch.maximum(mx, a), torch.minimum(mn, a)
            d1 = dt * (_pos(Wv(-1)) * ram * P(-1) - _neg(w) * ra * P(1)) / G.dzn + sm
            d2 = dt * (_pos(w) * ra - _neg(Wv(-1)) * ram) * p / G.dzn + sm
            z = torch.zeros_like(p)
            up = zfill(_only_inner(rn * (mx - p) / d1, z), 0.0)
            dn = zfill(_only_inner(rn * (p - mn) / d2, z), 0.0)
            w = zfill(_only_inner(_limit(w, up, dn, 1, 0, 0), z), 0.0)
        cur = [zfill(_only_inner(upwind(w, f), f), -s) for f, s in zip(cur, m)]
    return [f + s for f, s in zip(cur, m)]


def _poisson(G, b):
    """The zero-mean solution of the 7-point Laplacian (periodic sides,
    Neumann floor and lid; uniform spacing) by FFT and the eigenvectors of
    the vertical second difference."""
    d = float(G.dx[1, 0, 0])
    n = G.kp
    T = torch.zeros(n, n, device=DEV, dtype=torch.float64)
    i = torch.arange(n - 1, device=DEV)
    T[i, i + 1] = T[i + 1, i] = 1.0
    T -= torch.diag(T.sum(1))
    lz, Q = torch.linalg.eigh(T)
    lam = lambda m: 2.0 * torch.cos(2.0 * math.pi * torch.arange(m, device=DEV,
                                                                 dtype=torch.float64) / m) - 2.0
    f = torch.fft.fft2(_inner(b) @ Q, dim=(0, 1))
    e = (lam(G.ip)[:, None, None] + lam(G.jp)[None, :, None] + lz) / (d * d)
    e[0, 0, -1] = 1.0
    f = f / e
    f[0, 0, -1] = 0.0
    p = torch.zeros_like(b)
    _inner(p)[:] = torch.fft.ifft2(f, dim=(0, 1)).real @ Q.T
    p[0], p[-1] = p[-2].clone(), p[1].clone()
    p[:, 0], p[:, -1] = p[:, -2].clone(), p[:, 1].clone()
    p[:, :, 0], p[:, :, -1] = p[:, :, 1], p[:, :, -2]
    return p


def _subgrid(G, ph, f, z, s, sth, sq):
    """calculate_subgrid_3d: viscosities, stresses, momentum and scalar
    diffusion, added to the tendencies."""
    u, v, w, th = f["u"], f["v"], f["w"], f["th"]
    U, V, Wv = _sh(u), _sh(v), _sh(w)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).reshape(1, 1, -1)
    dxm, dym, dzm = G.m(G.dx), G.m(G.dy), G.m(G.dz)
    dxnm, dynm = G.m(G.dxn), G.m(G.dyn)
    S = ((U(1) - U(1, 0, -1)) / dxm) ** 2 + ((u - U(0, 0, -1)) / dxm) ** 2
    S = S + ((V(1) - V(1, -1)) / dym) ** 2 + ((v - V(0, -1)) / dym) ** 2
    S = S + ((w - Wv(-1)) / dzm) ** 2 + ((Wv(1) - w) / G.dz) ** 2
    S = S + 0.5 * (((U(1) - u) / G.dzn + (Wv(0, 0, 1) - w) / G.dxn) ** 2 +
                   ((U(1, 0, -1) - U(0, 0, -1)) / G.dz + (w - Wv(0, 0, -1)) / dxnm) ** 2)
    S = S + 0.5 * (((w - Wv(0, -1)) / dynm + (V(1, -1) - V(0, -1)) / G.dzn) ** 2 +
                   ((Wv(0, 1) - w) / G.dyn + (V(1) - v) / G.dzn) ** 2)
    c = lambda k, di: (U(k, 0, di - 1) - U(k, -1, di - 1)) / dynm + (
        V(k, -1, di) - V(k, -1, di - 1)) / (G.dxn if di else dxnm)
    p2 = (U(0, 1, -1) - U(0, 0, -1)) / G.dyn + (v - V(0, 0, -1)) / dxnm
    p4 = (U(0, 1) - u) / G.dyn + (V(0, 0, 1) - v) / G.dxn
    p8 = (U(1, 1) - U(1)) / G.dyn + (V(1, 0, 1) - V(1)) / G.dxn
    S = S + 0.125 * (c(0, 0) ** 2 + 2.0 * p2 ** 2 + c(0, 1) ** 2 + p4 ** 2 + c(1, 0) ** 2 +
                     c(1, 1) ** 2 + p8 ** 2)
    ri = 9.81 * (_sh(th)(1) / G.p(G.thetan) - th / G.thetan) / G.dzn / (S + float(np.float32(1e-15)))
    x = (1.0 - ri / 0.25) ** 4
    a = 1.0 / 0.95
    neg, mid = ri < 0, (ri >= 0) & (ri < 0.25)
    fm = torch.where(neg, (1.0 - 16.0 * ri).clamp(min=0).sqrt(), torch.where(mid, x, 0.0))
    fh = torch.where(neg, a * (1.0 - 40.0 * ri).clamp(min=0).sqrt(),
                     torch.where(mid, a * x * (1.0 - 1.2 * ri), 0.0))
    vm = t(ph.lamsq) * S.sqrt() * fm
    vt = t(ph.lamsq) * S.sqrt() * fh * G.rhoa
    del S, ri, x, fm, fh, neg, mid, p2, p4, p8
    vm[:, :, -3:], vt[:, :, -3:] = 0, 0
    # the surface layer
    z1, z0, z0th = float(G.dom.z[1]), ph.z0, ph.z0th
    logz = math.log(z1 / z0)
    k2 = 0.4 * 0.4
    th0, thn1 = float(G.dom.theta[0]), float(G.dom.thetan[1])
    vmag = 0.5 * ((u + U(0, 0, -1)) ** 2 + (v + V(0, -1)) ** 2)[:, :, 1].sqrt() + 1e-10
    dth = th[:, :, 1] + thn1 - th0
    rib = 9.81 * dth * (z1 - z0) ** 2 / (th0 * vmag ** 2 * (z1 - z0th))
    qq = (rib * z1 / z0).abs().sqrt()
    st = 1.0 / (1.0 + 4.7 * rib) ** 2
    gm = torch.where(rib <= 0, 1.0 - 9.4 * rib / (1.0 + 70.0 * k2 * qq / logz ** 2), st)
    gh = torch.where(rib <= 0, 1.0 - 9.4 * rib / (1.0 + 50.0 * k2 * qq / logz ** 2), st)
    us = 0.4 * vmag / logz * gm.sqrt()
    ts = k2 * vmag * dth / (us * 0.95 * logz ** 2) * gh
    vm[:, :, 0] = us ** 2 * (z1 - z0) / vmag
    vt[:, :, 0] = us * ts / (dth / (z1 - z0th) + 1e-10)
    for a in (vm, vt):  # exchange_full_wo: z planes of the interior stay
        floor, lid = a[1:-1, 1:-1, 0].clone(), torch.zeros_like(a[1:-1, 1:-1, -1])
        _fill(a)
        a[1:-1, 1:-1, 0], a[1:-1, 1:-1, -1] = floor, lid
    zu, zv, zw = z
    ZU, ZV, ZW, M = _sh(zu), _sh(zv), _sh(zw), _sh(vm)
    rn, ra = G.rhoan, G.rhoa
    vv = rn * (vm + M(-1))
    s8 = sum(M(k, j, i) for k in (0, -1) for j in (0, 1) for i in (0, 1))
    zero = torch.zeros_like(u)
    tau = [vv * (zu - ZU(0, 0, -1)) / dxm, vv * (zv - ZV(0, -1)) / dym, vv * (zw - ZW(-1)) / dzm,
           rn * 0.125 * s8 * ((ZU(0, 1) - zu) / G.dyn + (ZV(0, 0, 1) - zv) / G.dxn),
           ra * 0.5 * (vm + M(0, 0, 1)) * ((ZU(1) - zu) / G.dzn + (ZW(0, 0, 1) - zw) / G.dxn),
           ra * 0.5 * (vm + M(0, 1)) * ((ZW(0, 1) - zw) / G.dyn + (ZV(1) - zv) / G.dzn)]
    t11, t22, t33, t12, t13, t23 = (_sh(_fill_faces(_only_inner(a, zero))) for a in tau)
    inc = [(t11(0, 0, 1) - t11()) / G.dxn + (t12() - t12(0, -1)) / dym + (t13() - t13(-1)) / dzm,
           (t22(0, 1) - t22()) / G.dyn + (t12() - t12(0, 0, -1)) / dxm + (t23() - t23(-1)) / dzm,
           (t33(1) - t33()) / G.dzn + (t13() - t13(0, 0, -1)) / dxm + (t23() - t23(0, -1)) / dym]
    for n, lo in ((0, 2), (1, 2), (2, 1)):
        s[n][1:-1, 1:-1, lo:G.kp] += inc[n][1:-1, 1:-1, lo:G.kp]
        _fill(s[n])
    Vt = _sh(vt)
    vd = Vt(-1)
    ax = vt + Vt(0, 0, -1) + vd + Vt(-1, 0, -1)
    bx = Vt(0, 0, 1) + vt + Vt(-1, 0, 1) + vd
    ay = vt + Vt(0, -1) + vd + Vt(-1, -1)
    by = Vt(0, 1) + vt + Vt(-1, 1) + vd
    for T, out in [(th, sth)] + [(f["q"][n], sq[n]) for n in range(len(f["q"]))]:
        Ts = _sh(T)
        d = (0.25 * (ax * (Ts(0, 0, -1) - T) / dxnm - bx * (T - Ts(0, 0, 1)) / G.dxn) / dxm +
             0.25 * (ay * (Ts(0, -1) - T) / dynm - by * (T - Ts(0, 1)) / G.dyn) / dym +
             (vd * (Ts(-1) - T) / dzm - vt * (T - Ts(1)) / G.dz) / dzm)
        _inner(out)[:] += _inner(d / rn)
        _fill(out)


def _exact_step(case, seed):
    """One pass of the time loop from the initial state."""
    dom = _domain(case)
    G = Grid(dom)
    f = _step_fields(case, dom, seed)
    for n in ("u", "v", "w", "th"):
        _fill(f[n])
    for n in range(case["nq"]):
        _fill(f["q"][n])
    u, v, w, th = f["u"], f["v"], f["w"], f["th"]
    zu, zv, zw = u.clone(), v.clone(), w.clone()
    zw[:, :, 0] = -zw[:, :, 1]
    zu[:, :, 1], zv[:, :, 1] = 0, 0
    zw[:, :, -2] = -zw[:, :, -3]
    zw[:, :, -1] = 0
    zu[:, :, -2], zv[:, :, -2] = 0, 0
    ph = _physics(case, dom)
    mean = lambda a: a[1:-1, 1:-1].mean((0, 1)).reshape(1, 1, -1)
    thbar = mean(th)
    # sources
    U, V, Wv, T = _sh(u), _sh(v), _sh(w), _sh(th)
    rn, ra = G.rhoan, G.rhoa
    two = lambda d: 2.0 * (d + G.m(d))
    su = rn * ((U(0, 0, -1) * (u + U(0, 0, -1)) - U(0, 0, 1) * (u + U(0, 0, 1))) / two(G.dx) +
               (U(0, -1) * (V(0, -1) + V(0, -1, 1)) - U(0, 1) * (v + V(0, 0, 1))) / two(G.dyn) +
               (U(-1) * (Wv(-1) + Wv(-1, 0, 1)) - U(1) * (w + Wv(0, 0, 1))) / two(G.dzn))
    sv = rn * ((V(0, 0, -1) * (U(0, 0, -1) + U(0, 1, -1)) - V(0, 0, 1) * (u + U(0, 1))) / two(G.dxn) +
               (V(0, -1) * (v + V(0, -1)) - V(0, 1) * (v + V(0, 1))) / two(G.dy) +
               (V(-1) * (Wv(-1) + Wv(-1, 1)) - V(1) * (w + Wv(0, 1))) / two(G.dzn))
    sw = ra * ((Wv(0, 0, -1) * (U(0, 0, -1) + U(1, 0, -1)) - Wv(0, 0, 1) * (u + U(1))) / two(G.dxn) +
               (Wv(0, -1) * (V(0, -1) + V(1, -1)) - Wv(0, 1) * (v + V(1))) / two(G.dyn) +
               (Wv(-1) * (w + Wv(-1)) - Wv(1) * (w + Wv(1))) / two(G.dz) +
               9.81 * (th + T(1)) / (2.0 * G.theta + thbar + G.p(thbar)))
    zero = torch.zeros_like(u)
    sth, sq = zero.clone(), torch.zeros_like(f["q"])
    s = [_only_inner(a, zero) for a in (su, sv, sw)]
    if ph is not None:
        t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(DEV).reshape(1, 1, -1)
        inc = [rn * t(ph.dampfacn) * (zu - mean(u)) - rn * (zu - t(ph.u_force)) / ph.forcing_tau,
               rn * t(ph.dampfacn) * (zv - mean(v)) - rn * (zv - t(ph.v_force)) / ph.forcing_tau,
               ra * t(ph.dampfac) * zw - rn * (mean(w) - t(ph.w_subs))]
        for a, b in zip(s, inc):
            _inner(a)[:] += _inner(b)
        _inner(sth)[:] += _inner(t(ph.dampfacn) * th)
        _subgrid(G, ph, f, (zu, zv, zw), s, sth, sq)
    su, sv, sw = (_fill(a) for a in s)
    su[:, :, 0], sv[:, :, 0], sw[:, :, 0] = -su[:, :, 1], -sv[:, :, 1], 0
    for a in (su, sv, sw):
        a[:, :, -2:] = 0
    b = ((su - _sh(su)(0, 0, -1)) / G.m(G.dx) + (sv - _sh(sv)(0, -1)) / G.m(G.dy) +
         (sw - _sh(sw)(-1)) / G.m(G.dz))
    p = _poisson(G, b)
    # advection of theta about the reference state, and of q
    dref = G.thetan - G.m(G.thetan)
    dref[0, 0, 0] = 0
    th = th.clone()
    adv = case["dt"] * (0.5 / G.m(G.dz) * Wv(-1) * G.m(ra) * dref +
                        0.5 / G.dz * w * ra * (G.p(G.thetan) - G.thetan)) / rn
    th[:, :, 1:-1] -= adv[:, :, 1:-1]
    _fill(th)
    th = _mpdata(G, case["dt"], u, v, w, [th], case["kord"], True, True)[0]
    q = f["q"]
    for n in range(case["nq"]):
        q[n] = _mpdata(G, case["dt"], u, v, w, [q[n]], case["kord"], True, False)[0]
    if ph is not None:
        th = th + sth * case["dt"]
        q = q + sq * case["dt"]
    # momentum, time filter and halos of the new level
    P, dt2 = _sh(p), 2.0 * case["dt"]
    new = [zu + (su - (P(0, 0, 1) - p) / G.dxn) * dt2 / rn,
           zv + (sv - (P(0, 1) - p) / G.dyn) * dt2 / rn,
           zw + (sw - (P(1) - p) / G.dzn) * dt2 / ra]
    prev = [0.99 * a + 0.01 * z for a, z in zip((u, v, w), (zu, zv, zw))]
    for a in new:
        _fill(a)
    new[2][:, :, 0], new[2][:, :, -1] = 0, 0
    for a in new[:2]:
        a[:, :, 0], a[:, :, -1] = -a[:, :, 1], a[:, :, -2]
    out = {"u": new[0], "v": new[1], "w": new[2], "th": th, "p": None, "zu": prev[0],
           "zv": prev[1], "zw": prev[2]}
    if case["nq"]:
        out["q"] = q
    return out


def exact(case, seed):
    # (the pressure is defined up to a constant, which the iteration chooses:
    # it has no exact value, its gradient in the new velocities has)
    if case["op"] == "step":
        return _exact_step(case, seed)
    if case["op"] == "ensemble":
        out = []
        for n, s in enumerate(_shapes(case)):
            r = _exact_step(_member(case, s), 1000 * seed + n)
            out.append({k: r[k] for k in ("u", "v", "w", "th", "p")})
        return out
    if case["op"] == "solve":
        return None
    dom = _domain(case)
    G = Grid(dom)
    if case["op"] == "mpdata":
        u, v, w, q = _advect_fields(case, dom, seed)
        return torch.stack(_mpdata(G, 1.0, u, v, w, list(q), case["kord"], case["monotone"],
                                   case["nf"] == 1))
    w, q = _sediment_fields(case, dom, seed)
    return torch.stack(_sediment(G, 0.1, w, list(q), case["kord"], case["monotone"]))
