"""Workloads of the finite-volume path, timed through its public entry points.

A case is a dict of plain values; its ``kind`` says which program it stands for:

* ``explicit``  the explicit operator sweep (interpolate, grad, div linear and
  upwind, laplacian, snGrad) a time loop or a post-processing pass makes on one
  field.  ``order`` is the cell numbering the mesh comes in: ``block`` (the
  lexicographic order of a block mesher, stored as it is), ``zorder`` (a case
  renumbered beforehand), ``random`` (an arbitrary numbering, renumbered at
  import: every field is mapped in and every result mapped out).
* ``heat``      Euler steps of implicit heat conduction with ``dsl.solve``.
* ``poisson``   the pressure equation laplacian(1, p) = div(phi) by CG, FP64 or
  mixed precision.
* ``advection`` one implicit advection-diffusion step by BiCGStab.
* ``corrector`` the operators of one PISO corrector without its solves: momentum
  and pressure assembly, rAU, HbyA, fluxes, velocity updates.
* ``icofoam``   a whole time step of a lid-driven cavity.
* ``batch``     heat steps of many independent meshes in one batched engine.

``exact`` restates each of them in 64 bits with torch alone.
"""
from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import foamadapter_amd as fa
from foamadapter_amd import _lib, coupling, dsl, fvcc, la
from foamadapter_amd.piso import IcoFoam
from foamadapter_amd.runtime import DeviceArray

DEV = "cuda" if torch.cuda.is_available() else "cpu"
F64 = torch.float64


# ---------------------------------------------------------------------------
# the cases
# ---------------------------------------------------------------------------

def listed():
    return [
        # the smallest mesh of a test case: a sweep is launches and latency
        dict(name="sweep_small", kind="explicit", nx=16, ny=16, nz=16, order="block", prec="f64"),
        # a large case that was renumbered beforehand, in the default precision
        dict(name="sweep_large", kind="explicit", nx=192, ny=192, nz=192, order="zorder", prec="f64"),
        # the single-precision operators on a box with odd sides
        dict(name="sweep_single", kind="explicit", nx=171, ny=150, nz=133, order="zorder", prec="f32"),
        # a block mesh used as the mesher wrote it (no renumbering, the default of Mesh.from_poly)
        dict(name="sweep_block", kind="explicit", nx=97, ny=83, nz=61, order="block", prec="f64"),
        # fields that cross the boundary on a mesh renumbered at import
        dict(name="sweep_mapped", kind="explicit", nx=200, ny=150, nz=70, order="random", prec="f64"),
        # the heat transfer tutorial's loop on a small block mesh
        dict(name="heat_small", kind="heat", nx=32, ny=32, nz=32, order="block", precision="double", steps=5),
        # a pressure solve from rest, plain FP64
        dict(name="poisson_double", kind="poisson", nx=128, ny=128, nz=128, order="zorder", precision="double"),
        # the same equation with the mixed-precision option, odd sides
        dict(name="poisson_mixed", kind="poisson", nx=101, ny=96, nz=91, order="zorder", precision="mixed"),
        # a transported scalar: non-symmetric system, PBiCGStab
        dict(name="advection_step", kind="advection", nx=110, ny=100, nz=90, order="zorder", scheme="upwind"),
        # everything of a PISO corrector but the solves, at a size where bandwidth counts
        dict(name="corrector_large", kind="corrector", nx=150, ny=140, nz=130, order="zorder", scheme="linear"),
        # a whole time step of the cavity
        dict(name="icofoam_step", kind="icofoam", nx=64, ny=64, nz=64, order="zorder", scheme="upwind"),
        # a parameter study: many small systems at once
        dict(name="batch_heat", kind="batch", problems=40, lo=12, hi=64, steps=2),
    ]


def draw(rng):
    def logi(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    def box(lo, hi):
        # sides of a box of about exp(U[log lo, log hi]) cells, no side more than twice another
        n = logi(lo, hi)
        a, b = (rng.uniform(0.72, 1.4) for _ in range(2))
        e = n ** (1.0 / 3.0)
        x, y = max(3, round(e * a)), max(3, round(e * b))
        return dict(nx=x, ny=y, nz=max(3, min(int(n / (x * y)), 2 * x, 2 * y)))

    kind = rng.choice(["explicit", "explicit", "explicit", "heat", "poisson", "advection",
                       "corrector", "icofoam", "batch"])
    if kind == "explicit":
        return dict(kind=kind, **box(300, 6.5e6), order=rng.choice(["block", "zorder", "random"]),
                    prec=rng.choice(["f64", "f32"]))
    if kind == "heat":
        return dict(kind=kind, **box(300, 4e5), order=rng.choice(["block", "zorder"]),
                    precision=rng.choice(["double", "mixed"]), steps=rng.choice([2, 3, 5]))
    if kind == "poisson":
        return dict(kind=kind, **box(2000, 1.2e6), order=rng.choice(["block", "zorder"]),
                    precision=rng.choice(["double", "mixed"]))
    if kind == "advection":
        return dict(kind=kind, **box(2000, 1.2e6), order=rng.choice(["block", "zorder"]),
                    scheme=rng.choice(["upwind", "linear"]))
    if kind == "corrector":
        return dict(kind=kind, **box(2000, 2.5e6), order=rng.choice(["block", "zorder"]),
                    scheme=rng.choice(["upwind", "linear"]))
    if kind == "icofoam":
        return dict(kind=kind, **box(1000, 2.5e5), order=rng.choice(["block", "zorder"]),
                    scheme=rng.choice(["upwind", "linear"]))
    return dict(kind=kind, problems=rng.randint(6, 40), lo=rng.randint(8, 14), hi=rng.randint(20, 60),
                steps=rng.choice([1, 2, 3]))


# ---------------------------------------------------------------------------
# meshes: a jittered hexahedral block in OpenFOAM's face order, in plain torch
# ---------------------------------------------------------------------------

PATCHES = ("x0", "x1", "y0", "y1", "z0", "z1")


class Grid:
    """polyMesh primitives of an nx * ny * nz block and where its cells and faces sit."""

    def __init__(self, nx, ny, nz, order):
        n = (nx, ny, nz)
        self.n, self.N = n, nx * ny * nz
        self.h = 1.0 / max(n)
        i = torch.arange(self.N, device=DEV)
        ijk = torch.stack([i % nx, (i // nx) % ny, i // (nx * ny)], 1)
        if order == "zorder":
            key = torch.zeros(self.N, dtype=torch.int64, device=DEV)
            for b in range(max(n).bit_length()):
                for a in range(3):
                    key |= ((ijk[:, a] >> b) & 1) << (3 * b + a)
            cells = torch.argsort(key)
        elif order == "random":
            g = torch.Generator().manual_seed(self.N)
            cells = torch.randperm(self.N, generator=g).to(DEV)
        else:
            cells = i
        rank = torch.empty_like(cells)
        rank[cells] = i
        self.centre = (ijk[cells].to(F64) + 0.5) * self.h
        cid = rank.view(nz, ny, nx)
        # points, the inner ones displaced by up to a fifth of a cell
        px, py, pz = nx + 1, ny + 1, nz + 1
        p = torch.arange(px * py * pz, device=DEV)
        pijk = torch.stack([p % px, (p // px) % py, p // (px * py)], 1)
        inner = torch.ones(p.numel(), dtype=torch.bool, device=DEV)
        for a in range(3):
            inner &= (pijk[:, a] > 0) & (pijk[:, a] < n[a])
        # a fixed displacement per point, from its index
        shake = torch.stack([torch.frac(torch.sin((p + 1).to(F64) * (12.9898 + 7.1 * a)) * 43758.5453)
                             for a in range(3)], 1)
        self.points = (pijk.to(F64) + 0.2 * shake * inner[:, None]) * self.h
        pid = p.view(pz, py, px)
        own, nbr, quad, mid, area, sign = [], [], [], [], [], []
        sides = []
        for a in range(3):
            d = 2 - a  # tensor dimension of axis a
            # the four points of the face on the + side of a cell, turning about +axis
            lay = pid.narrow(d, 1, n[a])
            q = self._corners(lay, d)
            lo, hi = cid.narrow(d, 0, n[a] - 1), cid.narrow(d, 1, n[a] - 1)
            qi = q.narrow(d, 0, n[a] - 1).reshape(-1, 4)
            lo, hi = lo.reshape(-1), hi.reshape(-1)
            up = lo < hi
            own.append(torch.minimum(lo, hi))
            nbr.append(torch.maximum(lo, hi))
            quad.append(torch.where(up[:, None], qi, qi.flip(1)))
            e = torch.zeros(3, dtype=F64, device=DEV)
            e[a] = 0.5 * self.h
            mid.append(self.centre[lo] + e)
            s = torch.where(up, 1.0, -1.0).to(F64)
            sign.append(s)
            area.append(torch.full_like(s, a))
            first = self._corners(pid.narrow(d, 0, n[a]), d).narrow(d, 0, 1)
            sides.append((cid.narrow(d, 0, 1).reshape(-1), first.reshape(-1, 4).flip(1), -e, a, -1.0))
            sides.append((cid.narrow(d, n[a] - 1, 1).reshape(-1),
                          q.narrow(d, n[a] - 1, 1).reshape(-1, 4), e, a, 1.0))
        own, nbr, quad, mid, axis, sign = (torch.cat(x) for x in (own, nbr, quad, mid, area, sign))
        o = torch.argsort(own * self.N + nbr)
        own, nbr, quad, mid, axis, sign = (x[o] for x in (own, nbr, quad, mid, axis, sign))
        self.F, self.B = own.numel(), sum(s[0].numel() for s in sides)
        start, self.patches, self.patch_of = self.F, [], []
        for k, (c, q, e, a, s) in enumerate(sides):
            self.patches.append(fa.mesh.Patch(PATCHES[k], "wall", start, c.numel()))
            self.patch_of.append(torch.full((c.numel(),), k, device=DEV))
            start += c.numel()
            own, quad = torch.cat([own, c]), torch.cat([quad, q])
            mid = torch.cat([mid, self.centre[c] + e])
            axis = torch.cat([axis, torch.full((c.numel(),), a, dtype=F64, device=DEV)])
            sign = torch.cat([sign, torch.full((c.numel(),), s, dtype=F64, device=DEV)])
        self.patch_of = torch.cat(self.patch_of)
        # internal faces, then boundary faces: cells, points, place, direction
        self.own, self.nbr, self.quad = own, nbr, quad
        self.mid, self.axis, self.sign = mid, axis.long(), sign
        self.fc = own[self.F:]

    @staticmethod
    def _corners(lay, d):
        """[..., 4] corner points of the faces normal to tensor dimension d."""
        u, v = {2: (1, 0), 1: (0, 2), 0: (2, 1)}[d]  # the tensor dimensions that span them
        nu, nv = lay.shape[u] - 1, lay.shape[v] - 1

        def at(a, b):
            return lay.narrow(u, a, nu).narrow(v, b, nv)
        return torch.stack([at(0, 0), at(1, 0), at(1, 1), at(0, 1)], -1)

    def poly(self):
        i32 = lambda t: t.to(torch.int32).cpu().numpy()  # noqa: E731
        nF = self.own.numel()
        return fa.PolyMesh(self.points.cpu().numpy(), np.arange(0, 4 * nF + 1, 4, dtype=np.int32),
                           i32(self.quad.reshape(-1)), i32(self.own), i32(self.nbr), self.patches)

    def geometry(self):
        """OpenFOAM's mesh geometry (primitiveMesh, surfaceInterpolation)."""
        own, nbr, F = self.own, self.nbr, self.F
        p = [self.points[self.quad[:, k]] for k in range(4)]
        est = (p[0] + p[1] + p[2] + p[3]) / 4
        sumN, sumA, sumAc = torch.zeros_like(est), 0.0, torch.zeros_like(est)
        for k in range(4):
            a, b = p[k], p[(k + 1) % 4]
            nn = torch.linalg.cross(b - a, est - a)
            m = nn.norm(dim=1, keepdim=True)
            sumN, sumA, sumAc = sumN + nn, sumA + m, sumAc + m * (a + b + est)
        Cf, Sf = sumAc / (3 * sumA), 0.5 * sumN
        cnt = torch.zeros(self.N, dtype=F64, device=DEV).index_add_(0, own, torch.ones_like(Cf[:, 0]))
        cnt.index_add_(0, nbr, torch.ones_like(Cf[:F, 0]))
        ce = torch.zeros(self.N, 3, dtype=F64, device=DEV).index_add_(0, own, Cf).index_add_(0, nbr, Cf[:F])
        ce = ce / cnt[:, None]
        po = (Sf * (Cf - ce[own])).sum(1)
        pn = (Sf[:F] * (ce[nbr] - Cf[:F])).sum(1)
        vol = torch.zeros(self.N, dtype=F64, device=DEV).index_add_(0, own, po).index_add_(0, nbr, pn)
        cc = torch.zeros_like(ce).index_add_(0, own, po[:, None] * (0.75 * Cf + 0.25 * ce[own]))
        cc.index_add_(0, nbr, pn[:, None] * (0.75 * Cf[:F] + 0.25 * ce[nbr]))
        C = cc / vol[:, None]
        g = dict(V=vol / 3, C=C, Sf=Sf[:F], Sfb=Sf[F:], magSf=Sf[:F].norm(dim=1), magSfb=Sf[F:].norm(dim=1))
        so = (Sf[:F] * (Cf[:F] - C[own[:F]])).sum(1).abs()
        sn = (Sf[:F] * (C[nbr] - Cf[:F])).sum(1).abs()
        d = C[nbr] - C[own[:F]]
        g["w"] = sn / (so + sn)
        g["nodc"] = 1 / torch.maximum((Sf[:F] * d).sum(1) / g["magSf"], 0.05 * d.norm(dim=1))
        nf = Sf[F:] / g["magSfb"][:, None]
        g["dcb"] = 1 / (nf * (Cf[F:] - C[self.fc])).sum(1).abs()
        return g


_kept = {}  # the mesh last used: a program makes many passes on one mesh


def _grid(case, n=None):
    key = ("grid", n, case["order"]) if n else ("grid", case["nx"], case["ny"], case["nz"], case["order"])
    if key not in _kept:
        if not n:
            _drop()
        _kept[key] = Grid(n, n, n, case["order"]) if n else Grid(*key[1:])
    return _kept[key]


def _drop():
    for k in [k for k in _kept if k != "ctx"]:
        v = _kept.pop(k)
        if isinstance(v, fa.Mesh):
            v.close()


def _ctx():
    if "ctx" not in _kept:
        _kept["ctx"] = fa.Context()
    return _kept["ctx"]


def _mesh(case, n=None):
    grid = _grid(case, n)
    key = ("mesh", n)
    if key not in _kept:
        _kept[key] = fa.Mesh.from_poly(_ctx(), grid.poly(), renumber=case["order"] == "random")
    return grid, _kept[key]


# ---------------------------------------------------------------------------
# fields: smooth modes with a little noise, from the seed
# ---------------------------------------------------------------------------

def _smooth(gen, x, lo, hi, noise=0.05):
    """Values in about [lo, hi] at the places x: three waves and noise."""
    out = torch.zeros(x.shape[0], dtype=F64, device=DEV)
    par = torch.rand(3, 5, generator=gen, dtype=F64)
    for a, kx, ky, kz, ph in par.tolist():
        out += (0.3 + a) * torch.cos(6.0 * (kx * x[:, 0] + ky * x[:, 1] + kz * x[:, 2]) + 6.28 * ph)
    rough = torch.Generator(device=DEV).manual_seed(int(torch.randint(1 << 30, (1,), generator=gen)))
    out += noise * (2 * torch.rand(x.shape[0], generator=rough, dtype=F64, device=DEV) - 1)
    return lo + (hi - lo) * (0.5 + out / 6.0)


def _velocity(x, amp):
    """A divergence-free recirculation with amplitude and phase from the seed."""
    a, ph = amp
    s, c = torch.sin(math.pi * x[:, 0] + ph), torch.cos(math.pi * x[:, 0] + ph)
    return a * torch.stack([s * torch.cos(math.pi * x[:, 1]), -c * torch.sin(math.pi * x[:, 1]),
                            0.3 * torch.sin(2 * math.pi * x[:, 0]) * torch.cos(math.pi * x[:, 1])], 1)


def _fields(case, seed, grid):
    """The inputs of a case in the caller's numbering, 64 bits (32 where the case says so)."""
    gen = torch.Generator().manual_seed(int(seed) * 7919 + 17)
    kind, F = case["kind"], grid.F
    fcell = grid.own[F:]
    amp = (0.5 + float(torch.rand(1, generator=gen)), float(torch.rand(1, generator=gen)))
    vel = _velocity(grid.mid, amp)
    phi = grid.sign * grid.h ** 2 * vel.gather(1, grid.axis[:, None])[:, 0]
    f = {"phi": phi}
    if kind == "explicit":
        f["T"] = _smooth(gen, grid.centre, 280.0, 320.0)
        f["Tb"] = _smooth(gen, grid.mid[F:], 280.0, 320.0)
        f["Tg"] = _smooth(gen, grid.mid[F:], -40.0, 40.0)
        f["gamma"] = _smooth(gen, grid.mid, 0.5, 2.0)
        if case["prec"] == "f32":
            f = {k: v.float() for k, v in f.items()}
    elif kind == "heat":
        f["T"] = _smooth(gen, grid.centre, 300.0, 400.0, 0.5)
        wall = 300.0 + 100.0 * torch.rand(6, generator=gen, dtype=F64).to(DEV)
        f["Tb"] = wall[grid.patch_of]
        f["gamma"] = torch.full((F + grid.B,), 1e-2, dtype=F64, device=DEV)
    elif kind == "advection":
        f["T"] = _smooth(gen, grid.centre, 0.0, 1.0)
        f["Tb"] = _smooth(gen, grid.mid[F:], 0.0, 1.0)
        f["gamma"] = torch.full((F + grid.B,), 1e-3, dtype=F64, device=DEV)
    elif kind == "poisson":
        # the flux of an unprojected predictor: its divergence varies from cell to cell
        rough = torch.Generator(device=DEV).manual_seed(int(torch.randint(1 << 30, (1,), generator=gen)))
        f["phi"] = grid.h ** 2 * (2 * torch.rand(F + grid.B, generator=rough, dtype=F64, device=DEV) - 1)
        f["gamma"] = torch.ones(F + grid.B, dtype=F64, device=DEV)
    elif kind in ("corrector", "icofoam"):
        f["phi"][F:] = 0.0
        f["U"] = torch.stack([_smooth(gen, grid.centre, -0.3, 0.3, 0.02) for _ in range(3)], 1)
        f["Ub"] = torch.zeros(grid.B, 3, dtype=F64, device=DEV)
        f["Ub"][grid.patch_of == 3, 0] = 1.0  # the moving lid
        f["p"] = _smooth(gen, grid.centre, -0.1, 0.1)
        f["pb"] = f["p"][fcell]
        f["gamma"] = torch.full((F + grid.B,), 1e-2, dtype=F64, device=DEV)
    return f


SOLVER_U = {"solver": "PBiCGStab", "tolerance": 1e-5, "relTol": 0.0}
SOLVER_P = {"solver": "PCG", "tolerance": 1e-6, "relTol": 0.05}
HEAT_DT, ADV_DT = 1e-3, 0.02
EXPLICIT_BCS = ["fixedValue", "fixedGradient", "fixedValue", "fixedValue", "fixedGradient", "fixedValue"]


def _members(case, seed):
    """The batch's problems: edge, diffusivity and input seed of each."""
    gen = torch.Generator().manual_seed(977)  # the meshes are the case's, the fields the seed's
    u = torch.rand(case["problems"], 2, generator=gen, dtype=F64).tolist()
    la_, lb = math.log(case["lo"]), math.log(case["hi"])
    return [(round(math.exp(la_ + a * (lb - la_))), 10.0 ** (-4 + 3 * b), 1000 * int(seed) + k)
            for k, (a, b) in enumerate(u)]


def _member_fields(n, kappa, seed, grid):
    f = _fields({"kind": "heat"}, seed, grid)
    f["gamma"] = f["gamma"] * (kappa / 1e-2)
    return f


# ---------------------------------------------------------------------------
# prepare and run
# ---------------------------------------------------------------------------

class Held(DeviceArray):
    """A torch tensor as the framework's device array (the tensor owns the memory)."""

    def __init__(self, ctx, t):
        self.t = t.contiguous()
        self.ctx, self.shape = ctx, tuple(t.shape)
        self.dtype = np.dtype({torch.float32: np.float32, F64: np.float64}[t.dtype])
        self.nbytes = t.numel() * t.element_size()
        self._ptr = ctypes.c_void_p(self.t.data_ptr())

    def close(self):
        self._ptr = ctypes.c_void_p()


class _Shown:
    """A device array of the framework as torch can see it."""

    def __init__(self, a):
        self.a = a
        self.__cuda_array_interface__ = dict(shape=a.shape, typestr=a.dtype.str, version=2,
                                             data=(a.ptr.value, False), strides=None)


def _tensor(a):
    return a.t if isinstance(a, Held) else torch.as_tensor(_Shown(a), device=DEV)


def _copy(ctx, dst, src):
    _lib.call("fv_memcpy_d2d", ctx.handle, dst.ptr, src.ptr, dst.nbytes)


def prepare(case, seed):
    s = _PREPARE[case["kind"]](case, seed)
    if DEV == "cuda":
        torch.cuda.synchronize()
    return s


def run(state):
    return state["run"](state)


def _space(ctx, *shape, dtype=F64):
    return Held(ctx, torch.empty(shape, dtype=dtype, device=DEV))


def _prepare_explicit(case, seed):
    grid, m = _mesh(case)
    ctx, N, nFB = _ctx(), grid.N, grid.F + grid.B
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    dt = f["T"].t.dtype
    return dict(run=_run_explicit, ctx=ctx, mesh=m, f=f, mapped=case["order"] == "random",
                bc=fa.BoundaryConditions(m, EXPLICIT_BCS),
                out=dict(interp=_space(ctx, nFB, dtype=dt), grad=_space(ctx, N, 3, dtype=dt),
                         div=_space(ctx, N, dtype=dt), upwind=_space(ctx, N, dtype=dt),
                         lap=_space(ctx, N, dtype=dt), sngrad=_space(ctx, nFB, dtype=dt)),
                ops=(fvcc.SurfaceInterpolation(ctx, m, ["linear"]), fvcc.GaussGreenGrad(ctx, m),
                     fvcc.GaussGreenDiv(ctx, m, ["Gauss", "linear"]),
                     fvcc.GaussGreenDiv(ctx, m, ["Gauss", "upwind"]),
                     fvcc.GaussGreenLaplacian(ctx, m, ["Gauss", "linear", "uncorrected"]),
                     fvcc.FaceNormalGradient(ctx, m, ["uncorrected"])))


def _run_explicit(s):
    m, f, o = s["mesh"], s["f"], s["out"]
    T, phi, gamma = f["T"], f["phi"], f["gamma"]
    if s["mapped"]:
        T, gamma = m.to_device(T, "cell"), m.to_device(gamma, "face")
        phi = m.to_device(phi, "face", oriented=True)
    T = fvcc.VolumeField(m, T, f["Tb"], s["bc"], "T", f["Tg"])
    phi, gamma = fvcc.SurfaceField(m, phi), fvcc.SurfaceField(m, gamma)
    lin, grd, dl, du, lap, sng = s["ops"]
    lin.interpolate(T, fvcc.SurfaceField(m, o["interp"]))
    grd.grad(T, 1.0, o["grad"])
    dl.div(o["div"], phi, T, 1.0)
    du.div(o["upwind"], phi, T, 1.0)
    lap.laplacian(o["lap"], gamma, T, 1.0)
    sng.faceNormalGrad(T, fvcc.SurfaceField(m, o["sngrad"]))
    if s["mapped"]:
        o = dict(interp=m.to_caller(o["interp"], "face"), grad=m.to_caller(o["grad"], "cell"),
                 div=m.to_caller(o["div"], "cell"), upwind=m.to_caller(o["upwind"], "cell"),
                 lap=m.to_caller(o["lap"], "cell"),
                 sngrad=m.to_caller(o["sngrad"], "face", oriented=True))
    return {k: _tensor(v) for k, v in o.items()}


def _prepare_heat(case, seed):
    grid, m = _mesh(case)
    ctx = _ctx()
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    T = fvcc.VolumeField(m, _space(ctx, grid.N), f["Tb"], fa.BoundaryConditions(m, ["fixedValue"] * 6), "T")
    T.old_time = fvcc.VolumeField(m, _space(ctx, grid.N), None)
    return dict(run=_run_heat, ctx=ctx, T0=f["T"], T=T, steps=case["steps"],
                eqn=dsl.imp.ddt(T) - dsl.imp.laplacian(fvcc.SurfaceField(m, f["gamma"]), T),
                solver={"relTol": 1e-10, "maxIter": 1000, "precision": case["precision"]})


def _run_heat(s):
    T = s["T"]
    _copy(s["ctx"], T.internal, s["T0"])
    _copy(s["ctx"], T.old_time.internal, s["T0"])
    for k in range(s["steps"]):
        dsl.solve(s["eqn"], T, k * HEAT_DT, HEAT_DT, solver=s["solver"])
    return T.internal.t


def _prepare_poisson(case, seed):
    grid, m = _mesh(case)
    ctx = _ctx()
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    p = fvcc.VolumeField(m, _space(ctx, grid.N), Held(ctx, torch.zeros(grid.B, dtype=F64, device=DEV)),
                         fa.BoundaryConditions(m, ["fixedValue"] + ["zeroGradient"] * 5), "p")
    eqn = (dsl.imp.laplacian(fvcc.SurfaceField(m, f["gamma"]), p)
           - dsl.exp.div(fvcc.SurfaceField(m, f["phi"])))
    return dict(run=_run_poisson, p=p, eqn=eqn, keep=f,
                solver={"relTol": 1e-8, "maxIter": 20000, "precision": case["precision"], "checkEvery": 64})


def _run_poisson(s):
    p = s["p"]
    p.internal.fill(0.0)
    dsl.solve(s["eqn"], p, 0.0, 1.0, solver=s["solver"])
    return {"p": p.internal.t, "pb": p.boundary.t}


def _prepare_advection(case, seed):
    grid, m = _mesh(case)
    ctx = _ctx()
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    T = fvcc.VolumeField(m, _space(ctx, grid.N), f["Tb"], fa.BoundaryConditions(m, ["fixedValue"] * 6), "T")
    T.old_time = fvcc.VolumeField(m, _space(ctx, grid.N), None)
    eqn = (dsl.imp.ddt(T) + dsl.imp.div(fvcc.SurfaceField(m, f["phi"]), T, case["scheme"])
           - dsl.imp.laplacian(fvcc.SurfaceField(m, f["gamma"]), T))
    return dict(run=_run_advection, ctx=ctx, T0=f["T"], T=T, eqn=eqn,
                solver={"solver": "PBiCGStab", "relTol": 1e-10, "maxIter": 1000})


def _run_advection(s):
    T = s["T"]
    _copy(s["ctx"], T.internal, s["T0"])
    _copy(s["ctx"], T.old_time.internal, s["T0"])
    dsl.solve(s["eqn"], T, 0.0, ADV_DT, solver=s["solver"])
    return T.internal.t


def _prepare_corrector(case, seed):
    grid, m = _mesh(case)
    ctx, N, nFB = _ctx(), grid.N, grid.F + grid.B
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    ubc, pbc = fa.BoundaryConditions(m, ["fixedValue"] * 6), fa.BoundaryConditions(m, ["zeroGradient"] * 6)
    U = fvcc.VolumeField(m, f["U"], f["Ub"], ubc, "U")
    U.old_time = fvcc.VolumeField(m, f["U"], None)
    p = fvcc.VolumeField(m, f["p"], f["pb"], pbc, "p")
    nu, phi = fvcc.SurfaceField(m, f["gamma"]), fvcc.SurfaceField(m, f["phi"])
    rAUf, phiH = fvcc.SurfaceField(m, _space(ctx, nFB)), fvcc.SurfaceField(m, _space(ctx, nFB))
    dt = 0.5 * grid.h
    return dict(run=_run_corrector, U=U, p=p, rAUf=rAUf, phiH=phiH,
                UEqn=dsl.PDESolver(dsl.imp.ddt(U) + dsl.imp.div(phi, U, case["scheme"])
                                   - dsl.imp.laplacian(nu, U), U, 0.0, dt),
                pEqn=dsl.PDESolver(dsl.imp.laplacian(rAUf, p) - dsl.exp.div(phiH), p, 0.0, dt),
                lin=fvcc.SurfaceInterpolation(ctx, m, ["linear"]), res=_space(ctx, N),
                phiN=fvcc.SurfaceField(m, _space(ctx, nFB)),
                UN=fvcc.VolumeField(m, _space(ctx, N, 3), f["Ub"], ubc, "U"))


def _run_corrector(s):
    U, p, rAUf, phiH = s["U"], s["p"], s["rAUf"], s["phiH"]
    uls = s["UEqn"].assemble()
    rAU, HbyA = coupling.computeRAUandHByA(uls, uls.rhs3, U)
    coupling.constrainHbyA(U, p, HbyA)
    s["lin"].interpolate(rAU, rAUf)
    coupling.flux(HbyA, out=phiH)
    pls = s["pEqn"].assemble()
    pls.residual(p.internal, s["res"])
    coupling.updateFaceVelocity(phiH, pls, p, s["phiN"])
    coupling.updateVelocity(HbyA, rAU, p, s["UN"])
    return {"rAUf": rAUf.values.t, "phiHbyA": phiH.values.t, "residual": s["res"].t,
            "phi": s["phiN"].values.t, "U": s["UN"].internal.t}


def _prepare_icofoam(case, seed):
    grid, m = _mesh(case)
    ctx = _ctx()
    f = {k: Held(ctx, v) for k, v in _fields(case, seed, grid).items()}
    hold = {k: Held(ctx, f[k].t.clone()) for k in ("U", "p", "pb", "phi")}
    U = fvcc.VolumeField(m, hold["U"], f["Ub"], fa.BoundaryConditions(m, ["fixedValue"] * 6), "U")
    p = fvcc.VolumeField(m, hold["p"], hold["pb"], fa.BoundaryConditions(m, ["zeroGradient"] * 6), "p")
    sol = IcoFoam(U, p, fvcc.SurfaceField(m, hold["phi"]), fvcc.SurfaceField(m, f["gamma"]), 0.5 * grid.h,
                  fvSchemes={"div": "Gauss " + case["scheme"]},
                  fvSolution={"U": SOLVER_U, "p": SOLVER_P,
                              "PISO": {"nCorrectors": 2, "pRefCell": 0, "pRefValue": 0}})
    return dict(run=_run_icofoam, ctx=ctx, sol=sol, f=f, hold=hold)


def _run_icofoam(s):
    for k, v in s["hold"].items():
        _copy(s["ctx"], v, s["f"][k])
    rep = s["sol"].step()
    return {"U": s["hold"]["U"].t, "p": s["hold"]["p"].t, "phi": s["hold"]["phi"].t, "coNum": rep.coNum}


def _prepare_batch(case, seed):
    ctx, probs = _ctx(), []
    if _kept.get("batch") != (case["problems"], case["lo"], case["hi"]):
        _drop()
        _kept["batch"] = (case["problems"], case["lo"], case["hi"])
    batch = la.Batch(ctx, "mixed", tile_rows=4096, chunk=16)
    for n, kappa, sd in _members(case, seed):
        grid, m = _mesh({"order": "block"}, n)
        f = {k: Held(ctx, v) for k, v in _member_fields(n, kappa, sd, grid).items()}
        ls = la.LinearSystem(la.SparsityPattern.readOrCreate(m))
        x, xo = _space(ctx, grid.N), _space(ctx, grid.N)
        batch.add(ls, x, xo)
        probs.append((ls, xo, HEAT_DT, f["gamma"], fa.BoundaryConditions(m, ["fixedValue"] * 6),
                      f["Tb"], None, x, f["T"]))
    heat = la.HeatAssembly([p[:7] for p in probs])
    return dict(run=_run_batch, ctx=ctx, batch=batch, heat=heat, probs=probs, steps=case["steps"],
                solver={"relTol": 1e-8, "maxIter": 5000})


def _run_batch(s):
    for p in s["probs"]:
        _copy(s["ctx"], p[7], p[8])
        _copy(s["ctx"], p[1], p[8])
    for _ in range(s["steps"]):
        s["heat"].assemble(-1.0)
        s["batch"].solve(s["solver"])
    return [p[7].t for p in s["probs"]]


_PREPARE = {"explicit": _prepare_explicit, "heat": _prepare_heat, "poisson": _prepare_poisson,
            "advection": _prepare_advection, "corrector": _prepare_corrector,
            "icofoam": _prepare_icofoam, "batch": _prepare_batch}


# ---------------------------------------------------------------------------
# the least a pass moves and computes
# ---------------------------------------------------------------------------

def _sizes(c):
    nx, ny, nz = c["nx"], c["ny"], c["nz"]
    return (nx * ny * nz, (nx - 1) * ny * nz + nx * (ny - 1) * nz + nx * ny * (nz - 1),
            2 * (nx * ny + ny * nz + nx * nz))


def _sweep_bytes(N, F, B, e):
    """interpolate, grad, div linear, div upwind, laplacian, snGrad: e bytes a value, int32 indices."""
    face = (2 * e + 8) + (4 * e + 8) + (2 * e + 8) + (e + 8) + (3 * e + 8) + (2 * e + 8)
    cell = e + 5 * e + 3 * e + 3 * e + 3 * e + e
    bnd = 2 * e + (4 * e + 4) + (2 * e + 4) + (2 * e + 4) + (4 * e + 4) + (3 * e + 4)
    return face * F + cell * N + bnd * B


def _heat_assembly(N, F, B):
    return 56 * F + 40 * N + 36 * B


def _cg(N, F, its, mixed):
    return its * (2 * F * (8 if mixed else 12) + N * (48 if mixed else 96)) + 60 * F + 60 * N


def work(case):
    kind = case["kind"]
    if kind == "batch":
        b = fl = 0
        for n, kappa, _ in _members(case, 0):
            N, F, B = _sizes(dict(nx=n, ny=n, nz=n))
            its = 4 + 120 * math.sqrt(kappa * HEAT_DT) * n
            b += case["steps"] * (_heat_assembly(N, F, B) + _cg(N, F, its, True))
            fl += case["steps"] * (its * (4 * F + 14 * N) + 6 * F)
        return {"bytes": b, "flops": fl}
    N, F, B = _sizes(case)
    if kind == "explicit":
        e = 8 if case["prec"] == "f64" else 4
        b = _sweep_bytes(N, F, B, e)
        if case["order"] == "random":  # three fields in, six results out
            b += (4 + 2 * e) * ((N + 2 * (F + B)) + (4 * N + 2 * (F + B))) + 4 * e * N
        return {"bytes": b, "flops": 46 * F + 8 * N}
    if kind == "heat":
        its = 5 * case["steps"]
        return {"bytes": case["steps"] * _heat_assembly(N, F, B) + _cg(N, F, its, case["precision"] == "mixed"),
                "flops": its * (4 * F + 14 * N)}
    if kind == "poisson":
        its = 6.5 * max(case["nx"], case["ny"], case["nz"])
        return {"bytes": _cg(N, F, its, case["precision"] == "mixed") + 40 * F + 40 * N,
                "flops": its * (4 * F + 14 * N)}
    if kind == "advection":
        its = 12
        return {"bytes": its * (2 * 24 * F + 200 * N) + 80 * F + 80 * N, "flops": its * (8 * F + 30 * N)}
    corr = F * (64 + 60 + 24 + 56 + 40 + 48 + 56 + 40) + N * (88 + 136 + 8 + 24 + 40 + 40 + 40 + 96)
    if kind == "corrector":
        return {"bytes": corr, "flops": 90 * F + 60 * N}
    its = 3 * 4 * 2 + 2 * 1.2 * max(case["nx"], case["ny"], case["nz"])
    return {"bytes": 2 * corr + _cg(N, F, its, False), "flops": 180 * F + 120 * N + its * (4 * F + 14 * N)}


# ---------------------------------------------------------------------------
# the same results in 64 bits, by torch alone
# ---------------------------------------------------------------------------

class Exact:
    """Finite-volume operators on a Grid's geometry."""

    def __init__(self, grid):
        self.g, self.grid = grid.geometry(), grid
        self.o, self.n, self.fc, self.F, self.N = grid.own[:grid.F], grid.nbr, grid.fc, grid.F, grid.N

    def gather(self, face, bnd, minus=None):
        out = torch.zeros((self.N,) + tuple(face.shape[1:]), dtype=F64, device=DEV)
        out.index_add_(0, self.o, face).index_add_(0, self.n, -(face if minus is None else minus))
        return out.index_add_(0, self.fc, bnd)

    def lin(self, T):
        w = self.g["w"] if T.dim() == 1 else self.g["w"][:, None]
        return w * T[self.o] + (1 - w) * T[self.n]

    def grad(self, T, Tb):
        return self.gather(self.g["Sf"] * self.lin(T)[:, None], self.g["Sfb"] * Tb[:, None]) / self.g["V"][:, None]

    def div(self, phi, T=None, Tb=None, upwind=False):
        pf, pb = phi[:self.F], phi[self.F:]
        if T is None:
            return self.gather(pf, pb) / self.g["V"]
        Tf = torch.where(pf >= 0, T[self.o], T[self.n]) if upwind else self.lin(T)
        return self.gather(pf * Tf, pb * Tb) / self.g["V"]

    def flux(self, U, Ub):
        return torch.cat([(self.g["Sf"] * self.lin(U)).sum(1), (self.g["Sfb"] * Ub).sum(1)])


class System:
    """diag, upper (owner row), lower (neighbour row), right-hand side."""

    def __init__(self, ex):
        z = lambda n: torch.zeros(n, dtype=F64, device=DEV)  # noqa: E731
        self.ex, self.d, self.up, self.lo, self.b = ex, z(ex.N), z(ex.F), z(ex.F), z(ex.N)
        self.bm, self.br = z(ex.grid.B), z(ex.grid.B)

    def ddt(self, Told, dt):
        self.d += self.ex.g["V"] / dt
        self.b += self.ex.g["V"] / dt * Told

    def div(self, phi, Tb, upwind):  # fixedValue boundaries
        ex, pf = self.ex, phi[:self.ex.F]
        lam = (pf >= 0).to(F64) if upwind else ex.g["w"]
        lower = -lam * pf
        upper = lower + pf
        self.up += upper
        self.lo += lower
        self.d.index_add_(0, ex.o, -lower).index_add_(0, ex.n, -upper)
        self.b.index_add_(0, ex.fc, -phi[ex.F:] * Tb)

    def laplacian(self, gamma, Tb, fixed, c):  # fixed: per boundary face, else zero gradient
        ex = self.ex
        u = c * gamma[:ex.F] * ex.g["magSf"] * ex.g["nodc"]
        self.up += u
        self.lo += u
        ic = c * gamma[ex.F:] * ex.g["magSfb"] * ex.g["dcb"] * fixed
        self.d.index_add_(0, ex.o, -u).index_add_(0, ex.n, -u).index_add_(0, ex.fc, -ic)
        self.b.index_add_(0, ex.fc, -ic * Tb)
        self.bm += ic
        self.br += ic * Tb

    def off(self, x):
        e = self.ex
        up, lo = (self.up, self.lo) if x.dim() == 1 else (self.up[:, None], self.lo[:, None])
        return torch.zeros_like(x).index_add_(0, e.o, up * x[e.n]).index_add_(0, e.n, lo * x[e.o])

    def mul(self, x):
        return self.d * x + self.off(x)

    def cg(self, x, rtol, atol=0.0, most=20000):
        """Jacobi-preconditioned CG, stopped on ||b - A x|| after each update."""
        bn = self.b.norm().item() or 1.0
        r = self.b - self.mul(x)
        p, z = None, r / self.d
        rz = (r * z).sum()
        for _ in range(most):
            rn = r.norm().item()
            if rn <= rtol * bn or rn <= atol:
                break
            p = z.clone() if p is None else z + beta * p  # noqa: F821
            q = self.mul(p)
            a = rz / (p * q).sum()
            x = x + a * p
            r = r - a * q
            z = r / self.d
            new = (r * z).sum()
            beta, rz = new / rz, new
        return x

    def bicgstab(self, x, rtol, atol=0.0, most=1000):
        """Right-preconditioned (Jacobi) BiCGStab, stopped on ||r|| before each iteration."""
        bn = self.b.norm().item() or 1.0
        r = self.b - self.mul(x)
        rh, p, v = r.clone(), None, None
        rho = al = om = 1.0
        for _ in range(most):
            rn = r.norm().item()
            if rn <= rtol * bn or rn <= atol:
                break
            new = (rh * r).sum()
            p = r.clone() if p is None else r + (new / rho) * (al / om) * (p - om * v)
            rho = new
            y = p / self.d
            v = self.mul(y)
            al = rho / (rh * v).sum()
            s = r - al * v
            z = s / self.d
            t = self.mul(z)
            om = (t * s).sum() / (t * t).sum()
            x = x + al * y + om * z
            r = s - om * t
        return x


def exact(case, seed):
    if case["kind"] == "batch":
        out = []
        for n, kappa, sd in _members(case, seed):
            ex = Exact(Grid(n, n, n, "block"))
            f = _member_fields(n, kappa, sd, ex.grid)
            out.append(_heat_steps(ex, f, case["steps"], 1e-11))
        return out
    grid = _grid(case)
    ex, f = Exact(grid), {k: v.double() for k, v in _fields(case, seed, grid).items()}
    return _EXACT[case["kind"]](case, ex, f)


def _exact_explicit(case, ex, f):
    g, F = ex.g, ex.F
    T, Tb, gamma = f["T"], f["Tb"], f["gamma"]
    grads = torch.tensor([k == "fixedGradient" for k in EXPLICIT_BCS], device=DEV)[ex.grid.patch_of]
    snb = torch.where(grads, f["Tg"], g["dcb"] * (Tb - T[ex.fc]))
    sn = g["nodc"] * (T[ex.n] - T[ex.o])
    lap = ex.gather(gamma[:F] * g["magSf"] * sn, gamma[F:] * g["magSfb"] * snb) / g["V"]
    return dict(interp=torch.cat([ex.lin(T), Tb]), grad=ex.grad(T, Tb), div=ex.div(f["phi"], T, Tb),
                upwind=ex.div(f["phi"], T, Tb, True), lap=lap, sngrad=torch.cat([sn, snb]))


def _heat_steps(ex, f, steps, rtol):
    T, one = f["T"], torch.ones_like(f["Tb"])
    for _ in range(steps):
        s = System(ex)
        s.ddt(T, HEAT_DT)
        s.laplacian(f["gamma"], f["Tb"], one, -1.0)
        T = s.cg(T, rtol)
    return T


def _exact_heat(case, ex, f):
    return _heat_steps(ex, f, case["steps"], 1e-12)


def _exact_poisson(case, ex, f):
    fixed = (ex.grid.patch_of == 0).to(F64)
    zero = torch.zeros(ex.grid.B, dtype=F64, device=DEV)
    s = System(ex)
    s.laplacian(f["gamma"], zero, fixed, 1.0)
    s.b += ex.div(f["phi"]) * ex.g["V"]
    p = s.cg(torch.zeros_like(s.b), 1e-8)
    return {"p": p, "pb": torch.where(fixed > 0, zero, p[ex.fc])}


def _exact_advection(case, ex, f):
    s = System(ex)
    s.ddt(f["T"], ADV_DT)
    s.div(f["phi"], f["Tb"], case["scheme"] == "upwind")
    s.laplacian(f["gamma"], f["Tb"], torch.ones_like(f["Tb"]), -1.0)
    return s.bicgstab(f["T"], 1e-12)


def _momentum(ex, f, phi, U, dt, upwind):
    """The momentum matrix and its three right-hand sides."""
    b3 = []
    for k in range(3):
        s = System(ex)
        s.ddt(U[:, k], dt)
        s.div(phi, f["Ub"][:, k], upwind)
        s.laplacian(f["gamma"], f["Ub"][:, k], torch.ones_like(f["pb"]), -1.0)
        b3.append(s.b)
    return s, torch.stack(b3, 1)


def _predict(ex, f, s, b3, U):
    """rAUf, HbyA, phiHbyA and rAU of a corrector."""
    rau = ex.g["V"] / s.d
    H = (b3 - s.off(U)) * (rau / ex.g["V"])[:, None]
    rauf = torch.cat([ex.lin(rau), rau[ex.fc]])
    return rau, rauf, H, ex.flux(H, f["Ub"])


def _pressure(ex, rauf, phiH, pb):
    s = System(ex)
    s.laplacian(rauf, pb, torch.zeros_like(pb), 1.0)
    s.b += ex.div(phiH) * ex.g["V"]
    return s


def _new_flux(ex, s, phiH, p):
    inner = phiH[:ex.F] - (s.lo * p[ex.n] - s.up * p[ex.o])
    return torch.cat([inner, phiH[ex.F:] - (s.br - s.bm * p[ex.fc])])


def _exact_corrector(case, ex, f):
    s, b3 = _momentum(ex, f, f["phi"], f["U"], 0.5 * ex.grid.h, case["scheme"] == "upwind")
    rau, rauf, H, phiH = _predict(ex, f, s, b3, f["U"])
    ps = _pressure(ex, rauf, phiH, f["pb"])
    return {"rAUf": rauf, "phiHbyA": phiH, "residual": ps.mul(f["p"]) - ps.b,
            "phi": _new_flux(ex, ps, phiH, f["p"]),
            "U": H - rau[:, None] * ex.grad(f["p"], f["pb"])}


def _exact_icofoam(case, ex, f):
    U, p, phi, dt = f["U"], f["p"], f["phi"], 0.5 * ex.grid.h
    mag = phi.abs()
    co = 0.5 * dt * (ex.gather(mag[:ex.F], mag[ex.F:], -mag[:ex.F]) / ex.g["V"]).max().item()
    s, b3 = _momentum(ex, f, phi, U, dt, case["scheme"] == "upwind")
    cols = []
    for k in range(3):
        s.b = b3[:, k].contiguous()
        cols.append(s.bicgstab(U[:, k].contiguous(), 0.0, SOLVER_U["tolerance"]))
    U = torch.stack(cols, 1)
    for _ in range(2):
        rau, rauf, H, phiH = _predict(ex, f, s, b3, U)
        ps = _pressure(ex, rauf, phiH, p[ex.fc])
        ps.d[0] += ps.d[0].clone()  # setReference(cell 0, value 0)
        p = ps.cg(p, SOLVER_P["relTol"], SOLVER_P["tolerance"])
        phi = _new_flux(ex, ps, phiH, p)
        U = H - rau[:, None] * ex.grad(p, p[ex.fc])
    return {"U": U, "p": p, "phi": phi, "coNum": co}


_EXACT = {"explicit": _exact_explicit, "heat": _exact_heat, "poisson": _exact_poisson,
          "advection": _exact_advection, "corrector": _exact_corrector, "icofoam": _exact_icofoam}
