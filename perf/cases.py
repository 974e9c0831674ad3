"""The framework's work as its users have it done: measured cases of the public entry points.

Four kinds, each over the sizes that the repository's configurations, tests and benchmark
use and the generic ones between them (nx/2 and ny products of 2, 3, 5; any nz):

* ``step``      whole time steps of a resident run (``Context.timestep``), DNS and the LES
                models, FP64 and mixed form; the outputs are the new u, v, w, p spectra;
* ``ensemble``  one step of every member of an uneven ensemble from its captured graphs;
* ``horfft``    the batched 2-D transform on device fields, forward and then inverse;
* ``helmholtz`` the batched Chebyshev-Helmholtz solve on device fields, in FP64 or with
                FP32 projections and one FP64 refinement;
* ``dfdz``      the wall-normal derivative of device fields.

``prepare`` is what a run holds before the call (context, state past its three start-up
steps, device arrays), ``run`` one pass.  Passes are ordered on the program's own stream,
as a program that post-processes the fields there orders them.
"""

from __future__ import annotations

import ctypes
import math

import numpy as np
import torch

import lsbflow_amd as L
from lsbflow_amd import _lib
from lsbflow_amd.core import Ensemble, setup_case

PI = math.pi
MODELS = {"none": None, "static": 0, "dynamic": 1, "sigma": 2}
STARTUP = 3  # Euler, BDF2 and the first BDF3 step: their coefficients differ from the rest


def listed():
    return [
        # the smallest resident run, some steps of the 64 x 65 x 32 DNS: launches and latency
        dict(name="dns_64x65x32", kind="step", nx=64, nz=64, ny=32, model="none", mixed=False, steps=4),
        # the 256 x 129 x 128 dynamic-model LES of the accuracy runs
        dict(name="les_dynamic_mixed_256x129x128", kind="step", nx=256, nz=128, ny=128, model="dynamic", mixed=True,
             steps=1),
        # the benchmark's workload
        dict(name="les_sigma_mixed_512x193x256", kind="step", nx=512, nz=192, ny=256, model="sigma", mixed=True,
             steps=1),
        # its dynamic-model companion in FP64, the heaviest step
        dict(name="les_dynamic_fp64_512x193x256", kind="step", nx=512, nz=192, ny=256, model="dynamic", mixed=False,
             steps=1),
        # an ordinary LES on lengths with a factor of 3, as the uneven ensemble's larger grids
        dict(name="les_static_mixed_192x97x96", kind="step", nx=192, nz=96, ny=96, model="static", mixed=True,
             steps=2),
        # the same in FP64 on a ragged grid: factors of 3 and 5, an even number of planes
        dict(name="les_sigma_fp64_240x114x120", kind="step", nx=240, nz=113, ny=120, model="sigma", mixed=False,
             steps=1),
        # members of the uneven static-model ensemble stepped together
        dict(name="ensemble_mixed_6", kind="ensemble", members=6, mixed=True, steps=1),
        # velocity-sized batches of the 2-D transform: the benchmark's grid and a ragged one
        dict(name="horfft_512x193x256", kind="horfft", nx=512, nz=192, ny=256, fields=3),
        dict(name="horfft_192x65x60", kind="horfft", nx=192, nz=64, ny=60, fields=2),
        # every pencil of a 512 x 193 x 256 grid for four right-hand sides
        dict(name="helmholtz_fp64_512x193x256", kind="helmholtz", nx=512, nz=192, ny=256, fields=4, mode="fp64"),
        # the solve with FP32 projections and an FP64 refinement
        dict(name="helmholtz_refined_256x129x128", kind="helmholtz", nx=256, nz=128, ny=128, fields=3, mode="refine"),
        # the derivative of a scalar and a vector field
        dict(name="dfdz_320x129x160", kind="dfdz", nx=320, nz=128, ny=160, fields=4),
    ]


def _smooth(lo, hi):
    return [n for n in range(lo, hi + 1) if _is_smooth(n)]


def _is_smooth(n):
    for p in (2, 3, 5):
        while n % p == 0:
            n //= p
    return n == 1


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _near(values, x):
    return min(values, key=lambda v: abs(math.log(v / x)))


def draw(rng):
    kind = rng.choice(["step", "step", "step", "horfft", "horfft", "helmholtz", "dfdz"])
    points = math.exp(rng.uniform(math.log(64 * 65 * 32), math.log(512 * 193 * 256)))
    nz = _log_int(rng, 48, 192)
    aspect = math.exp(rng.uniform(math.log(1.0), math.log(4.0)))  # nx / ny
    ny = _near([n for n in _smooth(24, 256) if n % 2 == 0], min(256.0, max(24.0, math.sqrt(points / (nz + 1) / aspect))))
    nx = 2 * _near(_smooth(24, 256), min(256.0, max(24.0, points / (nz + 1) / ny / 2)))
    c = dict(kind=kind, nx=nx, nz=nz, ny=ny)
    if kind == "step":
        model = rng.choice(["none", "static", "dynamic", "sigma"])
        if nx < 96 or ny < 48:  # an LES at these viscosities needs some horizontal resolution
            model = "none"
        c.update(model=model, mixed=rng.random() < 0.5, steps=4 if points < 1.0e6 else 1)
    else:
        c["fields"] = rng.randint(1, 4)
    if kind == "helmholtz":
        c["mode"] = rng.choice(["fp64", "refine"])
    return c


# ------------------------------------------------------------------- the workloads
def flow(case, seed):
    """The configuration of a step case (lsbflow_amd.cases): the DNS as configured but with
    the exact wall-normal operator, without which a run of thousands of steps grows; the
    LES runs the suction/blowing ceiling with the switches and the time-step rule of the
    ensemble's members."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    model = MODELS[case["model"]]
    if model is None:
        return L.cases.CASES["c1_dns"].with_(nx=nx, ny=ny, nz=nz, seed=seed, dct_exact=1)
    base = L.cases.CASES["c2_dyn_les"]
    dz_top = 0.5 * base.zlen * (1.0 - math.cos(PI / nz))
    return base.with_(nx=nx, ny=ny, nz=nz, sgsmodel=model, seed=seed, xnu=0.2 / 5.0e4,
                      dt=min(2.5e-4, 0.15 * dz_top / base.samp), nut_ceil0=0 if model == 1 else 1)


def members(case, seed):
    return [m.with_(seed=seed + 31 * i) for i, m in enumerate(L.cases.ensemble_members(16)[: case["members"]])]


_stream = None


def program_stream():
    """The stream on which the calling program orders its work."""
    global _stream
    if _stream is None:
        _stream = torch.cuda.Stream()
    return _stream


class _DeviceArray:
    """A context's device memory for torch; keeps the context alive."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr="<f8", data=(ptr, False), version=3)


def _fields(ctx):
    return {k: torch.as_tensor(_DeviceArray(ctx, p, ctx.sshape), device="cuda")
            for k, p in zip(("u", "v", "w", "p"), ctx.device_ptrs())}


def _started(flow_case, mixed):
    ctx = setup_case(flow_case, precision=1 if mixed else 0)
    ctx.state_set(*L.cases.initial_condition(flow_case))
    ctx.timestep(STARTUP)
    return ctx


def _bare_context(case):
    """A context for the kernel-level entries: the benchmark's channel, no state."""
    return setup_case(L.cases.CASES["c2_dyn_les"].with_(nx=case["nx"], ny=case["ny"], nz=case["nz"]))


def _generator(seed, device="cuda"):
    return torch.Generator(device=device).manual_seed(seed)


def _smooth_pencils(case, seed):
    """(fields, nzp, ny, nx) with Chebyshev coefficients N(0,1) exp(-0.1 n), as the batched
    solve's tests and benchmark draw them."""
    n = case["nz"] + 1
    coef = torch.randn((n, case["fields"] * case["ny"] * case["nx"]), generator=_generator(seed), dtype=torch.float64,
                       device="cuda")
    coef *= torch.exp(-0.1 * torch.arange(n, device="cuda", dtype=torch.float64))[:, None]
    k = np.arange(n)
    cheb = torch.from_numpy(np.cos(PI * np.outer(k, k) / (n - 1))).cuda()
    out = (cheb @ coef).reshape(n, case["fields"], case["ny"], case["nx"])
    return out.permute(1, 0, 2, 3).contiguous()


def _physical(case, seed):
    """(fields, nzp, ny, nx + 2) velocity-like rows, the two pads of each row zero."""
    x = torch.zeros((case["fields"], case["nz"] + 1, case["ny"], case["nx"] + 2), dtype=torch.float64, device="cuda")
    x[..., : case["nx"]] = torch.randn(x.shape[:-1] + (case["nx"],), generator=_generator(seed), dtype=torch.float64,
                                       device="cuda")
    return x


def _dtnui(case):
    """sigma of a velocity solve: 1/(nu dt) at the benchmark's viscosity and time step."""
    return 1.0 / (0.2 / 1.0e5 * 2.5e-4)


def prepare(case, seed):
    if case["kind"] == "step":
        return dict(case=case, ctx=_started(flow(case, seed), case["mixed"]))
    if case["kind"] == "ensemble":
        ctxs = [_started(m, case["mixed"]) for m in members(case, seed)]
        return dict(case=case, ctxs=ctxs, ens=Ensemble(ctxs))
    ctx = _bare_context(case)
    if case["kind"] == "horfft":
        x = _physical(case, seed)
        spec = torch.empty(x.shape[:-1] + (case["nx"],), dtype=torch.float64, device="cuda")
        return dict(case=case, ctx=ctx, x=x, spec=spec, back=torch.empty_like(x))
    x = _smooth_pencils(case, seed)
    return dict(case=case, ctx=ctx, x=x, out=torch.empty_like(x))


def _ptr(t):
    return ctypes.c_void_p(t.data_ptr())


def run(state):
    case, s = state["case"], program_stream()
    lib = _lib.lib()
    handle = ctypes.c_void_p(s.cuda_stream)
    if case["kind"] == "step":
        ctx = state["ctx"]
        own = torch.cuda.ExternalStream(ctx.stream())
        own.wait_stream(s)
        ctx.timestep(case["steps"])
        s.wait_stream(own)
        return _fields(ctx)
    if case["kind"] == "ensemble":
        own = torch.cuda.ExternalStream(state["ctxs"][0].stream())
        own.wait_stream(s)
        state["ens"].timestep(case["steps"])
        s.wait_stream(own)
        return [_fields(ctx) for ctx in state["ctxs"]]
    ctx, n = state["ctx"], case["fields"]
    if case["kind"] == "horfft":
        _lib.check(lib.lsb_horfft_dev(ctx.h, _ptr(state["x"]), _ptr(state["spec"]), -1, n, handle), "horfft")
        _lib.check(lib.lsb_horfft_dev(ctx.h, _ptr(state["back"]), _ptr(state["spec"]), 1, n, handle), "horfft")
        return dict(spec=state["spec"], back=state["back"])
    if case["kind"] == "helmholtz":  # in place: the program keeps its right-hand sides
        with torch.cuda.stream(s):
            state["out"].copy_(state["x"])
        if case["mode"] == "fp64":
            rc = lib.lsb_solve_helmholtz_dev(ctx.h, _ptr(state["out"]), _dtnui(case), n, handle)
        else:
            rc = lib.lsb_solve_helmholtz_mixed_dev(ctx.h, _ptr(state["out"]), _dtnui(case), n, 2, handle)
        _lib.check(rc, "helmholtz")
        return state["out"]
    _lib.check(lib.lsb_dfdz_dev(ctx.h, _ptr(state["x"]), _ptr(state["out"]), n, handle), "dfdz")
    return state["out"]


def _step_work(nx, ny, nzp, mixed):
    """One step's state read and written once (u, v, w and their two past levels, the two
    past N, p and its past level; the new u, v, w, p, N), and the operations of its 8
    wall-normal contractions and 8 eigen-projections in half-size parity pairs and 17
    2-D transforms."""
    n = nx * ny * nzp
    hist = 4 if mixed else 8
    bytes_ = n * (11 * 8 + 6 * hist + 4 * 8 + 3 * hist)
    flops = 16.0 * nzp * n + 17 * 2.5 * n * math.log2(nx * ny)
    return dict(bytes=bytes_, flops=flops)


def work(case):
    if case["kind"] == "ensemble":
        each = [_step_work(m.nx, m.ny, m.nzp, case["mixed"]) for m in members(case, 0)]
        return {k: case["steps"] * sum(w[k] for w in each) for k in ("bytes", "flops")}
    nx, ny, nzp = case["nx"], case["ny"], case["nz"] + 1
    if case["kind"] == "step":
        w = _step_work(nx, ny, nzp, case["mixed"])
        return {k: case["steps"] * v for k, v in w.items()}
    n = nx * ny * nzp * case["fields"]
    if case["kind"] == "horfft":
        return dict(bytes=2 * 8 * (n + n * (nx + 2) // nx), flops=2 * 2.5 * n * math.log2(nx * ny))
    return dict(bytes=16 * n, flops=(2.0 if case["kind"] == "helmholtz" else 1.0) * n * nzp)


def tolerance(case):
    """About four times what another order of the same sums shows over the ranges (dense
    instead of parity-split operators, separate instead of fused passes, the 64-bit
    reference below): the pressure, a divergence over k^2 dt, sets the FP64 steps'
    figures, FP32's rounding in the nonlinear chain the mixed ones'."""
    if case["kind"] in ("step", "ensemble"):
        return {"rel": 1e-6, "max": 2e-4} if case["mixed"] else {"rel": 2e-7, "max": 2e-5}
    if case["kind"] == "horfft":
        return {"rel": 4e-15, "max": 4e-14}
    if case["kind"] == "helmholtz":
        return {"rel": 1e-14, "max": 2e-13} if case["mode"] == "fp64" else {"rel": 4e-13, "max": 2e-11}
    return {"rel": 1e-13, "max": 5e-12}


# ------------------------------------------------- the same in plain 64-bit torch
def exact(case, seed):
    if case["kind"] == "step":
        return _exact_step(flow(case, seed), STARTUP + case["steps"])
    if case["kind"] == "ensemble":
        return [_exact_step(m, STARTUP + case["steps"]) for m in members(case, seed)]
    nx, ny, n = case["nx"], case["ny"], case["nz"] + 1
    if case["kind"] == "horfft":
        g = _Horizontal(nx, ny, 2.0 * PI, PI)
        x = _physical(case, seed)[..., :nx]
        spec = torch.stack([g.forward(f) for f in x])
        back = torch.zeros(x.shape[:-1] + (nx + 2,), dtype=torch.float64, device="cuda")
        for f in range(case["fields"]):
            back[f, ..., :nx] = g.inverse(spec[f])
        return dict(spec=_reals(spec), back=back)
    z = _Vertical(n, 2.0, True)
    x = _smooth_pencils(case, seed)
    if case["kind"] == "dfdz":
        return torch.stack([z.apply(z.dct, f) for f in x])
    g = _Horizontal(nx, ny, 2.0 * PI, PI)
    k2 = g.k2.repeat_interleave(2, dim=1)
    return torch.stack([z.solve(f, k2 + _dtnui(case)) for f in x])


def _reals(c):
    return torch.view_as_real(c.contiguous()).reshape(c.shape[:-1] + (2 * c.shape[-1],))


class _Horizontal:
    """Fourier in x and y: (planes, ny, nx) reals <-> (planes, ny, nx/2) coefficients."""

    def __init__(self, nx, ny, xlen, ylen):
        self.nx, self.ny = nx, ny
        self.ikx = 2j * PI / xlen * torch.arange(nx // 2, dtype=torch.float64, device="cuda")[None, :]
        j = torch.arange(ny, dtype=torch.float64, device="cuda")
        j = torch.where(j >= ny // 2, j - ny, j)
        self.iky = 2j * PI / ylen * j[:, None]
        self.k2 = self.ikx.imag ** 2 + self.iky.imag ** 2

    def forward(self, x):
        return torch.fft.fft(torch.fft.rfft(x, dim=-1)[..., : self.nx // 2], dim=-2) / (self.nx * self.ny)

    def inverse(self, c):
        c = torch.fft.ifft(c, dim=-2, norm="forward")
        full = torch.zeros(c.shape[:-1] + (self.nx // 2 + 1,), dtype=torch.complex128, device="cuda")
        full[..., : self.nx // 2] = c
        full[..., 0].imag.zero_()
        return torch.fft.irfft(full, n=self.nx, dim=-1, norm="forward")


class _Vertical:
    """Chebyshev points z = zlen/2 (1 + cos(pi k/nz)): the collocation derivative (also of a
    reference-scaled top coefficient) and the Dirichlet solves in its eigenvectors."""

    def __init__(self, n, zlen, exact_top):
        k = np.arange(n)
        self.n = n
        self.z = zlen / 2.0 * (1.0 + np.cos(PI * k / (n - 1)))
        c = np.where((k == 0) | (k == n - 1), 2.0, 1.0)
        cheb = np.cos(PI * np.outer(k, k) / (n - 1))       # T_m at point i
        to_coef = 2.0 / (n - 1) * cheb / np.outer(c, c)
        der = np.zeros((n, n))                              # coefficients of d/dz
        for m in range(n):
            for q in range(m - 1, -1, -2):
                der[q, m] = 2.0 * m / (1.0 if q else 2.0) * 2.0 / zlen
        d = cheb @ der @ to_coef
        if not exact_top:                                   # chebyshev.f90:242: alpha(n) not over zlen
            der[:, n - 1] *= zlen
        dct = d if exact_top else cheb @ der @ to_coef
        i, j = np.meshgrid(k, k, indexing="ij")
        with np.errstate(divide="ignore", invalid="ignore"):
            # x_i - x_j = 2 sin((i + j) pi/2nz) sin((j - i) pi/2nz); the diagonal closes the rows
            s = c[i] / c[j] * (-1.0) ** (i + j) / (
                2.0 * np.sin((i + j) * PI / (2 * (n - 1))) * np.sin((j - i) * PI / (2 * (n - 1))))
        s[k, k] = 0.0
        s[k, k] = -s.sum(axis=1)
        d = s * 2.0 / zlen
        d2 = d @ d
        lam, e = np.linalg.eig(d2[1:-1, 1:-1])
        up = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
        self.lam, self.e, self.ei = up(lam.real), up(e.real), up(np.linalg.inv(e.real))
        self.dct, self.dct2 = up(d if exact_top else dct), up((d if exact_top else dct) @ (d if exact_top else dct))
        b, h = 50.0, zlen
        bot = (np.exp(-b * self.z) - np.exp(b * (self.z - 2.0 * h))) / (1.0 - math.exp(-2.0 * b * h))
        top = np.exp(b * (self.z - h)) * (1.0 - np.exp(-2.0 * b * self.z)) / (1.0 - math.exp(-2.0 * b * h))
        self.bot, self.top, self.b2 = up(bot), up(top), b * b

    def apply(self, m, f):
        r = torch.view_as_real(f.contiguous()) if f.is_complex() else f
        r = (m @ r.reshape(self.n, -1)).reshape(r.shape)
        return torch.view_as_complex(r) if f.is_complex() else r

    def solve(self, rhs, s, bc_top=None, bc_bot=None):
        """(D2 - s) u = rhs on the interior, u the given planes (or zero) at the ends."""
        if bc_top is not None:
            col = lambda v: v[:, None, None]  # noqa: E731
            rhs = (rhs - (self.b2 - s) * col(self.bot) * bc_bot - (self.b2 - s) * col(self.top) * bc_top)
        q = torch.view_as_real(rhs[1:-1].contiguous()) if rhs.is_complex() else rhs[1:-1].contiguous()
        t = (self.ei @ q.reshape(self.n - 2, -1)).reshape(q.shape)
        den = self.lam[:, None, None] - s[None]
        t /= den[..., None] if rhs.is_complex() else den
        t = (self.e @ t.reshape(self.n - 2, -1)).reshape(q.shape)
        out = torch.zeros_like(rhs)
        out[1:-1] = torch.view_as_complex(t) if rhs.is_complex() else t
        if bc_top is not None:
            out += col(self.bot) * bc_bot + col(self.top) * bc_top
        return out


class _Models:
    """The eddy-viscosity models on physical gradients g[l][m] = du_l/dx_m."""

    def __init__(self, c, v):
        z = v.z
        dx, dy = c.xlen / (c.nx - 1.0), c.ylen / (c.ny - 1.0)  # the reference's spacings
        dz = np.empty(v.n)
        dz[0], dz[-1] = z[0] - z[1], z[-2] - z[-1]
        dz[1:-1] = 0.5 * (z[:-2] - z[2:])
        self.c, self.z = c, z
        width = (dx * dy * dz) ** (1.0 / 3.0)
        ceil0 = width.copy()
        if c.nut_ceil0:
            ceil0[0] = 0.0
        wall0 = ceil0.copy()
        wall0[-1] = 0.0
        if not c.nut_ceil0:
            wall0[0] = (dx * dy * dz[-1]) ** (1.0 / 3.0)
        self.width, self.sigma_width, self.static_width = width, ceil0, wall0
        self.wz = self._z_weights(c.a, c.b), self._z_weights(1.0, 1.0)

    def _z_weights(self, a, b):
        z, n = self.z, len(self.z)
        w = np.zeros((3, n))
        w[1] = 2.0 * a + b
        for k in range(1, n - 1):
            up, dn = z[k] - z[k - 1], z[k + 1] - z[k]
            mid = (n + 1) // 2 - 1
            if k == mid:
                w[:, k] = a, b, a
            elif k < mid:
                w[:, k] = a * 2 * up / (dn + up), a * 2 * (1 - up / dn) + b, a * 2 * up * up / (dn * (dn + up))
            else:
                w[:, k] = a * 2 * dn * dn / (up * (dn + up)), a * 2 * (1 - dn / up) + b, a * 2 * dn / (dn + up)
        return torch.from_numpy(w).cuda()[:, :, None, None]

    def _filter(self, q, which):
        a, b = (self.c.a, self.c.b) if which == 0 else (1.0, 1.0)
        w, s = self.wz[which], 2.0 * a + b
        for axis in (-1, -2):
            q = (a * torch.roll(q, 1, axis) + b * q + a * torch.roll(q, -1, axis)) / s
        out = w[1] * q / s
        out[0], out[-1] = q[0], q[-1]
        out[1:-1] += (w[0, 1:-1] * q[:-2] + w[2, 1:-1] * q[2:]) / s
        return out

    @staticmethod
    def _plane(a):
        return torch.from_numpy(np.ascontiguousarray(a)).cuda()[:, None, None]

    def stress(self, u, g):
        """tau[l][m], l <= m."""
        pairs = [(l, m) for l in range(3) for m in range(l, 3)]
        strain = {(l, m): 0.5 * (g[l][m] + g[m][l]) for l, m in pairs}
        twice = {p: (1.0 if p[0] == p[1] else 2.0) for p in pairs}
        norm = lambda s: torch.sqrt(sum(2.0 * twice[p] * s[p] * s[p] for p in pairs))  # noqa: E731
        model = self.c.sgsmodel
        if model == 0:
            wall = [k for k in range(len(self.z)) if self.z[k] == 0.0 or abs(self.z[k]) == 0.5]
            utau = math.sqrt(abs(float(sum(g[0][2][k] for k in wall).mean()) * self.c.xnu / len(wall)))
            damp = 1.0 - np.exp(-self.z * utau / self.c.xnu / 25.0)
            nu = -self._plane((self.c.cs * self.static_width * damp) ** 2) * norm(strain)
            return {p: nu * s for p, s in strain.items()}
        if model == 2:
            nu = 2.0 * self._sigma(g)
            return {p: nu * s for p, s in strain.items()}
        d2 = self._plane(self.width ** 2)
        sn = norm(strain)
        hat = {p: self._filter(s, 0) for p, s in strain.items()}
        hn = norm(hat)
        num = den = 0.0
        uh = [self._filter(x, 0) for x in u]
        for l, m in pairs:
            mij = 2.0 * (self._filter(d2 * sn * strain[l, m], 0) - 4.0 * d2 * hn * hat[l, m])
            lij = self._filter(u[l] * u[m], 0) - uh[l] * uh[m]
            num = num + twice[l, m] * mij * lij
            den = den + twice[l, m] * mij * mij
        cd = torch.nan_to_num(self._filter(num, 1) / self._filter(den, 1), nan=0.0).clamp(0.0, 0.04)
        return {p: -2.0 * cd * d2 * sn * s for p, s in strain.items()}

    def _sigma(self, g):
        G = [[sum(g[k][a] * g[k][b] for k in range(3)) for b in range(3)] for a in range(3)]
        i1 = G[0][0] + G[1][1] + G[2][2]
        i2 = 0.5 * (i1 ** 2 - sum(G[a][b] * G[b][a] for a in range(3) for b in range(3)))
        i3 = (G[0][0] * (G[1][1] * G[2][2] - G[1][2] * G[2][1]) - G[0][1] * (G[1][0] * G[2][2] - G[1][2] * G[2][0])
              + G[0][2] * (G[1][0] * G[2][1] - G[1][1] * G[2][0]))
        a1 = (i1 ** 2 / 9.0 - i2 / 3.0).abs()
        pre = (i1 ** 3 / 27.0 - i1 * i2 / 6.0 + 0.5 * i3) / torch.sqrt(a1) ** 3
        a3 = torch.where((pre >= 1.0) | torch.isnan(pre), 0.0, torch.acos(pre.clamp(-1.0, 1.0)) / 3.0)
        sa = torch.sqrt(a1)
        s1, s2, s3 = (torch.sqrt((i1 / 3.0 + t).abs()) for t in (
            2.0 * sa * torch.cos(a3), -2.0 * sa * torch.cos(PI / 3.0 + a3), -2.0 * sa * torch.cos(PI / 3.0 - a3)))
        ds = s3 * (s1 - s2) * (s2 - s3)
        ds = torch.where(s1 != 0.0, ds / torch.where(s1 != 0.0, s1, 1.0) ** 2, ds)
        ds = torch.where((ds < 0.0) | torch.isnan(ds), 0.0, ds)
        return -self._plane((1.35 * self.sigma_width) ** 2) * ds


def _exact_step(c, steps):
    """The state after ``steps`` time steps from the seeded start (bctype 3; top_bc 0 or 2)."""
    h = _Horizontal(c.nx, c.ny, c.xlen, c.ylen)
    v = _Vertical(c.nz + 1, c.zlen, c.dct_exact == 1)
    model = _Models(c, v) if c.sgsflag else None
    ubar, ubarp, ubarpp = (torch.from_numpy(np.ascontiguousarray(a)).cuda()[:, None, None]
                           for a in L.cases.base_flow(c))
    u = [torch.view_as_complex(torch.from_numpy(f).cuda().reshape(c.nz + 1, c.ny, c.nx // 2, 2))
         for f in L.cases.initial_condition(c)]
    zero = torch.zeros_like(u[0])
    p, pn = zero, zero
    un, unm, nl, nlm = ([zero] * 3 for _ in range(4))
    # the spectral filter of dealiasflag 2
    kmax = math.hypot(c.nx // 2 * 2 * PI / c.xlen, c.ny // 2 * 2 * PI / c.ylen)
    theta = (torch.sqrt(h.k2) - kmax * c.kc) / (kmax - kmax * c.kc)
    damp = torch.where(theta >= 0.0, torch.exp(-c.filt_amp * theta ** (2 * c.filt_order)), 1.0)
    x = torch.from_numpy(L.cases.xpts(c)).cuda() - c.x0
    inflow = torch.exp(-(((x - 0.4 * c.xlen) / (0.05 * c.xlen)) ** 2))
    top_w = h.forward(torch.from_numpy(L.cases.ceiling_profile(c)).cuda().expand(1, c.ny, c.nx))[0]
    for istep in range(1, steps + 1):
        uf = [f * damp for f in u]
        phys = [h.inverse(f) for f in uf]
        g = [[h.inverse(h.ikx * f), h.inverse(h.iky * f), h.inverse(v.apply(v.dct, f))] for f in uf]
        phys[0] = phys[0] + ubar
        g[0][2] = g[0][2] + ubarp
        n = [-0.5 * h.forward(sum(phys[m] * g[l][m] for m in range(3))) for l in range(3)]
        tau = model.stress(phys, g) if model else {}
        del g
        for l in range(3):
            for m in range(3):
                q = 0.5 * phys[l] * phys[m]
                if tau:
                    q += tau[min(l, m), max(l, m)]
                q = h.forward(q)
                n[l] -= h.ikx * q if m == 0 else h.iky * q if m == 1 else v.apply(v.dct, q)
        del tau, phys, q
        ab = {1: (1.0, 0.0, 0.0), 2: (2.0, -1.0, 0.0)}.get(istep, (3.0, -3.0, 1.0))
        bdf, beta = {1: ((1.0, 0.0, 0.0), 1.0), 2: ((2.0, -0.5, 0.0), 2.0 / 3.0)}.get(
            istep, ((3.0, -1.5, 1.0 / 3.0), 6.0 / 11.0))
        a0 = 1.0 / (c.xnu * c.dt)
        s = h.k2 + a0 / beta
        rhs = [-a0 * (c.dt * (ab[0] * n[l] + ab[1] * nl[l] + ab[2] * nlm[l])
                      + bdf[0] * u[l] + bdf[1] * un[l] + bdf[2] * unm[l]) for l in range(3)]
        rhs[0][:, 0, 0] -= ubarpp[:, 0, 0]
        ps = {1: zero, 2: p}.get(istep, 2.0 * p - pn)
        dtb = c.dt * beta
        top = [-rhs[0][0] / s, -rhs[1][0] / s]
        if c.top_bc == 2:
            for l, ik in enumerate((h.ikx, h.iky)):
                free, wall = h.inverse(top[l][None]), h.inverse(dtb * (ik * ps[0])[None])
                top[l] = h.forward((1.0 - inflow) * free + inflow * wall)[0]
        top.append(top_w + c.xnu * dtb * torch.view_as_complex(
            (v.dct2[:1] @ torch.view_as_real(u[2]).reshape(v.n, -1)).reshape(c.ny, c.nx // 2, 2)))
        bot = [dtb * h.ikx * ps[-1], dtb * h.iky * ps[-1], torch.zeros_like(top_w)]
        new = [v.solve(rhs[l], s, top[l], bot[l]) for l in range(3)]
        del rhs, ps
        div = h.ikx * new[0] + h.iky * new[1]
        w = v.solve(-v.apply(v.dct, div) - h.k2 * new[2], h.k2, top_w, torch.zeros_like(top_w))
        pnew = torch.where(h.k2 == 0.0, 0.0, -(v.apply(v.dct, w) + div) / (h.k2 * dtb))
        new = [new[0] - dtb * h.ikx * pnew, new[1] - dtb * h.iky * pnew, w]
        for f in new:  # real fields: Hermitian kx = 0 column, no ky-Nyquist row
            f[:, 0, 0].imag.zero_()
            col = f[:, 1:, 0]
            f[:, 1:, 0] = 0.5 * (col + col.flip(1).conj())
            f[:, c.ny // 2] = 0.0
        u, un, unm, nl, nlm, p, pn = new, u, un, n, nl, pnew, p
    return {k: _reals(f) for k, f in zip("uvwp", u + [p])}
