"""The work a program has this library do, for timing and for comparing outputs.

Every case goes through the Python binding's public entry points (the C ABI
behind them): the two grid Poisson solves on device arrays from small grids to
512^3, with the options their callers use (ghost-fluid jumps, re-projection
with a warm start, the learned preconditioner), the velocity passes after a
projection, the whole sub-step on host arrays as the drop-in classes call it,
and the network's training gradients. Grids, interfaces and fields are those
of sfp.scenes (the benchmark's and the tests'), generated on the GPU.
"""
from __future__ import annotations

import math
import os
import sys
import time

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "simferrofluid-cuda_amd"))
import sfp  # noqa: E402
from sfp import learn  # noqa: E402

DEV = "cuda:0"
F64 = torch.float64


# ---------------------------------------------------------------- the cases
def listed():
    return [
        # an interactive preview grid: solids cutting cells, surface tension
        # jumps, a volume correction -- every branch of the assembly, and so
        # little data that the call's latency is all there is
        dict(name="pressure_20_jump", kind="pressure", nx=20, ny=20, nz=20, jump=True, solid=True),
        # a small off-centre container, odd in every axis (no z row of whole
        # 4-cell groups on any level)
        dict(name="magnetic_33x27x45", kind="magnetic", nx=33, ny=27, nz=45, chi=4.0, warm=False),
        # the 64^3 projection (sphere drop over a pool) of a desktop run
        dict(name="pressure_64", kind="pressure", nx=64, ny=64, nz=64, jump=False, solid=False),
        # the 128^3 magnetostatic potential
        dict(name="magnetic_128", kind="magnetic", nx=128, ny=128, nz=128, chi=2.0, warm=False),
        # two projections of one time step on a ragged grid: Project, then
        # Reproject (same matrix, new velocities, warm start)
        dict(name="reproject_131x129x133", kind="reproject", nx=131, ny=129, nz=133),
        # the magnetic solves of two consecutive time steps on a flat
        # container: the second starts from the first's potential
        dict(name="magnetic_warm_160x96x224", kind="magnetic", nx=160, ny=96, nz=224, chi=2.0,
             warm=True),
        # the benchmark's 256^3 projection and magnetic solve
        dict(name="pressure_256", kind="pressure", nx=256, ny=256, nz=256, jump=False, solid=False),
        dict(name="magnetic_256", kind="magnetic", nx=256, ny=256, nz=256, chi=2.0, warm=False),
        # the learned preconditioner (network inference, then its fall-back)
        dict(name="learned_256", kind="learned", nx=256, ny=256, nz=256, chi=2.0),
        # the largest production grid: the 512^3 spike interface
        dict(name="spike_512", kind="spike", nx=512, ny=512, nz=512, chi=4.0),
        # the drop-in classes' sub-step: projection, extrapolation and wall
        # condition on host arrays
        dict(name="substep_host_64", kind="substep", nx=64, ny=64, nz=64),
        # training the preconditioner: loss and gradients of a batch of crops
        dict(name="unet_gradients_8x32", kind="unet", batch=8, nx=32, ny=32, nz=32),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _grid(rng, lo, hi):
    """A box whose mean extent is log-uniform over lo..hi, with mild aspect
    ratios; a third of them cubes, half of the extents whole groups of four."""
    n = _log(rng, lo, hi)
    if rng.random() < 0.33:
        return (n, n, n)
    d = [max(lo // 2, int(n * rng.uniform(0.7, 1.3))) for _ in range(3)]
    if rng.random() < 0.5:
        d = [(v + 3) // 4 * 4 for v in d]
    return tuple(d)


def draw(rng):
    kind = rng.choice(["pressure", "pressure", "magnetic", "magnetic", "reproject", "spike",
                       "learned", "substep", "unet"])
    chi = round(0.5 * 16.0 ** rng.random(), 2)
    if kind == "unet":
        dims = [4 * rng.randint(4, 10) for _ in range(3)]
        return dict(kind=kind, batch=rng.randint(1, 8), nx=dims[0], ny=dims[1], nz=dims[2])
    if kind == "learned":
        dims = [8 * v for v in _grid(rng, 10, 32)]
        return dict(kind=kind, nx=dims[0], ny=dims[1], nz=dims[2], chi=chi)
    if kind == "substep":
        nx, ny, nz = _grid(rng, 16, 96)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind == "reproject":
        nx, ny, nz = _grid(rng, 24, 200)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz)
    if kind == "spike":
        nx, ny, nz = _grid(rng, 192, 384)
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, chi=4.0)
    nx, ny, nz = _grid(rng, 16, 300)
    if kind == "magnetic":
        return dict(kind=kind, nx=nx, ny=ny, nz=nz, chi=chi, warm=rng.random() < 0.5)
    return dict(kind=kind, nx=nx, ny=ny, nz=nz, jump=rng.random() < 0.5, solid=rng.random() < 0.5)


# ---------------------------------------------------------------- scenes
class Scene:
    """One case's inputs: the geometry of sfp.scenes with its random parts
    drawn from the seed, as FP64 arrays on the GPU."""

    def __init__(self, case, seed):
        self.n = (case["nx"], case["ny"], case["nz"])
        self.h = 1.0 / max(self.n)
        self.origin = tuple(0.5 - v * self.h / 2 for v in self.n)
        self.rng = np.random.default_rng(seed)
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(int(seed))

    def face_shape(self, a):
        return tuple(v + (1 if i == a else 0) for i, v in enumerate(self.n))

    def axes(self, face=None):
        """Broadcastable cell-centre (or face-centre) coordinates."""
        out = []
        for a in range(3):
            m = self.n[a] + (1 if a == face else 0)
            o = self.origin[a] + (0.0 if a == face else self.h / 2)
            shape = [1, 1, 1]
            shape[a] = m
            out.append((o + torch.arange(m, dtype=F64, device=DEV) * self.h).reshape(shape))
        return out

    def faces(self, fn):
        return [fn(a) for a in range(3)]

    def uniform(self, shape, lo, hi):
        return torch.rand(shape, dtype=F64, device=DEV, generator=self.gen) * (hi - lo) + lo

    def pool(self):
        """Distance to a drop above a pool, both moved a little by the seed."""
        X, Y, Z = self.axes()
        dx, dy, dz, dr, dp = self.rng.uniform(-0.02, 0.02, 5)
        lo = [self.origin[a] for a in range(3)]
        ext = [v * self.h for v in self.n]
        c = [lo[0] + (0.5 + dx) * ext[0], lo[1] + (0.6 + dy) * ext[1], lo[2] + (0.5 + dz) * ext[2]]
        drop = torch.sqrt((X - c[0]) ** 2 + (Y - c[1]) ** 2 + (Z - c[2]) ** 2) - (0.2 + dr) * min(ext)
        return torch.minimum(drop, Y - (lo[1] + (0.25 + dp) * ext[1])).contiguous()

    def wavy(self, modes, amp, mmax, level, shift=0.0):
        """A flat interface with random cosine modes (shift moves their phases)."""
        X, Y, Z = self.axes()
        a = self.rng.uniform(0.0, amp, modes)
        m = self.rng.integers(1, mmax + 1, modes)
        n = self.rng.integers(1, mmax + 1, modes)
        t = self.rng.uniform(0.0, 2.0 * math.pi, modes)
        s = torch.zeros((self.n[0], 1, self.n[2]), dtype=F64, device=DEV)
        out = []
        for sh in (0.0, shift):
            s = torch.zeros_like(s)
            for k in range(modes):
                s += a[k] * torch.cos(2.0 * math.pi * (int(m[k]) * X + int(n[k]) * Z) + (t[k] + sh))
            out.append((Y - (self.origin[1] + level * self.n[1] * self.h) - s).contiguous())
        return out

    def velocity(self):
        """Uniform noise in [-1, 1] smoothed by three 3x3x3 box means."""
        def one(a):
            u = self.uniform(self.face_shape(a), -1.0, 1.0)
            for _ in range(3):
                for ax in range(3):
                    lo = torch.cat([u.narrow(ax, 0, 1), u.narrow(ax, 0, u.shape[ax] - 1)], ax)
                    hi = torch.cat([u.narrow(ax, 1, u.shape[ax] - 1),
                                    u.narrow(ax, u.shape[ax] - 1, 1)], ax)
                    u = (lo + u + hi) / 3.0
            return u.contiguous()
        return self.faces(one)

    def obstacle(self, face):
        """Distance to a ball standing in the pool, at the faces of one axis,
        and its gradient's component along that axis."""
        P = self.axes(face)
        c = [self.origin[a] + f * self.n[a] * self.h for a, f in enumerate((0.35, 0.2, 0.6))]
        r = torch.sqrt(sum((P[a] - c[a]) ** 2 for a in range(3)))
        return r - 0.13 * min(self.n) * self.h, (P[face] - c[face]) / r.clamp_min(self.h)

    def fraction(self, solid):
        """Solid fraction: 1 on the box faces; with `solid`, the ball too,
        with cut faces around it."""
        def one(a):
            f = torch.zeros(self.face_shape(a), dtype=F64, device=DEV)
            if solid:
                f = (0.5 - self.obstacle(a)[0] / self.h).clamp(0.0, 1.0).contiguous()
            f.select(a, 0).fill_(1.0)
            f.select(a, self.n[a]).fill_(1.0)
            return f
        return self.faces(one)

    def zero_faces(self):
        return self.faces(lambda a: torch.zeros(self.face_shape(a), dtype=F64, device=DEV))

    def normals(self):
        """Outward normals at the faces: the ball's inside the box, the
        walls' on it."""
        def one(a):
            g = self.obstacle(a)[1].expand(self.face_shape(a)).clone()
            g.select(a, 0).fill_(1.0)
            g.select(a, self.n[a]).fill_(-1.0)
            return g
        return self.faces(one)


class State:
    """A case's context, its inputs and its output arrays."""

    def __init__(self, case, scene):
        self.case, self.scene = case, scene

    def open(self, **params):
        sc = self.scene
        self.ctx = sfp.Context(sc.n, sc.h, sc.origin, max_iters=200, **params)
        # work the caller orders before a solve goes on the context's stream
        self.stream = torch.cuda.ExternalStream(sfp.lib().sfp_stream(self.ctx.handle))


def _ptr(t):
    return None if t is None else [x.data_ptr() for x in t]


def prepare(case, seed):
    kind = case["kind"]
    if kind == "unet":
        return _prepare_unet(case, seed)
    sc = Scene(case, seed)
    s = State(case, sc)
    if kind in ("pressure", "reproject", "substep"):
        solid = kind == "substep" or bool(case.get("solid"))
        s.phi = sc.pool()
        s.fraction = sc.fraction(solid)
        s.vel0 = sc.velocity()
        s.us = sc.zero_faces()
        s.jump, s.vol_error = None, 0.0
        if solid:  # the ball moves
            s.us = sc.faces(lambda a: torch.full(sc.face_shape(a), (0.2, -0.1, 0.3)[a], dtype=F64,
                                                 device=DEV))
        if case.get("jump"):
            s.jump = sc.faces(lambda a: sc.uniform(sc.face_shape(a), -0.15, 0.15))
            s.vol_error = 0.0137
        if kind == "reproject":
            s.vel1 = sc.velocity()
            s.out1 = [torch.empty_like(v) for v in s.vel0]
            s.pressure1 = torch.empty_like(s.phi)
        s.out = [torch.empty_like(v) for v in s.vel0]
        s.pressure = torch.empty_like(s.phi)
        if kind == "substep":
            s.host = dict(phi=s.phi.cpu().numpy(), velocity=[v.cpu().numpy() for v in s.vel0],
                          fraction=[v.cpu().numpy() for v in s.fraction],
                          solid_velocity=[v.cpu().numpy() for v in s.us], jump=None, vol_error=0.0)
            s.normal_dev = sc.normals()
            s.normal = [v.cpu().numpy() for v in s.normal_dev]
            s.colvel = s.host["solid_velocity"]
        s.open()
        return s
    # the magnetic potential
    spike = kind == "spike"
    s.phi, s.phi_next = sc.wavy(64, 0.005, 12, 0.2) if spike else sc.wavy(8, 0.01, 6, 0.3, shift=0.05)
    if not case.get("warm"):
        s.phi_next = None
    s.hext = sc.faces(lambda a: torch.full(sc.face_shape(a), (0.0, 1.5 if spike else 1.0, 0.0)[a],
                                           dtype=F64, device=DEV))
    s.band = 1.5 * sc.h
    s.potential = torch.empty_like(s.phi)
    s.field = [torch.empty_like(h) for h in s.hext]
    if s.phi_next is not None:
        s.potential_next = torch.empty_like(s.phi)
        s.field_next = [torch.empty_like(h) for h in s.hext]
    s.open()
    if kind == "learned":
        weights, meta = learn.load_weights()
        s.ctx.set_network(weights)
        s.ctx.set_params(**learn.learned_params(meta))
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "unet":
        loss, grads = s.net.gradients(s.x, s.t, s.m)
        return dict(loss=loss, grads=grads)
    ctx = s.ctx
    if kind == "substep":
        vel, p, _ = ctx.projection_substep(s.host, s.normal, s.colvel, steps=6, want_pressure=True)
        return dict(velocity=vel, pressure=p)
    if kind in ("pressure", "reproject"):
        # the projection updates the velocity in place: each pass projects
        # the same advected field
        with torch.cuda.stream(s.stream):
            torch._foreach_copy_(s.out, s.vel0)
        ctx.pressure_project_device(_ptr(s.out), s.phi.data_ptr(), _ptr(s.fraction), _ptr(s.us),
                                    _ptr(s.jump), s.vol_error, s.pressure.data_ptr())
        got = dict(velocity=s.out, pressure=s.pressure)
        if kind == "reproject":
            with torch.cuda.stream(s.stream):
                torch._foreach_copy_(s.out1, s.vel1)
            ctx.pressure_project_device(_ptr(s.out1), s.phi.data_ptr(), _ptr(s.fraction), _ptr(s.us),
                                        None, 0.0, s.pressure1.data_ptr(), reproject=True)
            got.update(velocity1=s.out1, pressure1=s.pressure1)
        return got
    ctx.reset_warm_start()
    ctx.magnetic_solve_device(s.phi.data_ptr(), _ptr(s.hext), s.case["chi"], s.band,
                              s.potential.data_ptr(), _ptr(s.field))
    got = dict(potential=s.potential, field=s.field)
    if s.phi_next is not None:
        ctx.magnetic_solve_device(s.phi_next.data_ptr(), _ptr(s.hext), s.case["chi"], s.band,
                                  s.potential_next.data_ptr(), _ptr(s.field_next))
        got.update(potential_next=s.potential_next, field_next=s.field_next)
    return got


def work(case):
    """Bytes: every input array read once and every output array written
    once. Flops: the network's three convolution passes (forward, input and
    weight gradients); the solves are bound by bytes."""
    n = case["nx"] * case["ny"] * case["nz"]
    kind = case["kind"]
    if kind == "unet":
        nv = n * case["batch"]
        per = [(4, 16, 1), (16, 16, 1), (16, 32, 8), (32, 32, 8), (32, 64, 64), (64, 64, 64),
               (64, 32, 8), (32, 32, 8), (32, 16, 1), (16, 16, 1)]
        fwd = sum(2 * 27 * ci * co * nv // div for ci, co, div in per)
        return dict(bytes=4 * (4 + 1 + 1) * nv + 2 * 4 * sfp.unet_param_count(), flops=3 * fwd)
    if kind in ("pressure", "reproject", "substep"):
        per = 8 + 24 * 3 + (24 if case.get("jump") else 0) + 24 + 8  # phi, 3 face fields; velocity, p
        if kind == "reproject":
            per += 24 + 24 + 8
        if kind == "substep":
            per += 24  # normals (the collider velocity is the solid velocity)
        return dict(bytes=per * n, flops=0)
    per = 8 + 24 + 8 + 24
    if case.get("warm"):
        per += 8 + 8 + 24
    return dict(bytes=per * n, flops=0)


# ---------------------------------------------------------------- 64-bit values
EXACT_LIMIT_S = 15.0


def _lo(x, a):
    return x.narrow(a, 0, x.shape[a] - 1)


def _hi(x, a):
    return x.narrow(a, 1, x.shape[a] - 1)


def _cg(diag, cpl, b, active):
    """Diagonally preconditioned CG on diag x - sum of couplings (cpl[a] on the
    interior faces of axis a) to 1e-14, or None when it takes too long."""
    inv = torch.where(active, 1.0 / diag, torch.zeros_like(diag))

    def apply(x):
        y = diag * x
        for a in range(3):
            _hi(y, a).sub_(cpl[a] * _lo(x, a))
            _lo(y, a).sub_(cpl[a] * _hi(x, a))
        return y * active

    x = torch.zeros_like(b)
    began = time.monotonic()
    for _ in range(4):  # restarts from the true residual
        r = b * active - apply(x)
        z = inv * r
        p = z.clone()
        rz = (r * z).sum()
        bb = float((b * active).square().sum().sqrt())
        if bb == 0.0:
            return x
        for it in range(20000):
            q = apply(p)
            al = rz / (p * q).sum()
            x += al * p
            r -= al * q
            z = inv * r
            rz1 = (r * z).sum()
            p = z + (rz1 / rz) * p
            rz = rz1
            if it % 50 == 49:
                if float(r.square().sum().sqrt()) <= 1e-14 * bb:
                    break
                if time.monotonic() - began > EXACT_LIMIT_S:
                    return None
        if float((b * active - apply(x)).square().sum().sqrt()) <= 1e-12 * bb:
            return x
    return x


def _divergence(s, vel, liquid):
    div = torch.zeros_like(s.phi)
    for a in range(3):
        w = 1.0 - s.fraction[a]
        flux = w * vel[a] + (1.0 - w) * s.us[a]
        div += _lo(flux, a) - _hi(flux, a)
    return div * liquid


def _exact_projection(s, vel, jump, vol_error, system=None):
    """Velocity and pressure of one projection (and its matrix for another)."""
    liq = s.phi <= 0
    if system is None:
        diag = torch.zeros_like(s.phi)
        cpl = []
        for a in range(3):
            w = _hi(_lo(1.0 - s.fraction[a], a), a)  # interior faces
            l0, l1 = _lo(liq, a), _hi(liq, a)
            p0, p1 = _lo(s.phi, a), _hi(s.phi, a)
            th = p0 / (p0 - p1)
            both = l0 & l1
            cpl.append(torch.where(both, w, torch.zeros_like(w)))
            g0 = torch.where(l0 & ~l1, w / th.clamp_min(0.001), torch.zeros_like(w))
            g1 = torch.where(l1 & ~l0, w / (p1 / (p1 - p0)).clamp_min(0.001), torch.zeros_like(w))
            _lo(diag, a).add_(cpl[a] + g0)
            _hi(diag, a).add_(cpl[a] + g1)
        active = liq
        diag = torch.where(active & (diag != 0), diag, torch.ones_like(diag))
        system = (diag, cpl)
    diag, cpl = system
    rhs = _divergence(s, vel, liq)
    if jump is not None:
        for a in range(3):
            w = _hi(_lo(1.0 - s.fraction[a], a), a)
            j = _hi(_lo(jump[a], a), a)
            l0, l1 = _lo(liq, a), _hi(liq, a)
            p0, p1 = _lo(s.phi, a), _hi(s.phi, a)
            zero = torch.zeros_like(w)
            _lo(rhs, a).add_(torch.where(l0 & ~l1, j * w / (p0 / (p0 - p1)).clamp_min(0.001), zero))
            _hi(rhs, a).add_(torch.where(l1 & ~l0, j * w / (p1 / (p1 - p0)).clamp_min(0.001), zero))
    rhs = torch.where(liq, rhs + vol_error, torch.zeros_like(rhs))
    p = _cg(diag, cpl, rhs, liq)
    if p is None:
        return None
    out = [v.clone() for v in vel]
    for a in range(3):
        u = _hi(_lo(out[a], a), a)
        w = _hi(_lo(1.0 - s.fraction[a], a), a)
        j = torch.zeros_like(w) if jump is None else _hi(_lo(jump[a], a), a)
        l0, l1 = _lo(liq, a), _hi(liq, a)
        f0, f1 = _lo(s.phi, a), _hi(s.phi, a)
        q0, q1 = _lo(p, a), _hi(p, a)
        th = f0 / (f0 - f1)
        zero = torch.zeros_like(w)
        d = torch.where(l0 & l1, (q1 - q0) * w, zero)
        d = torch.where(l0 & ~l1, (j - q0) * w / th.clamp_min(0.001), d)
        d = torch.where(l1 & ~l0, -(j - q1) * w / (1.0 - th).clamp_min(0.001), d)
        u.sub_(d)
    return out, p, system


def _exact_potential(s, phi):
    n, chi = s.scene.n, s.case["chi"]
    diag = torch.zeros_like(phi)
    b = torch.zeros_like(phi)
    cpl = []
    for a in range(3):
        ph = (_lo(phi, a) + _hi(phi, a)) * 0.5
        t = ph / s.band
        hv = (0.5 * (1.0 + t + torch.sin(math.pi * t) / math.pi))
        hv = torch.where(t < -1, torch.zeros_like(t), torch.where(t > 1, torch.ones_like(t), hv))
        mu = 1.0 + (1.0 - hv) * chi
        cpl.append(mu)
        _lo(diag, a).add_(mu)
        _hi(diag, a).add_(mu)
        f = (mu - 1.0) * _hi(_lo(s.hext[a], a), a) * s.scene.h
        _hi(b, a).add_(f)
        _lo(b, a).sub_(f)
    active = torch.ones_like(phi, dtype=torch.bool)
    active[0, 0, 0] = False  # the pinned cell
    x = _cg(diag, cpl, b, active)
    if x is None:
        return None
    field = []
    for a in range(3):
        h = s.hext[a].clone()
        if n[a] > 1:
            _hi(_lo(h, a), a).add_((_lo(x, a) - _hi(x, a)) / s.scene.h)
        field.append(h)
    return x, field


def _exact_extrapolate(s, vel, steps):
    out = []
    for a in range(3):
        v = vel[a].clone()
        liq = s.phi <= 0
        near = torch.zeros(v.shape, dtype=torch.bool, device=v.device)
        near.narrow(a, 0, s.phi.shape[a]).logical_or_(liq)
        near.narrow(a, 1, s.phi.shape[a]).logical_or_(liq)
        ok = near & (s.fraction[a] < 1)
        for _ in range(steps):
            cnt = torch.zeros_like(v)
            tot = torch.zeros_like(v)
            okd = ok.to(F64)
            vv = torch.where(ok, v, torch.zeros_like(v))
            for c in range(3):
                _hi(cnt, c).add_(_lo(okd, c))
                _lo(cnt, c).add_(_hi(okd, c))
                _hi(tot, c).add_(_lo(vv, c))
                _lo(tot, c).add_(_hi(vv, c))
            new = torch.where(cnt > 0, tot / cnt.clamp_min(1.0), torch.zeros_like(v))
            v = torch.where(ok, v, new)
            ok = ok | (cnt > 0)
        out.append(v)
    return out


def _at_faces(grid, b, a, n):
    """The field of face grid b interpolated at the face centres of grid a."""
    v = grid
    for c in range(3):
        size = n[c] + (1 if c == a else 0)
        off = (0.0 if c == a else 0.5) - (0.0 if c == b else 0.5)
        i = torch.arange(size, device=v.device)
        lo = i if off >= 0 else i - 1
        wt = off if off >= 0 else off + 1.0
        i0 = lo.clamp(0, v.shape[c] - 1)
        i1 = (lo + 1).clamp(0, v.shape[c] - 1)
        v = v.index_select(c, i0) * (1.0 - wt) + v.index_select(c, i1) * wt
    return v


def _exact_enforce(s, vel):
    n = s.scene.n
    out = []
    for a in range(3):
        u = [_at_faces(vel[b], b, a, n) for b in range(3)]
        u0 = [_at_faces(s.us[b], b, a, n) for b in range(3)]
        m = [_at_faces(s.normal_dev[b], b, a, n) for b in range(3)]
        z = m[0] * m[0] + m[1] * m[1] + m[2] * m[2]
        r = torch.where(z > 0, z.sqrt(), torch.ones_like(z))
        m = [x / r for x in m]
        dot = sum((u[b] - u0[b]) * m[b] for b in range(3))
        out.append(torch.where(s.fraction[a] == 1.0, u[a] - dot * m[a], vel[a]))
    return out


def exact(case, seed):
    kind = case["kind"]
    if case["nx"] * case["ny"] * case["nz"] > 20_000_000:
        return None
    s = prepare(case, seed)
    if kind == "unet":
        return _exact_unet(s)
    if kind in ("pressure", "reproject", "substep"):
        got = _exact_projection(s, s.vel0, s.jump, s.vol_error)
        if got is None:
            return None
        vel, p, system = got
        if kind == "substep":
            vel = _exact_enforce(s, _exact_extrapolate(s, vel, 6))
        out = dict(velocity=vel, pressure=p)
        if kind == "reproject":
            again = _exact_projection(s, s.vel1, None, 0.0, system)
            if again is None:
                return None
            out.update(velocity1=again[0], pressure1=again[1])
        return out
    got = _exact_potential(s, s.phi)
    if got is None:
        return None
    out = dict(potential=got[0], field=got[1])
    if s.phi_next is not None:
        nxt = _exact_potential(s, s.phi_next)
        if nxt is None:
            return None
        out.update(potential_next=nxt[0], field_next=nxt[1])
    return out


# ---------------------------------------------------------------- the network
CONVS = [(8, 16), (16, 16), (16, 32), (32, 32), (32, 64), (64, 64), (64, 32), (32, 32), (32, 16), (16, 16)]


def _prepare_unet(case, seed):
    """Crops of residuals with three operator features, their targets and
    masks, and He-scaled weights, as the training program holds them."""
    rng = np.random.default_rng(seed)
    s = State(case, None)
    shape = (case["batch"], case["nx"], case["ny"], case["nz"])
    p = []
    for k, (ci, co) in enumerate(CONVS):
        fan = 27 * (4 if k == 0 else ci)
        w = rng.standard_normal((27, co, ci)) * math.sqrt(2.0 / fan)
        if k == 0:
            w[:, :, 4:] = 0.0
        p += [w.ravel(), rng.standard_normal(co) * 0.05]
    p += [rng.standard_normal(16) * 0.25, np.full(1, 0.01)]
    s.params = np.concatenate(p).astype(np.float32)
    s.x = rng.standard_normal(shape + (4,), dtype=np.float32)
    s.t = rng.standard_normal(shape, dtype=np.float32)
    s.m = (rng.random(shape, dtype=np.float32) < 0.8).astype(np.float32)
    s.net = sfp.UNet(*shape, training=True)
    s.net.set_params(s.params)
    return s


def _exact_unet(s):
    """Loss and gradients of the network in 64 bits throughout."""
    B, X, Y, Z = s.x.shape[:4]
    if B * X * Y * Z > 600_000:
        return None
    p = torch.from_numpy(s.params).to(DEV, F64).requires_grad_(True)
    ws, o = [], 0
    for ci, co in CONVS:
        w = p[o:o + 27 * ci * co].reshape(27, co, ci)
        o += 27 * ci * co
        ws.append((w, p[o:o + co]))
        o += co

    def conv(k, v):
        w, b = ws[k]
        pad = torch.nn.functional.pad(v, (0, 0, 1, 1, 1, 1, 1, 1))
        y = b
        for t in range(27):
            i, j, l = t // 9, (t // 3) % 3, t % 3
            y = y + pad[:, i:i + v.shape[1], j:j + v.shape[2], l:l + v.shape[3]] @ w[t].t()
        return torch.relu(y)

    def pool(v):
        b, x, y, z, c = v.shape
        return v.reshape(b, x // 2, 2, y // 2, 2, z // 2, 2, c).mean(dim=(2, 4, 6))

    def up(v):
        for ax in (1, 2, 3):
            v = v.repeat_interleave(2, dim=ax)
        return v

    x = torch.zeros((B, X, Y, Z, 8), dtype=F64, device=DEV)
    x[..., :4] = torch.from_numpy(s.x).to(DEV, F64)
    e0 = conv(1, conv(0, x))
    e1 = conv(3, conv(2, pool(e0)))
    e2 = conv(5, conv(4, pool(e1)))
    d1 = conv(7, conv(6, up(e2)) + e1)
    d0 = conv(9, conv(8, up(d1)) + e0)
    z = d0 @ p[o:o + 16] + p[o + 16]
    m = torch.from_numpy(s.m).to(DEV, F64)
    loss = (m * (z - torch.from_numpy(s.t).to(DEV, F64)) ** 2).sum() / m.sum()
    loss.backward()
    return dict(loss=loss.detach(), grads=p.grad)
