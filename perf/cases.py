"""Performance cases: what a program built on this package has it do, through
its public entry points, with the same results computed in plain torch.

Each kind of work has one class: `Case(case, seed)` makes the inputs from the
seed alone, `prepare` puts them into the package's fields and solvers, `run`
is one pass as a user's program writes it, `exact` gives the pass's outputs in
64 bits without the package.

  diffusion_launch  one step of the explicit diffusion loop, kernel by kernel
                    through the Launcher (the smallest calls a program makes)
  diffusion_loop    many diffusion steps in one native call
  operators         grid operators on whole fields (post-processing, user
                    kernels), plain and masked
  set_functions     set! and FunctionField evaluation (initial conditions,
                    temperature-dependent buoyancy)
  stokes            PT Stokes iterations up to a convergence check
  stokes_launch     a physical step of the viscoelastic Stokes + T example,
                    kernel by kernel through the Launcher
  mixed_cycle       FP64 residual, FP32 correction sweeps, correction added
  thermal_step      a physical step of the Stokes + T solver
  sia_forward       ice-sheet steps with the adaptive time-step rule
  sia_gradient      the gradient of an ice-sheet misfit (checkpointed adjoint)
"""
import ctypes
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "chmy.jl_amd"))

import chmy  # noqa: E402
from chmy import _lib  # noqa: E402
from chmy.sia import SIA  # noqa: E402
from chmy.stokes import MixedPTStokes, PTStokes, free_slip_batch  # noqa: E402
from chmy.stokes_thermal import StokesThermal  # noqa: E402

C, V = chmy.Center(), chmy.Vertex()
F64 = torch.float64
_ARCH = []


def arch():
    if not _ARCH:
        _ARCH.append(chmy.Arch(chmy.MI355XBackend()))
    return _ARCH[0]


def listed():
    return [
        # the reference's diffusion example at its smallest: three launches and
        # two waits a step, so what counts is the cost of a call
        {"name": "diffusion_launch_64", "kind": "diffusion_launch", "nx": 64, "ny": 64, "nz": 0, "dtype": "f64"},
        # the 256^2 diffusion workload in native steps: launch-bound
        {"name": "diffusion_loop_256", "kind": "diffusion_loop", "nx": 256, "ny": 256, "nz": 0, "dtype": "f64",
         "steps": 100},
        # derived quantities of a 3D run: divergence, speed, interpolations,
        # a Laplacian, and the masked forms of an immersed boundary
        {"name": "operators_3d", "kind": "operators", "nx": 191, "ny": 175, "nz": 167, "dtype": "f64", "masked": True},
        # initial conditions of a 3D inclusion run and a buoyancy that follows T
        {"name": "set_functions_3d", "kind": "set_functions", "nx": 160, "ny": 144, "nz": 127, "dtype": "f64"},
        # an ordinary 2D solve between two convergence checks: small launches
        {"name": "stokes2d_127", "kind": "stokes", "nx": 127, "ny": 95, "nz": 0, "iters": 65, "rhog": True,
         "exact": False},
        # the large 2D solve with scattered inclusions
        {"name": "stokes2d_2047", "kind": "stokes", "nx": 2047, "ny": 2047, "nz": 0, "iters": 41, "rhog": False,
         "exact": False},
        # the large 3D solve with a weak inclusion: the package's main path
        {"name": "stokes3d_255", "kind": "stokes", "nx": 255, "ny": 255, "nz": 255, "iters": 41, "rhog": False,
         "exact": False},
        # the 3D example's own kernel sequence, as a ported program launches it
        {"name": "stokes3d_launch", "kind": "stokes_launch", "nx": 159, "ny": 143, "nz": 127, "iters": 4,
         "eta_field": False},
        # one defect-correction cycle: FP64 residual, FP32 sweeps, bf16 forcing
        {"name": "mixed_cycle_3d", "kind": "mixed_cycle", "nx": 207, "ny": 191, "nz": 175, "inner": 40},
        # a physical step of the coupled solver, temperature in every iteration
        {"name": "thermal_step_3d", "kind": "thermal_step", "nx": 175, "ny": 159, "nz": 143, "iters": 13},
        # ice-sheet growth with the time step chosen from max(D) each step
        {"name": "sia_forward_adaptive", "kind": "sia_forward", "nx": 250, "ny": 230, "steps": 24},
        # the ice-sheet gradient at its benchmark size: 300 steps, 30 checkpoints
        {"name": "sia_gradient_512", "kind": "sia_gradient", "nx": 512, "ny": 512, "steps": 300, "ncheck": 30},
    ]


def _size(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _dims(rng, nd, lo2, hi2, lo3, hi3):
    if nd == 2:
        return {"nx": _size(rng, lo2, hi2), "ny": _size(rng, lo2, hi2), "nz": 0}
    return {"nx": _size(rng, lo3, hi3), "ny": _size(rng, lo3, hi3), "nz": _size(rng, lo3, hi3)}


def draw(rng):
    kind = rng.choice(sorted(KINDS))
    nd = rng.choice((2, 3))
    dt = rng.choice(("f64", "f64", "f32"))
    if kind == "diffusion_launch":
        return {"kind": kind, **_dims(rng, nd, 32, 1024, 16, 200), "dtype": dt}
    if kind == "diffusion_loop":
        return {"kind": kind, **_dims(rng, nd, 32, 1024, 16, 160), "dtype": dt, "steps": rng.randint(20, 150)}
    if kind == "operators":
        return {"kind": kind, **_dims(rng, nd, 64, 2047, 32, 223), "dtype": dt, "masked": rng.random() < 0.5}
    if kind == "set_functions":
        return {"kind": kind, **_dims(rng, nd, 64, 2047, 32, 191), "dtype": dt}
    if kind == "stokes":
        return {"kind": kind, **_dims(rng, nd, 48, 2047, 24, 255), "iters": rng.randint(9, 41),
                "rhog": rng.random() < 0.4, "exact": rng.random() < 0.2}
    if kind == "stokes_launch":
        return {"kind": kind, **_dims(rng, nd, 48, 1535, 24, 175), "iters": rng.randint(2, 5),
                "eta_field": rng.random() < 0.4}
    if kind == "mixed_cycle":
        return {"kind": kind, **_dims(rng, nd, 64, 1535, 32, 191), "inner": 2 * rng.randint(5, 25)}
    if kind == "thermal_step":
        return {"kind": kind, **_dims(rng, nd, 64, 1023, 32, 175), "iters": rng.randint(5, 21)}
    if kind == "sia_forward":
        return {"kind": kind, "nx": _size(rng, 48, 512), "ny": _size(rng, 48, 512), "steps": rng.randint(8, 40)}
    return {"kind": kind, "nx": _size(rng, 48, 512), "ny": _size(rng, 48, 512), "steps": rng.randint(40, 300),
            "ncheck": rng.randint(6, 30)}


# --------------------------------------------------------------- plain fields
# A plain field is a torch array over Chmy's padded storage (x fastest, array
# dims reversed): logical index i of a dim sits at i + 1, with 2 points beyond
# the interior on each side.

DEV = torch.device("cuda" if torch.cuda.is_available() else "cpu")
TYPES = {"f64": torch.float64, "f32": torch.float32}


class Geometry:
    def __init__(self, dims, origin, extent):
        self.n, self.nd = tuple(dims), len(dims)
        self.o, self.L = tuple(origin), tuple(extent)
        self.h = tuple(e / n for e, n in zip(extent, dims))
        self.ih = tuple(1.0 / s for s in self.h)

    def grid(self):
        return chmy.UniformGrid(arch(), origin=self.o, extent=self.L, dims=self.n)

    def zeros(self, loc):
        return torch.zeros(tuple(n + l + 4 for n, l in zip(self.n, loc))[::-1], dtype=F64, device=DEV)

    def coords(self, loc):
        """Coordinates of every stored point, one broadcastable array a dim."""
        out = []
        for d in range(self.nd):
            i = torch.arange(-1, self.n[d] + loc[d] + 3, dtype=F64, device=DEV)
            x = (i - 1.0) * self.h[d] + (self.o[d] + (0.0 if loc[d] else 0.5 * self.h[d]))
            shape = [1] * self.nd
            shape[self.nd - 1 - d] = -1
            out.append(x.reshape(shape))
        return out

    def box(self, a, *shift):
        """View of `a` at I + shift for I in the Launcher box [0, n+1]."""
        sl = tuple(slice(1 + s, 1 + s + n + 2) for s, n in zip(shift or (0,) * self.nd, self.n))
        return a[sl[::-1]]

    def inner(self, a, loc):
        """The interior, x first, as interior(f) gives it."""
        sl = tuple(slice(2, 2 + n + l) for n, l in zip(self.n, loc))
        return a[sl[::-1]].permute(*reversed(range(self.nd)))

    def unit(self, d, s=1):
        e = [0] * self.nd
        e[d] = s
        return tuple(e)


def center(nd):
    return (0,) * nd


def vloc(d, nd):
    return tuple(1 if q == d else 0 for q in range(nd))


def tlocs(nd):
    if nd == 2:
        return [(0, 0), (0, 0), (1, 1)]
    return [(0, 0, 0)] * 3 + [(1, 1, 0), (1, 0, 1), (0, 1, 1)]


def geometry(case, origin=-0.5, extent=1.0):
    dims = (case["nx"], case["ny"]) + ((case["nz"],) if case["nz"] else ())
    return Geometry(dims, (origin,) * len(dims), (extent,) * len(dims))


def generator(seed):
    return np.random.default_rng(1000003 + int(seed))


def smooth(geo, loc, rng, amp=1.0, modes=3):
    """A seeded sum of products of cosines over the whole storage."""
    xs = geo.coords(loc)
    out = geo.zeros(loc)
    for _ in range(modes):
        term = amp * rng.uniform(0.3, 1.0)
        for d, x in enumerate(xs):
            k = 2.0 * math.pi * rng.uniform(0.3, 2.5) / geo.L[d]
            term = term * torch.cos(k * x + rng.uniform(0.0, 2.0 * math.pi))
        out += term
    return out


def rounded(a, dtype):
    return a.to(dtype).to(F64)


def put(field, a):
    field.data.copy_(a)


def filled(geo, loc, a, dtype=F64):
    g = geo.grid() if isinstance(geo, Geometry) else geo
    f = chmy.Field(arch(), g, tuple(V if l else C for l in loc), dtype)
    put(f, a)
    return f


def bc_rule(geo, a, loc, d, kind, left=0.0, right=0.0):
    """One dim of a first-order batch on `a`, tangential range 0..n+2."""
    m = geo.n[d] + loc[d]

    def plane(i):
        sl = [slice(1, geo.n[q] + 4) for q in range(geo.nd)]
        sl[d] = i + 1
        return tuple(sl[::-1])
    if kind == "dirichlet" and loc[d]:
        a[plane(1)] = left
        a[plane(m)] = right
    elif kind == "dirichlet":
        a[plane(0)] = 2.0 * left - a[plane(1)]
        a[plane(m + 1)] = 2.0 * right - a[plane(m)]
    else:
        a[plane(0)] = a[plane(1)] - geo.h[d] * left
        a[plane(m + 1)] = a[plane(m)] + geo.h[d] * right


def neumann(geo, a):
    for d in reversed(range(geo.nd)):
        bc_rule(geo, a, center(geo.nd), d, "neumann")


def free_slip(geo, Vs, values):
    for d in reversed(range(geo.nd)):
        for c, v in enumerate(Vs):
            if c == d:
                bc_rule(geo, v, vloc(c, geo.nd), d, "dirichlet", *values[c])
            else:
                bc_rule(geo, v, vloc(c, geo.nd), d, "neumann")


def shear(nd, rate=1.0):
    vals = [(0.0, 0.0)] * nd
    vals[0], vals[nd - 1] = (rate, -rate), (-rate, rate)
    return vals


def knots(geo, a, d, vertex):
    """(left, right) of `a` along d over the box: (I-e, I) of a Center dim,
    (I, I+e) of a Vertex dim."""
    if vertex:
        return geo.box(a), geo.box(a, *geo.unit(d))
    return geo.box(a, *geo.unit(d, -1)), geo.box(a)


def ddx(geo, a, d, vertex):
    lo, hi = knots(geo, a, d, vertex)
    return (hi - lo) * geo.ih[d]


def to_edges(geo, a, d, e):
    """A Center array at the edges with Vertex dims d and e, over the box."""
    m1, m2 = geo.unit(d, -1), geo.unit(e, -1)
    both = tuple(p + q for p, q in zip(m1, m2))
    return 0.25 * (geo.box(a) + geo.box(a, *m1) + geo.box(a, *m2) + geo.box(a, *both))


def edges_of(nd):
    return [(0, 1)] if nd == 2 else [(0, 1), (0, 2), (1, 2)]


def strain(geo, Vs):
    """Normal strain rates, edge strain rates and divergence over the box."""
    e = [ddx(geo, Vs[d], d, True) for d in range(geo.nd)]
    s = [0.5 * (ddx(geo, Vs[p], q, False) + ddx(geo, Vs[q], p, False)) for p, q in edges_of(geo.nd)]
    return e, s, sum(e[1:], e[0])


def force(geo, Pr, tau, rhog):
    """div(tau) - grad(Pr) - rho g per velocity component over the box."""
    nd, out = geo.nd, []
    for d in range(nd):
        r = -ddx(geo, Pr, d, False) + ddx(geo, tau[d], d, False)
        for k, (p, q) in enumerate(edges_of(nd)):
            if d in (p, q):
                r = r + ddx(geo, tau[nd + k], q if d == p else p, True)
        if rhog is not None and d == nd - 1:
            r = r - geo.box(rhog)
        out.append(r)
    return out


class PlainStokes:
    """The PT iteration in whole-array torch: update_stress!, update_velocity!
    and the free-slip batch, with a constant or a Center viscosity."""

    def __init__(self, geo, V_, tau, Pr, tau_old, values, *, eta, dt, G=1.0, rhog=None, f_V=None, f_P=None):
        self.geo, self.V, self.tau, self.Pr, self.tau_old = geo, V_, tau, Pr, tau_old
        self.values, self.G, self.rhog, self.f_V, self.f_P = values, G, rhog, f_V, f_P
        nd = geo.nd
        lt = min(geo.L) / (2.3 * math.pi)
        vdt = min(geo.h) / math.sqrt(nd * 1.1)
        th = lt * (0.5 + 4.0 / 3.0) / vdt
        self.dr, self.nu, self.dPr = 1.0 / (th + 1.0), vdt * lt, 0.5 / th
        self.eta = eta
        self.set_dt(dt)

    def set_dt(self, dt):
        self.dt, geo, nd = dt, self.geo, self.geo.nd
        ve = lambda x: 1.0 / (1.0 / x + 1.0 / (self.G * dt))  # noqa: E731
        if not torch.is_tensor(self.eta):
            self.etas = [self.eta] * len(self.tau)
            self.eve_c, self.eves, self.eve_v = ve(self.eta), [ve(self.eta)] * len(self.tau), [ve(self.eta)] * nd
            return
        self.etas = [geo.box(self.eta)] * nd + [to_edges(geo, self.eta, p, q) for p, q in edges_of(nd)]
        self.eves = [ve(x) for x in self.etas]
        self.eve_c = self.eves[0]
        ml = maxloc(geo, self.eta)
        self.eve_v = []
        for d in range(nd):
            lo, hi = knots(geo, ml, d, False)
            self.eve_v.append(ve(torch.maximum(lo, hi)))

    def residual_tau(self):
        """R_tau of the current state and the divergence, over the box."""
        geo, nd, Gdt = self.geo, self.geo.nd, self.G * self.dt
        e, s, dv = strain(geo, self.V)
        out = []
        for c, rate in enumerate([x - dv / 3.0 for x in e] + s):
            t = geo.box(self.tau[c])
            out.append(-(t - geo.box(self.tau_old[c])) / Gdt - t / self.etas[c] + 2.0 * rate)
        return out, dv

    def iterate(self, n):
        """n iterations; the last one's divergence and r_V over the box."""
        geo = self.geo
        for _ in range(n):
            r, dv = self.residual_tau()
            src = dv if self.f_P is None else dv - geo.box(self.f_P)
            geo.box(self.Pr).sub_(src * self.eve_c * self.dPr)
            for c, x in enumerate(r):
                geo.box(self.tau[c]).add_(x * self.eves[c] * self.dr)
            rV = force(geo, self.Pr, self.tau, self.rhog)
            if self.f_V is not None:
                rV = [x + geo.box(f) for x, f in zip(rV, self.f_V)]
            for d in range(geo.nd):
                geo.box(self.V[d]).add_(rV[d] * self.nu / self.eve_v[d])
            free_slip(geo, self.V, self.values)
        return dv, rV


def maxloc(geo, a):
    """max over the 3^N cell neighbourhood, on the box (zero elsewhere)."""
    out = torch.zeros_like(a)
    m = geo.box(a).clone()
    for k in range(3 ** geo.nd):
        s = tuple(k // 3 ** d % 3 - 1 for d in range(geo.nd))
        m = torch.maximum(m, geo.box(a, *s))
    geo.box(out).copy_(m)
    return out


def residual_fields(geo, dv, rV):
    """divV and r_V as stored over the box, r_V's boundary vertices zeroed,
    their interiors and largest magnitudes."""
    nd = geo.nd
    a = geo.zeros(center(nd))
    geo.box(a).copy_(dv)
    outs = [geo.inner(a, center(nd))]
    for d in range(nd):
        r = geo.zeros(vloc(d, nd))
        geo.box(r).copy_(rV[d])
        bc_rule(geo, r, vloc(d, nd), d, "dirichlet")
        outs.append(geo.inner(r, vloc(d, nd)))
    return outs, [float(x.abs().max()) for x in outs]


def interiors(geo, arrays, locs):
    return [geo.inner(a, l) for a, l in zip(arrays, locs)]


def state_locs(nd):
    return [vloc(d, nd) for d in range(nd)] + tlocs(nd) + [center(nd)]


def dt_diffusion(geo):
    return min(geo.h) ** 2 / 1e-4 / geo.nd / 2.1


def inclusions(geo, rng):
    """Viscosity of seeded round inclusions, 1e-3 to 1e3 times the background
    in 2D, one weak sphere near the middle in 3D, on the whole storage."""
    xs = geo.coords(center(geo.nd))
    eta = geo.zeros(center(geo.nd)) + 1.0
    for _ in range(32 if geo.nd == 2 else 1):
        if geo.nd == 2:
            c, r, v = rng.uniform(-0.5, 0.5, 2), rng.uniform(0.01, 0.04), 10.0 ** rng.uniform(-3.0, 3.0)
        else:
            c, r, v = rng.uniform(-0.05, 0.05, 3), rng.uniform(0.08, 0.12), 10.0 ** rng.uniform(-3.2, -2.8)
        r2 = sum((x - float(q)) ** 2 for x, q in zip(xs, c))
        eta = torch.where(r2 < r * r, torch.full_like(eta, v), eta)
    if geo.nd == 3:
        eta = eta * torch.exp(-0.1 * torch.exp(-sum(x * x for x in xs) / 0.05 ** 2))
    return eta


def flow(geo, rng, rate=1.0):
    """Pure shear with a smooth perturbation, boundary values applied; smooth
    stresses and pressure, as a solve under way holds them (scaled by rate)."""
    nd = geo.nd
    vs = []
    for d in range(nd):
        a = smooth(geo, vloc(d, nd), rng, 0.05)
        if d in (0, nd - 1):
            a = a + (-2.0 if d == 0 else 2.0) * geo.coords(vloc(d, nd))[d]
        vs.append(a.contiguous())
        vs[-1] *= rate
    free_slip(geo, vs, shear(nd, rate))
    tau = [smooth(geo, l, rng, 0.3 * rate) for l in tlocs(nd)]
    return vs, tau, smooth(geo, center(nd), rng, 0.3 * rate)


def load_state(S, vs, tau, pr):
    for f, a in zip(list(S.V) + list(S.tau) + [S.Pr], vs + tau + [pr]):
        put(f, a)
    S.sync_buffers()


def views(fields):
    return [f.interior() for f in fields]


def cells(case):
    return case["nx"] * case["ny"] * max(1, case.get("nz") or 1)


# --------------------------------------------------------------- the kinds

class DiffusionLaunch:
    def __init__(self, case, seed):
        self.geo, self.dtype = geometry(case, -1.0, 2.0), TYPES[case["dtype"]]
        rng, geo = generator(seed), self.geo
        xs = geo.coords(center(geo.nd))
        a = smooth(geo, center(geo.nd), rng, 0.1)
        for _ in range(4):
            r2 = sum((x - rng.uniform(-0.7, 0.7)) ** 2 for x in xs)
            a = a + rng.uniform(0.5, 2.0) * torch.exp(-r2 / rng.uniform(0.05, 0.2) ** 2)
        neumann(geo, a)
        self.C = rounded(a, self.dtype)
        self.chi, self.steps = 1.0, case.get("steps", 1)
        self.dt = min(geo.h) ** 2 / self.chi / geo.nd / 2.1

    def prepare(self):
        g = self.geo.grid()
        self.g, self.launch = g, chmy.Launcher(arch(), g)
        self.Cf = filled(g, center(g.nd), self.C, self.dtype)
        self.q = chmy.VectorField(arch(), g, self.dtype)
        self.bc = chmy.batch(g, (self.Cf, chmy.Neumann()))

    def run(self):
        k = chmy.kernels
        self.launch(arch(), self.g, (k.compute_q, (self.q, self.Cf, self.chi, self.g)))
        self.launch(arch(), self.g, (k.update_C, (self.Cf, self.q, self.dt, self.g)), bc=self.bc)
        return views([self.Cf] + list(self.q))

    def exact(self):
        geo, nd = self.geo, self.geo.nd
        q = [geo.zeros(vloc(d, nd)) for d in range(nd)]
        chi, dt = (float(torch.tensor(x, dtype=self.dtype)) for x in (self.chi, self.dt))
        for _ in range(self.steps):
            for d in range(nd):
                geo.box(q[d]).copy_(-chi * ddx(geo, self.C, d, False))
            geo.box(self.C).sub_(dt * sum(ddx(geo, q[d], d, True) for d in range(nd)))
            neumann(geo, self.C)
        return interiors(geo, [self.C] + q, [center(nd)] + [vloc(d, nd) for d in range(nd)])

    @staticmethod
    def work(case):
        nd, size = (3 if case["nz"] else 2), 8 if case["dtype"] == "f64" else 4
        return {"bytes": cells(case) * size * (2 + nd), "flops": cells(case) * case.get("steps", 1) * (6 * nd + 2)}


class DiffusionLoop(DiffusionLaunch):
    def prepare(self):
        super().prepare()
        g, nd = self.g, self.g.nd
        self.bufs, self.at = (self.Cf, filled(g, center(nd), self.C, self.dtype)), ctypes.c_int(0)
        self.counts = (ctypes.c_int32 * 6)(*[1 if k < 2 * nd else 0 for k in range(6)])
        self.rules = (_lib.ChmyBC * (2 * nd))(*[_lib.ChmyBC(_lib.NEUMANN, _lib.VALUE_ZERO, 0.0, None)
                                                for _ in range(2 * nd)])

    def run(self):
        g, ref = self.g, ctypes.byref
        q = (_lib.ChmyField * g.nd)(*[f.desc() for f in self.q])
        _lib.call("chmy_diffusion_iterate", ref(g.desc()), ref(self.bufs[0].desc()), ref(self.bufs[1].desc()), q,
                  self.counts, self.rules, self.chi, self.dt, self.steps, ref(self.at), chmy.current_stream())
        return views([self.bufs[self.at.value]] + list(self.q))


class Operators:
    def __init__(self, case, seed):
        self.geo, self.dtype, self.masked = geometry(case), TYPES[case["dtype"]], case["masked"]
        rng, geo, nd = generator(seed), self.geo, self.geo.nd
        keep = lambda a: rounded(a, self.dtype)  # noqa: E731
        self.V = [keep(smooth(geo, vloc(d, nd), rng)) for d in range(nd)]
        self.eloc = tlocs(nd)[nd]
        self.txy = keep(smooth(geo, self.eloc, rng))
        self.T = keep(smooth(geo, center(nd), rng))
        self.eta = keep(torch.exp(smooth(geo, center(nd), rng)))
        self.mid, self.rad = rng.uniform(-0.1, 0.1, nd), rng.uniform(0.15, 0.3)

    def mask(self, loc):
        """1 outside an immersed ball, 0 inside."""
        r2 = sum((x - float(c)) ** 2 for x, c in zip(self.geo.coords(loc), self.mid))
        return (r2 > self.rad ** 2).to(F64)

    def prepare(self):
        g, nd, dt = self.geo.grid(), self.geo.nd, self.dtype
        self.g, self.launch = g, chmy.Launcher(arch(), g)
        names = g.axes_names()
        new = lambda loc: chmy.Field(arch(), g, tuple(V if l else C for l in loc), dt)  # noqa: E731
        Vf = chmy.VectorField(arch(), g, dt)
        for f, a in zip(Vf, self.V):
            put(f, a)
        txy, T = filled(g, self.eloc, self.txy, dt), filled(g, center(nd), self.T, dt)
        eta, k = filled(g, center(nd), self.eta, dt), chmy.kernels
        c, e, last = center(nd), self.eloc, len(names) - 1
        self.todo = [(k.divg, new(c), (Vf,)), (k.vmag, new(c), (Vf,)), (k.lerp, new(c), (txy,)),
                     (k.hlerp, new(e), (eta,)), (k.partial, new(vloc(0, nd)), (T, 0)), (k.lapl, new(c), (T,))]
        if self.masked:
            w = chmy.FieldMask(arch(), g, dt)
            for f in w:
                put(f, self.mask(tuple(l.code for l in f.loc)))
            self.todo += [(k.divg, new(c), (Vf, w)), (k.partial, new(vloc(last, nd)), (T, w, last)),
                          (k.divg_grad, new(c), (T, eta, w))]

    def run(self):
        for kernel, dst, args in self.todo:
            self.launch(arch(), self.g, (kernel, (dst, *args, self.g)))
        return views([dst for _, dst, _ in self.todo])

    def exact(self):
        geo, nd = self.geo, self.geo.nd
        c, last = center(nd), nd - 1
        ih = [float(torch.tensor(x, dtype=self.dtype)) for x in geo.ih]

        def whole(box, loc):
            a = geo.zeros(loc)
            geo.box(a).copy_(box)
            return geo.inner(a, loc)

        def diff(a, d, vertex, at=None):
            sh = at or (0,) * nd
            e = geo.unit(d, 1 if vertex else -1)
            other = geo.box(a, *[p + q for p, q in zip(sh, e)])
            here = geo.box(a, *sh)
            return ((other - here) if vertex else (here - other)) * ih[d]

        def mean(a, dims, sign):
            """Average of the 2^m knots over dims, at I and I + sign e."""
            out = 0.0
            for q in range(1 << len(dims)):
                s = [0] * nd
                for b, d in enumerate(dims):
                    s[d] = sign if q >> b & 1 else 0
                out = out + geo.box(a, *s) / (1 << len(dims))
            return out

        def divergence(vs):
            return sum(diff(v, d, True) for d, v in enumerate(vs))

        def laplacian(a, k=None):
            out = 0.0
            for d in range(nd):
                e = geo.unit(d)
                hi, lo = diff(a, d, False, e), diff(a, d, False)
                if k is not None:
                    here, up, dn = geo.box(k), geo.box(k, *e), geo.box(k, *geo.unit(d, -1))
                    hi, lo = hi * (0.5 * (here + up)), lo * (0.5 * (dn + here))
                out = out + (hi - lo) * ih[d]
            return out

        ed = [d for d in range(nd) if self.eloc[d]]
        speed = sum(mean(v, [d], 1) ** 2 for d, v in enumerate(self.V)).sqrt()
        outs = [whole(divergence(self.V), c), whole(speed, c), whole(mean(self.txy, ed, 1), c),
                whole(1.0 / mean(1.0 / self.eta, ed, -1), self.eloc),
                whole(diff(self.T, 0, False), vloc(0, nd)), whole(laplacian(self.T), c)]
        if self.masked:
            T = self.T * self.mask(c)
            outs += [whole(divergence([v * self.mask(vloc(d, nd)) for d, v in enumerate(self.V)]), c),
                     whole(diff(T, last, False), vloc(last, nd)), whole(laplacian(T, self.eta), c)]
        return outs

    @staticmethod
    def work(case):
        nd, size = (3 if case["nz"] else 2), 8 if case["dtype"] == "f64" else 4
        arrays = (nd + 1) + (nd + 1) + 2 + 2 + 2 + 2 + ((2 * nd + 1) + 3 + 4 if case["masked"] else 0)
        return {"bytes": cells(case) * size * arrays, "flops": cells(case) * (30 * nd)}


def viscosity_of(*args):
    """Viscosity of two inclusions in a background that weakens with a warm
    spot; coordinates first, then (c0, r0, v0, c1, r1, v1) with one centre
    coordinate a dim."""
    nd = (len(args) - 4) // 3
    xs, c0, (r0, v0), c1, (r1, v1) = (args[:nd], args[nd:2 * nd], args[2 * nd:2 * nd + 2],
                                      args[2 * nd + 2:3 * nd + 2], args[3 * nd + 2:])
    d0 = sum(((x - c) ** 2 for x, c in zip(xs[1:], c0[1:])), (xs[0] - c0[0]) ** 2)
    d1 = sum(((x - c) ** 2 for x, c in zip(xs[1:], c1[1:])), (xs[0] - c1[0]) ** 2)
    return chmy.ifelse(d0 < r0 ** 2, v0, chmy.ifelse(d1 < r1 ** 2, v1, 1.0)) * np.exp(-0.1 * np.exp(-d0 / 0.01))


def temperature_of(*args):
    """A warm blob on a linear profile along the last dim."""
    nd = (len(args) - 2) // 2
    xs, c, width, amp = args[:nd], args[nd:2 * nd], args[2 * nd], args[2 * nd + 1]
    r2 = sum(((x - p) ** 2 for x, p in zip(xs[1:], c[1:])), (xs[0] - c[0]) ** 2)
    return amp * np.exp(-r2 / width ** 2) + 0.5 * (1.0 - 2.0 * xs[-1])


def buoyancy_of(grid, loc, *args):
    """rho g of the temperature averaged to the last velocity component."""
    idx, (T, rg, alpha) = args[:-3], args[-3:]
    down = tuple(i - 1 if d == len(idx) - 1 else i for d, i in enumerate(idx))
    return rg * (1.0 - alpha * (0.5 * (T[down] + T[idx])))


class SetFunctions:
    def __init__(self, case, seed):
        self.geo, self.dtype = geometry(case), TYPES[case["dtype"]]
        rng, nd = generator(seed), self.geo.nd
        ball = lambda: tuple(float(x) for x in rng.uniform(-0.3, 0.3, nd)) + (  # noqa: E731
            float(rng.uniform(0.05, 0.2)), float(10.0 ** rng.uniform(-3, 3)))
        self.eta_par = ball() + ball()
        self.T_par = tuple(float(x) for x in rng.uniform(-0.2, 0.2, nd)) + (float(rng.uniform(0.05, 0.2)),
                                                                          float(rng.uniform(0.5, 2.0)))
        self.rg, self.alpha = float(rng.uniform(0.5, 2.0)), float(rng.uniform(0.01, 0.2))

    def prepare(self):
        g, nd = self.geo.grid(), self.geo.nd
        self.g = g
        self.eta, self.T = (chmy.Field(arch(), g, C, self.dtype) for _ in range(2))

    def run(self):
        g = self.g
        chmy.set_(self.eta, viscosity_of, g, parameters=self.eta_par)
        chmy.set_(self.T, temperature_of, g, parameters=self.T_par)
        rhog = chmy.FunctionField(buoyancy_of, g, chmy.vector_location(g.nd - 1, g.nd), discrete=True,
                                  parameters=(self.T, self.rg, self.alpha))
        return views([self.eta, self.T, rhog.materialize(arch(), self.dtype)])

    def exact(self):
        geo, nd, c = self.geo, self.geo.nd, center(self.geo.nd)
        xs = [x.cpu().numpy() for x in geo.coords(c)]
        eta = torch.from_numpy(viscosity_of(*xs, *self.eta_par)).to(DEV)
        T = geo.zeros(c)
        geo.inner(T, c).copy_(geo.inner(torch.from_numpy(temperature_of(*xs, *self.T_par)).to(DEV), c))
        T = rounded(T, self.dtype)
        r = geo.zeros(vloc(nd - 1, nd))
        lo, hi = knots(geo, T, nd - 1, False)
        geo.box(r).copy_(self.rg * (1.0 - self.alpha * (0.5 * (lo + hi))))
        return [geo.inner(eta, c), geo.inner(T, c), geo.inner(r, vloc(nd - 1, nd))]

    @staticmethod
    def work(case):
        nd, size = (3 if case["nz"] else 2), 8 if case["dtype"] == "f64" else 4
        return {"bytes": cells(case) * size * 4, "flops": cells(case) * (12 * nd + 40)}


class Stokes:
    def __init__(self, case, seed):
        self.case, self.geo = case, geometry(case)
        rng, geo, nd = generator(seed), self.geo, self.geo.nd
        self.eta = inclusions(geo, rng)
        self.V, self.tau, self.Pr = flow(geo, rng)
        self.told = [smooth(geo, l, rng, 0.2, modes=2) for l in tlocs(nd)]
        self.rhog = smooth(geo, vloc(nd - 1, nd), rng) if case["rhog"] else None

    def prepare(self):
        geo = self.geo
        g = geo.grid()
        rhog = None if self.rhog is None else filled(g, vloc(geo.nd - 1, geo.nd), self.rhog)
        self.S = PTStokes(arch(), g, eta_field=self.eta.cpu().numpy(), G=1.0, dt=dt_diffusion(geo),
                          normal_values=dict(enumerate(shear(geo.nd))), rhog=rhog, exact=self.case["exact"])
        load_state(self.S, self.V, self.tau, self.Pr)
        for f, a in zip(self.S.tau_old, self.told):
            put(f, a)

    def run(self):
        S = self.S
        S.iterate(self.case["iters"], residual_last=True)
        err = S.residual()
        return [views(list(S.V) + list(S.tau) + [S.Pr]), views([S.divV] + list(S.r_V)), err]

    def exact(self):
        geo = self.geo
        P = PlainStokes(geo, self.V, self.tau, self.Pr, self.told, shear(geo.nd), eta=self.eta,
                        dt=dt_diffusion(geo), rhog=self.rhog)
        outs, err = residual_fields(geo, *P.iterate(self.case["iters"]))
        return [interiors(geo, P.V + P.tau + [P.Pr], state_locs(geo.nd)), outs, err]

    @staticmethod
    def work(case):
        # V, tau, Pr read and written once, tau_old and eta read, divV and r_V written
        nd, nt = (3, 6) if case["nz"] else (2, 3)
        arrays = 2 * (nd + nt + 1) + nt + 1 + (1 + nd) + (1 if case["rhog"] else 0)
        return {"bytes": cells(case) * 8 * arrays, "flops": cells(case) * case["iters"] * (150 if nd == 3 else 75)}


class SlowFlow:
    """A slow Stokes + T flow: a physical step is near the Maxwell time, so
    step after step of a few PT iterations each stays bounded."""
    ETA, G, LAM, RATE = 1.0, 1.0, 1e-9, 1e-4


class StokesLaunch(SlowFlow):
    def __init__(self, case, seed):
        self.case, self.geo = case, geometry(case)
        rng, geo, nd = generator(seed), self.geo, self.geo.nd
        self.V, self.tau, self.Pr = flow(geo, rng, self.RATE)
        self.eta = self.ETA * torch.exp(smooth(geo, center(nd), rng)) if case["eta_field"] else self.ETA
        self.T = smooth(geo, center(nd), rng) + 2.0
        neumann(geo, self.T)
        self.rhog = smooth(geo, vloc(nd - 1, nd), rng, 10.0 * self.RATE)
        self.dt = 0.1 * min(geo.h) / self.RATE / nd / 2.1

    def prepare(self):
        geo, a = self.geo, arch()
        g = geo.grid()
        nd = g.nd
        self.g, self.launch = g, chmy.Launcher(a, g)
        self.Vf, self.tauf = chmy.VectorField(a, g), chmy.TensorField(a, g)
        self.Prf, self.Tf, self.Told = (chmy.Field(a, g, C) for _ in range(3))
        self.told, self.rV, self.qT = chmy.TensorField(a, g), chmy.VectorField(a, g), chmy.VectorField(a, g)
        self.dV = chmy.Field(a, g, C)
        for f, x in zip(list(self.Vf) + list(self.tauf) + [self.Prf, self.Tf], self.V + self.tau + [self.Pr, self.T]):
            put(f, x)
        self.rg = filled(g, vloc(nd - 1, nd), self.rhog)
        self.par = PlainStokes(geo, self.V, self.tau, self.Pr, self.tau, shear(nd, self.RATE), eta=self.ETA,
                               dt=self.dt, G=self.G)
        self.etaf = self.ml = None
        if self.case["eta_field"]:
            self.etaf = filled(g, center(nd), self.eta)
            self.ml = chmy.Field(a, g, C)
            self.launch(a, g, (chmy.kernels.maxloc, (self.ml, self.etaf)))
        self.Vbc = free_slip_batch(g, self.Vf, dict(enumerate(shear(nd, self.RATE))))
        self.Tbc = chmy.batch(g, (self.Tf, chmy.Neumann()))

    def run(self):
        g, k, a, p, L = self.g, chmy.kernels, arch(), self.par, self.launch
        L(a, g, (k.update_old, (self.Tf, self.tauf, self.Told, self.told)))
        for _ in range(self.case["iters"]):
            L(a, g, (k.update_stress, (self.tauf, self.Prf, self.dV, self.Vf, self.told,
                                       self.ETA if self.etaf is None else self.etaf, p.eve_c, self.G, self.dt, p.dPr,
                                       p.dr, g)))
            if self.etaf is None:
                L(a, g, (k.update_velocity, (self.Vf, self.rV, self.Prf, self.tauf, self.rg, p.eve_c, p.nu, g)),
                  bc=self.Vbc)
            else:
                L(a, g, (k.update_velocity_visc, (self.Vf, self.rV, self.Prf, self.tauf, self.rg, self.ml, self.G,
                                                  self.dt, p.nu, g)), bc=self.Vbc)
            L(a, g, (k.update_thermal_flux, (self.qT, self.Tf, self.Vf, self.LAM, g)))
            L(a, g, (k.update_thermal, (self.Tf, self.Told, self.qT, self.dt, g)), bc=self.Tbc)
        return [views(list(self.Vf) + list(self.tauf) + [self.Prf]), views([self.Tf] + list(self.qT)),
                views([self.dV] + list(self.rV))]

    def exact(self):
        geo, nd = self.geo, self.geo.nd
        told, Told = [t.clone() for t in self.tau], self.T.clone()
        P = PlainStokes(geo, self.V, self.tau, self.Pr, told, shear(nd, self.RATE), eta=self.eta, dt=self.dt, G=self.G,
                        rhog=self.rhog)
        q = [geo.zeros(vloc(d, nd)) for d in range(nd)]
        for _ in range(self.case["iters"]):
            dv, rV = P.iterate(1)
            plain_thermal(geo, self.T, Told, q, P.V, self.LAM, self.dt)
        res = [geo.zeros(center(nd))] + [geo.zeros(vloc(d, nd)) for d in range(nd)]
        for x, y in zip(res, [dv] + rV):
            geo.box(x).copy_(y)
        locs = [center(nd)] + [vloc(d, nd) for d in range(nd)]
        return [interiors(geo, P.V + P.tau + [P.Pr], state_locs(nd)), interiors(geo, [self.T] + q, locs),
                interiors(geo, res, locs)]

    @staticmethod
    def work(case):
        nd, nt = (3, 6) if case["nz"] else (2, 3)
        arrays = 2 * (nd + nt + 2) + nt + 1 + (1 + nd) + nd + 1 + (1 if case["eta_field"] else 0)
        return {"bytes": cells(case) * 8 * arrays, "flops": cells(case) * case["iters"] * (180 if nd == 3 else 90)}


def plain_thermal(geo, T, Told, q, Vs, lam, dt):
    """update_thermal_flux!, update_thermal! and the Neumann batch on T."""
    for d in range(geo.nd):
        lo, hi = knots(geo, T, d, False)
        v = geo.box(Vs[d])
        geo.box(q[d]).copy_(-lam * (hi - lo) * geo.ih[d] + v.clamp(min=0.0) * lo + v.clamp(max=0.0) * hi)
    geo.box(T).copy_(geo.box(Told) - dt * sum(ddx(geo, q[d], d, True) for d in range(geo.nd)))
    neumann(geo, T)


class MixedCycle:
    def __init__(self, case, seed):
        self.case, self.geo = case, geometry(case)
        rng, geo = generator(seed), self.geo
        self.eta = inclusions(geo, rng)
        self.V, self.tau, self.Pr = flow(geo, rng)

    def prepare(self):
        geo = self.geo
        self.M = MixedPTStokes(arch(), geo.grid(), eta_field=self.eta.cpu().numpy(), G=1.0, dt=dt_diffusion(geo),
                               normal_values=dict(enumerate(shear(geo.nd))), inner=self.case["inner"])
        load_state(self.M.x, self.V, self.tau, self.Pr)

    def run(self):
        M = self.M
        err = M.refresh()
        M.cycle()
        return [views(list(M.x.V) + list(M.x.tau) + [M.x.Pr]), err]

    def exact(self):
        geo, nd, dt = self.geo, self.geo.nd, dt_diffusion(self.geo)
        zeros = lambda locs: [geo.zeros(l) for l in locs]  # noqa: E731
        x = PlainStokes(geo, self.V, self.tau, self.Pr, zeros(tlocs(nd)), shear(nd), eta=self.eta, dt=dt)
        r, dv = x.residual_tau()
        rV = force(geo, x.Pr, x.tau, None)
        _, err = residual_fields(geo, dv, rV)
        told, fV, fP = zeros(tlocs(nd)), zeros([vloc(d, nd) for d in range(nd)]), geo.zeros(center(nd))
        for a, b in zip(told + fV + [fP], [dt * t for t in r] + rV + [-dv]):
            geo.box(a).copy_(b)
        err.append(max(float(geo.inner(a, l).abs().max()) for a, l in zip(told, tlocs(nd))) / dt)
        del r, rV
        d = PlainStokes(geo, zeros([vloc(d, nd) for d in range(nd)]), zeros(tlocs(nd)), geo.zeros(center(nd)), told,
                        [(0.0, 0.0)] * nd, eta=self.eta, dt=dt, f_V=fV, f_P=fP)
        d.iterate(self.case["inner"])
        for a, b in zip(x.V + x.tau + [x.Pr], d.V + d.tau + [d.Pr]):
            geo.box(a).add_(geo.box(b))
        free_slip(geo, x.V, shear(nd))
        return [interiors(geo, x.V + x.tau + [x.Pr], state_locs(nd)), err]

    @staticmethod
    def work(case):
        nd, nt = (3, 6) if case["nz"] else (2, 3)
        return {"bytes": cells(case) * 8 * (2 * (nd + nt + 1) + nt + 1),
                "flops": cells(case) * (case["inner"] + 2) * (150 if nd == 3 else 75)}


class ThermalStep(SlowFlow):
    def __init__(self, case, seed):
        self.case, self.geo = case, geometry(case)
        rng, geo, nd = generator(seed), self.geo, self.geo.nd
        self.V, self.tau, self.Pr = flow(geo, rng, self.RATE)
        self.T = smooth(geo, center(nd), rng) + 2.0
        neumann(geo, self.T)
        self.rhog = smooth(geo, vloc(nd - 1, nd), rng, 10.0 * self.RATE)

    def prepare(self):
        geo = self.geo
        g, nd = geo.grid(), geo.nd
        self.M = StokesThermal(arch(), g, eta=self.ETA, G=self.G, lam_rhoCp=self.LAM,
                               rhog=filled(g, vloc(nd - 1, nd), self.rhog),
                               normal_values=dict(enumerate(shear(nd, self.RATE))))
        load_state(self.M.S, self.V, self.tau, self.Pr)
        put(self.M.T, self.T)
        self.M.apply_bc()

    def run(self):
        M, n = self.M, self.case["iters"]
        _, err = M.time_step(2, n, n, 0.0)
        S = M.S
        return [views(list(S.V) + list(S.tau) + [S.Pr, M.T]), err]

    def exact(self):
        geo, nd = self.geo, self.geo.nd
        lam = self.LAM
        vmax = [float(geo.inner(v, vloc(d, nd)).abs().max()) for d, v in enumerate(self.V)]
        dt = min(min(geo.h) ** 2 / lam / nd / 2.1, 0.1 * min(h / v for h, v in zip(geo.h, vmax)) / nd / 2.1)
        told, Told = [t.clone() for t in self.tau], self.T.clone()
        P = PlainStokes(geo, self.V, self.tau, self.Pr, told, shear(nd, self.RATE), eta=self.ETA, dt=dt, G=self.G,
                        rhog=self.rhog)
        q = [geo.zeros(vloc(d, nd)) for d in range(nd)]
        for _ in range(self.case["iters"]):
            dv, rV = P.iterate(1)
            plain_thermal(geo, self.T, Told, q, P.V, lam, dt)
        _, m = residual_fields(geo, dv, rV)
        err = [m[0] * (self.ETA / self.G)] + [x * geo.L[-1] / self.G for x in m[1:]]
        return [interiors(geo, P.V + P.tau + [P.Pr, self.T], state_locs(nd) + [center(nd)]), err]

    @staticmethod
    def work(case):
        nd, nt = (3, 6) if case["nz"] else (2, 3)
        arrays = 2 * (nd + nt + 2) + nt + 1 + 1
        return {"bytes": cells(case) * 8 * arrays, "flops": cells(case) * case["iters"] * (180 if nd == 3 else 90)}


class Ice:
    """Glen n = 3 shallow ice on a 250 km square: bumpy bed, an ice cap on it."""
    MB = (0.01, 1500.0, 2.0)

    def __init__(self, case, seed):
        self.case = case
        self.geo = Geometry((case["nx"], case["ny"]), (0.0, 0.0), (250e3, 250e3))
        rng, geo = generator(seed), self.geo
        X, Y = geo.coords((0, 0))
        self.B = geo.zeros((0, 0))
        for _ in range(8):
            cx, cy, s = rng.uniform(75e3, 175e3), rng.uniform(75e3, 175e3), rng.uniform(30e3, 60e3)
            self.B += rng.uniform(0.0, 1000.0) * torch.exp(-((X - cx) ** 2 + (Y - cy) ** 2) / s ** 2)
        r2 = ((X - 125e3) ** 2 + (Y - 125e3) ** 2) / rng.uniform(60e3, 80e3) ** 2
        self.H0 = rng.uniform(50.0, 150.0) * (1.0 - r2).clamp(min=0.0).sqrt()
        neumann(geo, self.H0)
        self.logA = math.log(1e-4) + smooth(geo, (0, 0), rng, 0.1)
        self.logA_obs = self.logA + smooth(geo, (0, 0), rng, 0.2)

    def solver(self):
        return SIA(arch(), self.geo.grid(), self.B.cpu().numpy(), self.logA.cpu().numpy(), mb=self.MB, dt_max=1.0)

    def diffusivity(self, H, A):
        """Surface gradients on the faces and D on the cells."""
        geo = self.geo
        S = self.B[1:-1, 1:-1] + H
        gx, gy = (S[:, 1:] - S[:, :-1]) * geo.ih[0], (S[1:, :] - S[:-1, :]) * geo.ih[1]
        ax, ay = 0.5 * (gx[1:-1, 1:] + gx[1:-1, :-1]), 0.5 * (gy[1:, 1:-1] + gy[:-1, 1:-1])
        h = H[1:-1, 1:-1]
        return gx, gy, A[2:-2, 2:-2] * h ** 5 * (ax * ax + ay * ay)

    def step(self, h, A, dt):
        """One step of the cells h; H is h with its Neumann ghosts."""
        geo, (a, b, c) = self.geo, self.MB
        H = torch.nn.functional.pad(h[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
        gx, gy, D = self.diffusivity(H, A)
        qx = torch.zeros(h.shape[0], h.shape[1] + 1, dtype=F64, device=h.device)
        qy = torch.zeros(h.shape[0] + 1, h.shape[1], dtype=F64, device=h.device)
        qx[:, 1:-1] = -0.5 * (D[:, 1:] + D[:, :-1]) * gx[1:-1, 1:-1]
        qy[1:-1, :] = -0.5 * (D[1:, :] + D[:-1, :]) * gy[1:-1, 1:-1]
        m = a * (self.B[2:-2, 2:-2] + h - b)
        m = torch.where(m < c, m, torch.full_like(m, c))
        div = (qx[:, 1:] - qx[:, :-1]) * geo.ih[0] + (qy[1:, :] - qy[:-1, :]) * geo.ih[1]
        x = h + dt * (m - div)
        return torch.where(x > 0, x, torch.zeros_like(x))


class SiaForward(Ice):
    def prepare(self):
        self.S = self.solver()
        self.S.reset(self.H0.cpu().numpy())

    def run(self):
        dts = self.S.forward(self.case["steps"])
        return [np.array(dts), self.S.H.interior()]

    def exact(self):
        geo, A, dts = self.geo, self.logA.exp(), []
        h = self.H0[2:-2, 2:-2].clone()
        for _ in range(self.case["steps"]):
            H = torch.nn.functional.pad(h[None, None], (1, 1, 1, 1), mode="replicate")[0, 0]
            dmax = float(self.diffusivity(H, A)[2].max())
            dts.append(min(min(geo.h) ** 2 / dmax / 4.1 if dmax > 0 else math.inf, 1.0))
            h = self.step(h, A, dts[-1])
        return [np.array(dts), h.t()]

    @staticmethod
    def work(case):
        return {"bytes": cells(case) * 8 * 4, "flops": cells(case) * case["steps"] * 120}


class SiaGradient(Ice):
    DT = 0.1

    def prepare(self):
        self.S = self.solver()
        self.h0 = self.H0.cpu().numpy()
        self.obs = self.observed().t()
        self.dts = [self.DT] * self.case["steps"]

    def observed(self):
        A, h = self.logA_obs.exp(), self.H0[2:-2, 2:-2].clone()
        for _ in range(self.case["steps"]):
            h = self.step(h, A, self.DT)
        return h

    def run(self):
        J, g = self.S.gradient(self.h0, self.obs, self.case["steps"], self.dts, self.case["ncheck"])
        return [J, g, self.S.lam.interior(), self.S.H.interior()]

    def exact(self):
        obs = self.observed()
        logA = self.logA.clone().requires_grad_(True)
        h0 = self.H0[2:-2, 2:-2].clone().requires_grad_(True)
        h = h0
        for _ in range(self.case["steps"]):
            h = torch.utils.checkpoint.checkpoint(self.step, h, logA.exp(), self.DT, use_reentrant=False)
        J = 0.5 * ((h - obs) ** 2).sum()
        gA, gH = torch.autograd.grad(J, (logA, h0))
        return [float(J.detach()), gA[2:-2, 2:-2].t(), gH.t(), h.detach().t()]

    @staticmethod
    def work(case):
        # the bed, A, H0 and the observation in; the gradient, lambda and H out
        return {"bytes": cells(case) * 8 * 7, "flops": cells(case) * case["steps"] * 500}


KINDS = {"diffusion_launch": DiffusionLaunch, "diffusion_loop": DiffusionLoop, "operators": Operators,
         "set_functions": SetFunctions, "stokes": Stokes, "stokes_launch": StokesLaunch, "mixed_cycle": MixedCycle,
         "thermal_step": ThermalStep, "sia_forward": SiaForward, "sia_gradient": SiaGradient}


def prepare(case, seed):
    state = KINDS[case["kind"]](case, seed)
    state.prepare()
    return state


def run(state):
    return state.run()


def exact(case, seed):
    return KINDS[case["kind"]](case, seed).exact()


def work(case):
    return KINDS[case["kind"]].work(case)
