"""What a program that uses this library spends its time on, as measurable cases.

Every case is a dict of plain values with a "kind": one solver family of the
C ABI (masterthesis_amd.capi) or the torch gradient over it.  prepare() builds
what such a program holds before the call (fields in device memory, made on
the GPU from the seed; coefficients; parameters), run() makes one pass through
the public entry points, exact() is the same result in 64 bits in plain torch.

Time loops go on from pass to pass, as a program's do ("the next K steps");
problems that a program restarts (the constant-coefficient run, the
TimeLinSpaceLin problem, the ensemble of an optimisation loop) start each pass
from their initial state.  Device arrays are torch tensors handed over by
address; grids are in the library's memAll layout, (z, y, x) with one ghost
layer.
"""
import ctypes as C
import math

import torch

from masterthesis_amd import autograd, capi

F32, F64, KAHAN = "f32", "f64", "f32_kahan"
CODE = {F32: capi.F32, F64: capi.F64, KAHAN: capi.F32_KAHAN}
HEATVAR = {F32: capi.HEATVAR_F32, F64: capi.HEATVAR_F64, KAHAN: capi.HEATVAR_F32_KAHAN}
_ctx = None


def listed():
    return [
        # the smallest problems: the reference's TimeLinSpaceLin system test,
        # every step re-evaluating the known fields and updating, a
        # convergence check at the end: launches and the one wait
        dict(name="timelin_step", kind="timelin", nx=32, ny=24, nz=20, dim=3, border="dirichlet", form="heat", steps=4),
        # the reference's constant-coefficient heat, 64^3 FP64, 100 steps
        dict(name="heat_run_64", kind="heat", nx=64, ny=64, nz=64, perf=False, steps=100),
        # the benchmark's workload: 512^3, FP32 with compensated increments
        dict(name="heatvar_kahan_512", kind="heatvar", nx=512, ny=512, nz=512, dtype=KAHAN, border="keep", steps=20),
        # an ordinary FP64 production grid with odd extents and a step count
        # that no number of steps per sweep divides
        dict(name="heatvar_f64_ragged", kind="heatvar", nx=201, ny=150, nz=131, dtype=F64, border="value", steps=50),
        # Pennes bioheat, the forward time loop one call per step
        dict(name="pennes_steps_256", kind="pennes", nx=256, ny=256, nz=256, dtype=F32, border="keep", steps=20),
        # perfusion gradient with a snapshot budget (forward recomputation
        # and reverse sweep), FP32 fields
        dict(name="pennes_grad_128", kind="pennes_grad", nx=128, ny=128, nz=128, dtype=F32, border="keep", steps=200,
             snapshots=40),
        # one evaluation of an optimisation over a diffusivity field through
        # torch.autograd, host tensors in and out, odd extents
        dict(name="kappa_autograd_96", kind="kappa", nx=97, ny=80, nz=75, dtype=KAHAN, border="keep", steps=30,
             snapshots=16),
        # Yee leapfrog at the benchmark's box, energy record every tenth step
        dict(name="yee_384", kind="yee", ncell=384, dtype=F32, steps=20, energy_every=10, second=True),
        # permittivity gradient, snapshots fewer than steps
        dict(name="yee_eps_grad_128", kind="yee_eps", ncell=128, dtype=F32, steps=40, snapshots=10),
        # the EMFDTD example: CPML on every face, a conductive sphere, FP64
        dict(name="emfdtd_200", kind="emfdtd", n=200, d=10, radius=40.0, steps=20),
        # the MRI-data brain example on the reference's grid, FP64
        dict(name="mri_brain", kind="mri", nx=120, ny=120, nz=50, steps=50),
        # the ensemble of 4096 two-dimensional problems with its gradient
        dict(name="batch2d_4096", kind="batch2d", nprob=4096, nmin=32, nmax=256, steps=500, gradient=True, graph=True),
    ]


def _logint(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _xyz(rng, lo, hi, nodes):
    """Three extents in lo..hi with at most `nodes` nodes in all."""
    while True:
        n = [_logint(rng, lo, hi) for _ in range(3)]
        if n[0] * n[1] * n[2] <= nodes:
            return dict(nx=n[0], ny=n[1], nz=n[2])


def draw(rng):
    kind = rng.choice(["timelin", "heat", "heatvar", "heatvar", "pennes", "pennes_grad", "kappa", "yee", "yee_eps",
                       "emfdtd", "mri", "batch2d"])
    dtype = rng.choice([F32, F64, KAHAN])
    if kind == "timelin":
        dim = rng.choice([1, 2, 3])
        n = [_logint(rng, 8, 80) if p < dim else 1 for p in range(3)]
        return dict(kind=kind, nx=n[0], ny=n[1], nz=n[2], dim=dim, form=rng.choice(["heat", "pennes"]),
                    border=rng.choice(["dirichlet", "neumann", "cauchy"]), steps=rng.randint(1, 20))
    if kind == "heat":
        n = _xyz(rng, 20, 320, 1.2e7)
        return dict(kind=kind, **n, perf=rng.random() < 0.3, steps=_logint(rng, 10, 200))
    if kind == "heatvar":
        n = _xyz(rng, 24, 480, 6e7)
        return dict(kind=kind, **n, dtype=dtype, border=rng.choice(["keep", "value"]), steps=rng.randint(1, 60))
    if kind == "pennes":
        return dict(kind=kind, **_xyz(rng, 24, 320, 2e7), dtype=dtype, border=rng.choice(["keep", "keep", "tumor"]),
                    steps=rng.randint(1, 40))
    if kind == "pennes_grad":
        steps = _logint(rng, 8, 250)
        return dict(kind=kind, **_xyz(rng, 20, 160, 2.2e6), dtype=dtype, border=rng.choice(["keep", "keep", "tumor"]),
                    steps=steps, snapshots=_logint(rng, 3, steps))
    if kind == "kappa":
        steps = _logint(rng, 6, 60)
        return dict(kind=kind, **_xyz(rng, 16, 120, 8e5), dtype=dtype, border="keep", steps=steps,
                    snapshots=_logint(rng, 3, steps))
    if kind == "yee":
        return dict(kind=kind, ncell=_logint(rng, 24, 320), dtype=rng.choice([F32, F32, F64]),
                    steps=rng.randint(1, 40), energy_every=rng.choice([0, 1, 10]), second=rng.random() < 0.8)
    if kind == "yee_eps":
        steps = _logint(rng, 6, 60)
        return dict(kind=kind, ncell=_logint(rng, 16, 120), dtype=rng.choice([F32, F64]), steps=steps,
                    snapshots=_logint(rng, 3, steps))
    if kind == "emfdtd":
        n = _logint(rng, 32, 192)
        return dict(kind=kind, n=n, d=rng.randint(4, 12), radius=rng.choice([0.0, 0.2 * n]), steps=rng.randint(1, 40))
    if kind == "mri":
        return dict(kind=kind, **_xyz(rng, 24, 180, 2e6), steps=rng.randint(5, 80))
    nmin = _logint(rng, 2, 128)
    return dict(kind=kind, nprob=_logint(rng, 1, 4096), nmin=nmin, nmax=rng.randint(nmin, 256),
                steps=_logint(rng, 10, 500), gradient=rng.random() < 0.7, graph=rng.random() < 0.5)


# ------------------------------------------------------------------ inputs
def _context():
    global _ctx
    if _ctx is None:
        _ctx = capi.Context(0)
    return _ctx


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _rand(gen, shape, lo=0.0, hi=1.0):
    return torch.rand(shape, generator=gen, device="cuda", dtype=torch.float64) * (hi - lo) + lo


def _randn(gen, shape):
    return torch.randn(shape, generator=gen, device="cuda", dtype=torch.float64)


def _dt(case):
    return torch.float64 if case["dtype"] == F64 else torch.float32


def _shape(c):
    return (c["nz"], c["ny"], c["nx"])


def _axes(c):
    """Node coordinates x, y, z on the unit cube, broadcastable to (z, y, x)."""
    x, y, z = (torch.arange(n, device="cuda", dtype=torch.float64) / (n - 1) for n in (c["nx"], c["ny"], c["nz"]))
    return x[None, None, :], y[None, :, None], z[:, None, None]


def _hh(c):
    return [(1.0 / (n - 1)) ** 2 for n in (c["nx"], c["ny"], c["nz"])]


def _memall(nodes, dtype):
    """A field with one ghost layer around the node array (ghosts 0)."""
    return torch.nn.functional.pad(nodes, [1, 1] * nodes.dim()).to(dtype).contiguous()


def _sines(c):
    x, y, z = _axes(c)
    return torch.sin(math.pi * x) * torch.sin(math.pi * y) * torch.sin(math.pi * z)


def _heatvar_inputs(c, seed):
    """u: a sine mode on top of the border value with noise of 1e-3 on inner
    nodes, kappa = 1 + 0.5 sin sin with seeded phases; as the field type holds them."""
    gen = _gen(seed)
    x, y, z = _axes(c)
    noise = _rand(gen, _shape(c), -1e-3, 1e-3)
    inner = torch.zeros_like(noise)
    inner[1:-1, 1:-1, 1:-1] = 1.0
    ph = _rand(gen, 3, 0.0, 2 * math.pi)
    kappa = 1.0 + 0.5 * torch.sin(2 * math.pi * x + ph[0]) * torch.sin(2 * math.pi * y + ph[1]) + 0.0 * z
    u = 1.0 + _sines(c) + noise * inner
    return u.to(_dt(c)), kappa.to(_dt(c))


def _heatvar_tau(c):
    return 0.9 / sum(2 * 1.5 / h for h in _hh(c))


def _pennes_inputs(c, seed):
    """Deviation from the arterial temperature: a start of a few tenths of a
    kelvin, log-normal perfusion (median 0.5), a Gaussian source."""
    gen = _gen(seed)
    x, y, z = _axes(c)
    w = (0.5 * torch.exp(0.3 * _randn(gen, _shape(c)))).clamp(max=3.0)
    q = 50.0 * torch.exp(-((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.5) ** 2) / 0.02)
    t = 0.5 * _sines(c) + 0.05 * _randn(gen, _shape(c))
    return [v.to(_dt(c)) for v in (t, w, q)]


def _pennes_params(c):
    p = capi.PennesParams(cdiff=0.5, cperf=1.0, csrc=1.0, t_a=0.0)
    if c["border"] == "tumor":
        p.border_mode, p.k_cond, p.h_conv, p.t_inf, p.q_bc = capi.BORDER_TUMOR, 0.5, 10.0, -15.0, 0.2
    p.tau = 0.9 / (sum(2 * 0.5 / h for h in _hh(c)) + 3.0 + 20.0 * (c["nz"] - 1))
    return p


def _target_like(t, gen):
    """A measured final state: the start, lowered, with noise."""
    return (0.9 * t.double() + 0.02 * _randn(gen, t.shape)).to(t.dtype)


def _yee_start(n, seed, dtype):
    """Six (N+1)^3 arrays: a Gaussian Ez pulse near the centre, seeded place
    and width, zero on the walls; H a weak smooth field inside."""
    gen = _gen(seed)
    m = n + 1
    a = torch.arange(m, device="cuda", dtype=torch.float64)
    r = _rand(gen, 4)
    cx, cy, cz = ((0.4 + 0.2 * r[q]) * n for q in range(3))
    s = (0.03 + 0.03 * r[3]) * n + 1.0
    gx, gy, gz = (torch.exp(-((a + o - c) ** 2) / (2 * s * s)) for c, o in ((cx, 0.0), (cy, 0.0), (cz, 0.5)))
    f = torch.zeros((6, m, m, m), device="cuda", dtype=dtype)
    ez = gz[:, None, None] * gy[None, :, None] * gx[None, None, :]
    f[2, :n, 1:n, 1:n] = ez[:n, 1:n, 1:n].to(dtype)
    f[3, :n, :n, :] = (0.1 * ez[:n, :n, :]).to(dtype)
    return f


def _eps_inputs(c, seed):
    """A dielectric sphere (about 4) in a slightly uneven medium, and a target."""
    n = c["ncell"]
    f = _yee_start(n, seed, _dt(c))
    gen = _gen(seed + 7)
    a = torch.arange(n + 1, device="cuda", dtype=torch.float64) / n - 0.5
    r2 = a[:, None, None] ** 2 + a[None, :, None] ** 2 + a[None, None, :] ** 2
    eps = torch.where(r2 < 0.09, 4.0, 1.0) * (1.0 + 0.05 * _rand(gen, r2.shape))
    target = 0.1 * _yee_start(n, seed + 13, torch.float64)[:3]
    return f, eps.to(_dt(c)), target.to(_dt(c))


def _em_inputs(c, seed):
    """26 arrays: an Ez pulse (D = E in vacuum), no conduction current, psi
    zero, a conductive sphere away from the source."""
    n = c["n"]
    gen = _gen(seed)
    r = _rand(gen, 4)
    a = torch.arange(n, device="cuda", dtype=torch.float64)

    def bell(p):
        cen = (0.35 + 0.3 * r[p]) * n
        return torch.exp(-((a - cen) ** 2) / (2 * (0.04 * n + 1.0) ** 2))
    f = torch.zeros((26, n, n, n), device="cuda", dtype=torch.float64)
    ez = (0.5 + r[3]) * bell(2)[:, None, None] * bell(1)[None, :, None] * bell(0)[None, None, :]
    f[8, :n - 1, 1:, 1:] = ez[:n - 1, 1:, 1:]
    sigma = torch.zeros((n, n, n), device="cuda", dtype=torch.float64)
    if c["radius"] > 0:
        b = (a - 0.5 * n) ** 2
        sigma[b[:, None, None] + b[None, :, None] + b[None, None, :] < c["radius"] ** 2] = 3.546e7
    g = sigma * (0.5 / 299792458.0) / 8.85418781762e-12
    f[24], f[25] = 1.0 / (1.0 + g), g
    f[2] = f[24] * f[8]
    f[11] = f[25] * f[2]
    return f


def _em_params(c):
    n = c["n"]
    q = n // 4
    return capi.emfdtd_params(n, d=c["d"], src=(q, q, q), sink=(q + 3, q + 3, q + 3), t0=10.0, spread=4.0)


def _mri_inputs(c, seed):
    """Temperature and nine node materials of brain tissue with a tumour
    region, uneven by some per cent; a disc of open skull on the last face."""
    gen = _gen(seed)
    s = _shape(c)
    x, y, z = _axes(c)
    tum = ((x - 0.5) ** 2 + (y - 0.5) ** 2 + (z - 0.7) ** 2 < 0.04).double()
    surf = torch.zeros(s, device="cuda", dtype=torch.float64)
    surf[-1] = ((x - 0.5) ** 2 + (y - 0.5) ** 2 < 0.09).double()[0]
    one = torch.ones(s, device="cuda", dtype=torch.float64)
    mat = [1040.0 * (1 + 0.05 * _rand(gen, s)), 3650.0 * (1 + 0.05 * _rand(gen, s)), 0.5 + 0.2 * _rand(gen, s),
           1052.0 * one, 3800.0 * one, 0.004 + 0.006 * _rand(gen, s) + 0.002 * tum, 36.5 + 0.5 * tum,
           25000.0 * _rand(gen, s), surf]
    t = 36.0 + 0.5 * tum + 0.1 * _randn(gen, s)
    return t, [m.contiguous() for m in mat]


MRI_EXTENT = (0.14, 0.16, 0.14)


def _mri_params(c):
    h = [e / (n - 1) for e, n in zip(MRI_EXTENT, (c["nx"], c["ny"], c["nz"]))]
    tau = 0.4 / sum(2.0 * 0.7 / (1040.0 * 3650.0) / hp ** 2 for hp in h)
    return h, capi.MriParams(tau=tau, h_conv=10.0, t_amb=22.0, q_bc=0.0, q_skull=0.0, epsilon=0.98, sigma=5.670373e-8)


def _batch_inputs(c, seed):
    """Edges uniform in nmin..nmax (the same for every seed: the ensemble's
    grids are fixed, its parameters and states are not), kappa in [0.1, 1]."""
    g0 = torch.Generator().manual_seed(c["nprob"] + 1000 * c["nmin"] + c["nmax"])
    n = torch.randint(c["nmin"], c["nmax"] + 1, (c["nprob"],), generator=g0)
    gen = _gen(seed)
    kappa = _rand(gen, c["nprob"], 0.1, 1.0).float()
    tau = (0.9 / 4.0 / (n.double() - 1) ** 2).float().cuda()
    off = torch.cumsum(n * n, 0) - n * n
    total = int((n * n).sum())
    nd, od = n.cuda(), off.cuda()
    who = torch.repeat_interleave(torch.arange(c["nprob"], device="cuda"), nd * nd, output_size=total)
    at = torch.arange(total, device="cuda") - od[who]
    edge = nd[who]
    i, j = at % edge, at // edge
    inner = (i > 0) & (i < edge - 1) & (j > 0) & (j < edge - 1)
    u = torch.sin(math.pi * i / (edge - 1)) * torch.sin(math.pi * j / (edge - 1)) + 0.01 * _randn(gen, total)
    u = torch.where(inner, u, torch.zeros_like(u)).float()
    dec = torch.exp(-2 * math.pi ** 2 * 1.1 * kappa.double() * c["steps"] * tau.double())
    target = (u.double() * dec[who]).float()
    order = torch.argsort(-((n + 31) // 32), stable=True).int().cuda()
    return dict(n=nd.int(), off=od, kappa=kappa, tau=tau, order=order, u0=u, target=target)


TIMELIN_BORDER = {"dirichlet": capi.BORDER_FIELD, "neumann": capi.BORDER_NEUMANN, "cauchy": capi.BORDER_CAUCHY}


def _timelin(c, seed):
    """Geometry, time step, start time and first node of the problem
    u = (1 + t)(1 + sum x); the seed moves the domain and the start time."""
    g = torch.Generator().manual_seed(seed)
    r = torch.rand(4, generator=g).tolist()
    dim = c["dim"]
    n = [c["nx"], c["ny"], c["nz"]][:dim]
    h = [1.0 / (m - 1) for m in n]
    tau = 0.4 / (sum(2.0 / q ** 2 for q in h) + 1.0)
    return n, h, tau, r[3], [r[p] if p < dim else 0.0 for p in range(3)]


# ------------------------------------------------------------------ prepare
def _geom(c):
    return capi.geom((c["nx"], c["ny"], c["nz"]))


def prepare(case, seed):
    c, ctx = case, _context()
    s = dict(case=c, ctx=ctx, L=ctx.L, which=C.c_int(0), at=0)
    kind = c["kind"]
    if kind == "timelin":
        n, h, tau, t, x0 = _timelin(c, seed)
        s["geom"], s["t"], s["tau"] = capi.geom(n, h=h), t, tau
        k = capi.TimelinParams(form=capi.KNOWN_PENNES_TIMELIN if c["form"] == "pennes" else capi.KNOWN_HEAT_TIMELIN,
                               border_mode=TIMELIN_BORDER[c["border"]], rho_c=1.0, rhob_cb_w=1.0, lam=1.0, alpha=1.0,
                               epsilon=1.0, sigma=1.0)
        k.x0[:] = x0
        s["known"] = k
        s["p"] = capi.Heat7Params(tau=tau, coeff_a=1.0, rhoc_inv=1.0, perf_c=1.0, perf_w=1.0,
                                  has_perf=int(c["form"] == "pennes"), has_source=1, border_mode=k.border_mode, lam=1.0,
                                  alpha=1.0, epsilon=1.0, sigma=1.0)
        nodes = math.prod(n)
        s["u"] = [torch.zeros([m + 2 for m in reversed(n)], device="cuda", dtype=torch.float64) for _ in range(2)]
        s["f"] = [torch.zeros(nodes, device="cuda", dtype=torch.float64) for _ in range(2)]
        s["g"] = [torch.zeros(nodes, device="cuda", dtype=torch.float64) for _ in range(2)]
    elif kind == "heat":
        s["geom"] = _geom(c)
        s["u0"] = _memall(_heat_start(c, seed), torch.float64)
        s["u"] = [torch.zeros_like(s["u0"]) for _ in range(2)]
        s["p"] = capi.Heat7Params(tau=_heat_tau(c), coeff_a=1.0, rhoc_inv=1.0, perf_c=1.0, perf_w=0.5,
                                  has_perf=int(c["perf"]), border_mode=capi.BORDER_VALUE)
    elif kind == "heatvar":
        u, kappa = _heatvar_inputs(c, seed)
        s["geom"] = _geom(c)
        s["u"] = [_memall(u, _dt(c)), _memall(u, _dt(c))]
        s["c"] = [torch.zeros_like(s["u"][0]) for _ in range(2)] if c["dtype"] == KAHAN else [None, None]
        s["kappa"] = _memall(kappa, _dt(c))
        s["tau"] = _heatvar_tau(c)
        capi.check(s["L"].scafes_coef_changed(ctx.h, s["kappa"].data_ptr()))
    elif kind in ("pennes", "pennes_grad"):
        t, w, q = (_memall(v, _dt(c)) for v in _pennes_inputs(c, seed))
        s["geom"], s["p"] = _geom(c), _pennes_params(c)
        s["w"], s["q"] = w, q
        if kind == "pennes":
            s["u"] = [t, t.clone()]
            s["c"] = [torch.zeros_like(t) for _ in range(2)]
            capi.check(s["L"].scafes_coef_changed(ctx.h, w.data_ptr()))
        else:
            s["t0"], s["target"] = t, _memall(_target_like(t[1:-1, 1:-1, 1:-1], _gen(seed + 5)), _dt(c))
            s["grad"] = torch.zeros_like(t, dtype=torch.float64)
    elif kind == "kappa":
        u, kappa = _heatvar_inputs(c, seed)
        target = _target_like(u, _gen(seed + 5))
        s["u0"], s["kappa"], s["target"] = (_memall(v, torch.float64).cpu() for v in (u, kappa, target))
        s["kappa"].requires_grad_(True)
        s["misfit"] = autograd.KappaMisfit(ctx, (c["nx"], c["ny"], c["nz"]), _heatvar_tau(c), c["steps"],
                                           snapshots=c["snapshots"], dtype=c["dtype"], border=c["border"])
    elif kind == "yee":
        f = _yee_start(c["ncell"], seed, _dt(c))
        s["f"] = [f, torch.zeros_like(f) if c["second"] else None]
        every = c["energy_every"]
        s["energy"] = torch.zeros((c["steps"] + every - 1) // every if every else 1, dtype=torch.float64)
    elif kind == "yee_eps":
        s["f"], s["eps"], s["target"] = _eps_inputs(c, seed)
        s["grad"] = torch.zeros_like(s["eps"], dtype=torch.float64)
    elif kind == "emfdtd":
        s["f"], s["p"] = _em_inputs(c, seed), _em_params(c)
        s["sink"] = torch.zeros(c["steps"], device="cuda", dtype=torch.float64)
    elif kind == "mri":
        t, mat = _mri_inputs(c, seed)
        h, s["p"] = _mri_params(c)
        s["geom"] = capi.geom((c["nx"], c["ny"], c["nz"]), h=h)
        s["u"] = [_memall(t, torch.float64), _memall(t, torch.float64)]
        s["mat"], s["ptrs"] = mat, (capi.vp * 9)(*[m.data_ptr() for m in mat])
        s["coef"] = torch.zeros((4,) + tuple(s["u"][0].shape), device="cuda", dtype=torch.float64)
        torch.cuda.synchronize()
        capi.check(s["L"].scafes_mri_coef_f64(ctx.h, C.byref(s["geom"]), 1, s["ptrs"], C.byref(s["p"]),
                                              s["coef"].data_ptr()))
    else:
        s.update(_batch_inputs(c, seed))
        s["u"] = torch.zeros_like(s["u0"])
        s["J"] = torch.zeros(c["nprob"], device="cuda", dtype=torch.float64)
        s["grad"] = torch.zeros_like(s["J"])
    torch.cuda.synchronize()  # the library works on its own stream
    return s


def _heat_start(c, seed):
    """A sine mode (and its second harmonic in x) with seeded amplitudes."""
    r = _rand(_gen(seed), 2)
    x, y, z = _axes(c)
    u = (0.5 + r[0]) * _sines(c)
    u += 0.3 * r[1] * torch.sin(2 * math.pi * x) * torch.sin(math.pi * y) * torch.sin(math.pi * z)
    out = torch.zeros_like(u)
    out[1:-1, 1:-1, 1:-1] = u[1:-1, 1:-1, 1:-1]
    return out


def _heat_tau(c):
    return 0.9 / (sum(2.0 / h for h in _hh(c)) + (0.5 if c["perf"] else 0.0))


# ------------------------------------------------------------------ run
def run(s):
    return RUN[s["case"]["kind"]](s)


def _run_timelin(s):
    L, h, g, p, k = s["L"], s["ctx"].h, C.byref(s["geom"]), C.byref(s["p"]), C.byref(s["known"])
    a, b = s["u"]
    f, f2 = s["f"]
    gg, g2 = s["g"]
    t = s["t"]
    rc = L.scafes_known_timelin_f64(h, g, k, t, f.data_ptr(), gg.data_ptr(), a.data_ptr(), 1)
    for _ in range(s["case"]["steps"]):
        t += s["tau"]
        rc |= L.scafes_known_timelin_f64(h, g, k, t, f2.data_ptr(), g2.data_ptr(), None, 0)
        rc |= L.scafes_heat7_step_f64(h, g, 1, a.data_ptr(), b.data_ptr(), f.data_ptr(), gg.data_ptr(), g2.data_ptr(), p)
        a, b, f, f2, gg, g2 = b, a, f2, f, g2, gg
    change = C.c_double(0.0)
    rc |= L.scafes_reduce(h, g, capi.F64, a.data_ptr(), 1, b.data_ptr(), 1, capi.RED_MAX_ABS_DIFF, 0, C.byref(change))
    capi.check(rc)
    return {"u": a, "change": change.value}


def _run_heat(s):
    L, h = s["L"], s["ctx"].h
    u, u2 = s["u"]
    capi.check(L.scafes_memcpy_d2d(h, u.data_ptr(), s["u0"].data_ptr(), u.numel() * 8))
    capi.check(L.scafes_heat7_run_f64(h, C.byref(s["geom"]), C.c_int(1), capi.vp(u.data_ptr()), capi.vp(u2.data_ptr()),
                                      C.c_int(s["case"]["steps"]), C.byref(s["p"]), C.byref(s["which"])))
    return {"u": s["u"][s["which"].value]}


def _run_heatvar(s):
    c, at = s["case"], s["at"]
    u, u2, k, k2 = s["u"][at], s["u"][1 - at], s["c"][at], s["c"][1 - at]
    capi.check(s["L"].scafes_heat7var_run(s["ctx"].h, C.byref(s["geom"]), 1, HEATVAR[c["dtype"]], u.data_ptr(),
                                          u2.data_ptr(), None if k is None else k.data_ptr(),
                                          None if k2 is None else k2.data_ptr(), s["kappa"].data_ptr(), s["tau"],
                                          c["steps"], capi.BORDER_VALUE if c["border"] == "value" else capi.BORDER_KEEP,
                                          1.0, -1, C.byref(s["which"])))
    at = s["at"] = (at + s["which"].value) % 2
    out = {"u": s["u"][at]}
    if c["dtype"] == KAHAN:
        out["c"] = s["c"][at]
    return out


def _run_pennes(s):
    c, L, h, g, p = s["case"], s["L"], s["ctx"].h, C.byref(s["geom"]), C.byref(s["p"])
    at, rc, w, q = s["at"], 0, s["w"].data_ptr(), s["q"].data_ptr()
    u, k = [x.data_ptr() for x in s["u"]], [x.data_ptr() for x in s["c"]]
    if c["dtype"] == KAHAN:
        for _ in range(c["steps"]):
            rc |= L.scafes_pennes_step_kahan(h, g, 1, u[at], u[1 - at], k[at], k[1 - at], w, q, p)
            at = 1 - at
    else:
        code = CODE[c["dtype"]]
        for _ in range(c["steps"]):
            rc |= L.scafes_pennes_step(h, g, 1, code, u[at], u[1 - at], w, q, p)
            at = 1 - at
    capi.check(rc)
    s["at"] = at
    out = {"t": s["u"][at]}
    if c["dtype"] == KAHAN:
        out["c"] = s["c"][at]
    return out


def _run_pennes_grad(s):
    c, J = s["case"], C.c_double(0.0)
    capi.check(s["L"].scafes_pennes_gradient(s["ctx"].h, C.byref(s["geom"]), 1, CODE[c["dtype"]], s["t0"].data_ptr(),
                                             s["w"].data_ptr(), s["q"].data_ptr(), s["target"].data_ptr(),
                                             C.byref(s["p"]), c["steps"], c["snapshots"], s["grad"].data_ptr(),
                                             C.byref(J), None))
    return {"J": J.value, "grad": s["grad"]}


def _run_kappa(s):
    J = s["misfit"](s["kappa"], s["u0"], s["target"])
    grad, = torch.autograd.grad(J, s["kappa"])
    return {"J": J.detach(), "grad": grad}


def _run_yee(s):
    c, at = s["case"], s["at"]
    f2 = s["f"][1 - at]
    capi.check(s["L"].scafes_yee_run(s["ctx"].h, c["ncell"], CODE[c["dtype"]], 0.5, s["f"][at].data_ptr(),
                                     None if f2 is None else f2.data_ptr(), c["steps"], c["energy_every"],
                                     C.cast(s["energy"].data_ptr(), C.POINTER(C.c_double)), C.byref(s["which"])))
    at = s["at"] = (at + s["which"].value) % 2
    return {"f": s["f"][at], "energy": s["energy"]} if c["energy_every"] else {"f": s["f"][at]}


def _run_yee_eps(s):
    c, J = s["case"], C.c_double(0.0)
    capi.check(s["L"].scafes_yee_eps_gradient(s["ctx"].h, c["ncell"], CODE[c["dtype"]], 0.5, s["f"].data_ptr(),
                                              s["eps"].data_ptr(), s["target"].data_ptr(), c["steps"], c["snapshots"],
                                              s["grad"].data_ptr(), C.byref(J), None))
    return {"J": J.value, "grad": s["grad"]}


def _run_emfdtd(s):
    capi.check(s["L"].scafes_emfdtd_run(s["ctx"].h, C.byref(s["p"]), s["f"].data_ptr(), s["case"]["steps"], 0.0,
                                        s["sink"].data_ptr()))
    return {"f": s["f"][:12], "psi": s["f"][12:24], "sink": s["sink"]}


def _run_mri(s):
    L, h, g, p = s["L"], s["ctx"].h, C.byref(s["geom"]), C.byref(s["p"])
    at, rc, coef, u = s["at"], 0, s["coef"].data_ptr(), [x.data_ptr() for x in s["u"]]
    for _ in range(s["case"]["steps"]):
        rc |= L.scafes_mri_step_f64(h, g, 1, u[at], u[1 - at], s["ptrs"], coef, p)
        at = 1 - at
    capi.check(rc)
    s["at"] = at
    return {"t": s["u"][at]}


def _run_batch2d(s):
    c, L, h = s["case"], s["L"], s["ctx"].h
    p = {k: s[k].data_ptr() for k in ("n", "off", "kappa", "tau", "order", "u", "target", "J", "grad")}
    capi.check(L.scafes_memcpy_d2d(h, p["u"], s["u0"].data_ptr(), s["u"].numel() * 4))
    want = c["gradient"]
    capi.check(L.scafes_batch2d_run(h, c["nprob"], p["n"], p["off"], p["kappa"], p["tau"], p["order"], p["u"],
                                    p["target"] if want else None, p["J"] if want else None,
                                    p["grad"] if want else None, c["steps"], int(c["graph"])))
    return {"u": s["u"], "J": s["J"], "grad": s["grad"]} if want else {"u": s["u"]}


RUN = {"timelin": _run_timelin, "heat": _run_heat, "heatvar": _run_heatvar, "pennes": _run_pennes,
       "pennes_grad": _run_pennes_grad, "kappa": _run_kappa, "yee": _run_yee, "yee_eps": _run_yee_eps,
       "emfdtd": _run_emfdtd, "mri": _run_mri, "batch2d": _run_batch2d}


# ------------------------------------------------------------------ work
def work(case):
    """Bytes: the fields a pass takes in and the ones it leaves, once each;
    operations: additions and products of the node updates."""
    c, kind = case, case["kind"]
    es = 8 if c.get("dtype", F64) == F64 else 4
    if kind == "batch2d":
        g0 = torch.Generator().manual_seed(c["nprob"] + 1000 * c["nmin"] + c["nmax"])
        n = torch.randint(c["nmin"], c["nmax"] + 1, (c["nprob"],), generator=g0)
        nodes = int((n * n).sum())
        return {"bytes": nodes * (12 if c["gradient"] else 8), "flops": 9.0 * nodes * c["steps"]}
    if kind in ("yee", "yee_eps"):
        nodes = (c["ncell"] + 1) ** 3
        if kind == "yee":
            return {"bytes": 12 * es * nodes, "flops": 30.0 * nodes * c["steps"]}
        return {"bytes": (10 * es + 8) * nodes, "flops": (33.0 + 75.0) * nodes * c["steps"]}
    if kind == "emfdtd":
        nodes = c["n"] ** 3
        return {"bytes": (26 + 24) * 8 * nodes, "flops": 45.0 * nodes * c["steps"]}
    nodes, steps = c["nx"] * c["ny"] * c["nz"], c["steps"]
    if kind == "timelin":
        return {"bytes": 8 * nodes, "flops": 30.0 * nodes * steps}
    if kind == "heat":
        return {"bytes": 16 * nodes, "flops": 19.0 * nodes * steps}
    if kind == "heatvar":
        return {"bytes": (5 if c["dtype"] == KAHAN else 3) * es * nodes, "flops": 34.0 * nodes * steps}
    if kind == "pennes":
        return {"bytes": (6 if c["dtype"] == KAHAN else 4) * es * nodes, "flops": 25.0 * nodes * steps}
    if kind == "pennes_grad":
        return {"bytes": (4 * es + 8) * nodes, "flops": (25.0 + 28.0) * nodes * steps}
    if kind == "kappa":
        return {"bytes": (3 * 8 + 8) * nodes, "flops": (34.0 + 65.0) * nodes * steps}
    return {"bytes": 7 * 8 * nodes, "flops": 26.0 * nodes * steps}


# About four times the largest relative error against exact() seen over the
# declared ranges: FP64 4.7e-15 (gradients; the forward paths stay below
# 1.2e-15), FP32 fields 4.2e-7 (the kappa gradient; forward 2e-7), the
# ensemble 5.1e-5 (dJ/dkappa from FP32 states after 500 steps).
def tolerance(case):
    kind = case["kind"]
    if kind == "batch2d":
        return {"rel": 2e-4, "max": 1e-2}
    if kind in ("timelin", "heat", "mri", "emfdtd") or case["dtype"] == F64:
        return {"rel": 2e-14, "max": 1e-11}
    return {"rel": 2e-6, "max": 1e-4}


# ------------------------------------------------------------------ exact
def _pad(v):
    return torch.nn.functional.pad(v, [1, 1] * v.dim())


def _sl(axis, lo, hi):
    s = [slice(None)] * 3
    s[axis] = slice(lo, hi)
    return tuple(s)


def _second(u, axis):
    """Second difference along an axis on inner positions of that axis."""
    return u[_sl(axis, 0, -2)] + u[_sl(axis, 2, None)] - 2 * u[_sl(axis, 1, -1)]


def _core(v, skip):
    """Cuts the border layer off every axis but `skip`."""
    for q in range(3):
        if q != skip:
            v = v[_sl(q, 1, -1)]
    return v


def _exact_timelin(c, seed):
    n, h, tau, t, x0 = _timelin(c, seed)
    s = 1.0
    for p, m in enumerate(n):
        x = x0[p] + h[p] * torch.arange(m, device="cuda", dtype=torch.float64)
        s = s + x.reshape([-1 if q == len(n) - 1 - p else 1 for q in range(len(n))])
    return {"u": _pad(s * (1.0 + t + c["steps"] * tau)), "change": float(s.max()) * tau}


def _exact_heat(c, seed):
    u, tau, hh = _heat_start(c, seed), _heat_tau(c), _hh(c)
    for _ in range(c["steps"]):
        d = sum(_core(_second(u, q), q) * (tau / hh[2 - q]) for q in range(3))
        if c["perf"]:
            d = d - tau * 0.5 * u[1:-1, 1:-1, 1:-1]
        u[1:-1, 1:-1, 1:-1] += d
    return {"u": _pad(u)}


def _flux(u, k, axis):
    f = 0.5 * (k[_sl(axis, 1, None)] + k[_sl(axis, 0, -1)]) * (u[_sl(axis, 1, None)] - u[_sl(axis, 0, -1)])
    return _core(f[_sl(axis, 1, None)] - f[_sl(axis, 0, -1)], axis)


def _exact_heatvar(c, seed):
    u, k = (v.double() for v in _heatvar_inputs(c, seed))
    tau, hh = _heatvar_tau(c), _hh(c)
    if c["border"] == "value":
        u = torch.nn.functional.pad(u[1:-1, 1:-1, 1:-1], [1] * 6, value=1.0)
    for _ in range(c["steps"]):
        u[1:-1, 1:-1, 1:-1] += sum(_flux(u, k, q) * (tau / hh[2 - q]) for q in range(3))
    out = {"u": _pad(u)}
    if c["dtype"] == KAHAN:
        out["c"] = None
    return out


def _tumor_second(u, axis, h, p):
    """Second difference with the Tumor example's border forms."""
    a = 2 * h / p.k_cond
    lo, hi, e, w = u[_sl(axis, 0, 1)], u[_sl(axis, -1, None)], u[_sl(axis, 1, 2)], u[_sl(axis, -2, -1)]
    last = 2 * w - a * p.h_conv * (hi - p.t_inf) - 2 * hi if axis == 0 else 2 * w + a * p.q_bc - 2 * hi
    return torch.cat([2 * e + a * p.q_bc - 2 * lo, _second(u, axis), last], axis)


def _pennes_next(t, w, q, p, c):
    hh = _hh(c)
    if c["border"] == "tumor":
        d = sum(_tumor_second(t, a, math.sqrt(hh[2 - a]), p) * (p.tau * p.cdiff / hh[2 - a]) for a in range(3))
        return t + d - p.tau * p.cperf * w * t + p.tau * p.csrc * q
    cut = (slice(1, -1),) * 3
    d = sum(_core(_second(t, a), a) * (p.tau * p.cdiff / hh[2 - a]) for a in range(3))
    return t + _pad(d - p.tau * p.cperf * w[cut] * t[cut] + p.tau * p.csrc * q[cut])


def _exact_pennes(c, seed):
    t, w, q = (v.double() for v in _pennes_inputs(c, seed))
    p = _pennes_params(c)
    for _ in range(c["steps"]):
        t = _pennes_next(t, w, q, p, c)
    out = {"t": _pad(t)}
    if c["dtype"] == KAHAN:
        out["c"] = None
    return out


def _exact_pennes_grad(c, seed):
    ins = _pennes_inputs(c, seed)
    target = _target_like(ins[0], _gen(seed + 5)).double()
    t, w, q = (v.double() for v in ins)
    p = _pennes_params(c)
    w.requires_grad_(True)
    for _ in range(c["steps"]):
        t = _pennes_next(t, w, q, p, c)
    r = t - target
    if c["border"] != "tumor":
        r = r[1:-1, 1:-1, 1:-1]
    J = 0.5 * (r * r).sum()
    grad, = torch.autograd.grad(J, w)
    return {"J": J.detach(), "grad": _pad(grad)}


def _exact_kappa(c, seed):
    u, k = _heatvar_inputs(c, seed)
    target = _target_like(u, _gen(seed + 5)).double()
    u, k = u.double(), k.double().requires_grad_(True)
    tau, hh = _heatvar_tau(c), _hh(c)
    for _ in range(c["steps"]):
        u = u + _pad(sum(_flux(u, k, q) * (tau / hh[2 - q]) for q in range(3)))
    r = (u - target)[1:-1, 1:-1, 1:-1]
    J = 0.5 * (r * r).sum()
    grad, = torch.autograd.grad(J, k)
    return {"J": J.detach().cpu(), "grad": _pad(grad).cpu()}


def _h_next(e, h):
    """H after a half step in a PEC box; e and h are lists of three arrays."""
    x, y, z = slice(0, -1), slice(0, -1), slice(0, -1)
    d = [(e[1][1:, y, :] - e[1][z, y, :]) - (e[2][z, 1:, :] - e[2][z, y, :]),
         (e[2][z, :, 1:] - e[2][z, :, x]) - (e[0][1:, :, x] - e[0][z, :, x]),
         (e[0][:, 1:, x] - e[0][:, y, x]) - (e[1][:, y, 1:] - e[1][:, y, x])]
    p = torch.nn.functional.pad
    return [h[0] + p(0.5 * d[0], [0, 0, 0, 1, 0, 1]), h[1] + p(0.5 * d[1], [0, 1, 0, 0, 0, 1]),
            h[2] + p(0.5 * d[2], [0, 1, 0, 1, 0, 0])]


def _e_next(e, h, eps=None):
    """E after a half step (walls stay zero); eps: relative permittivity."""
    b, m, a = slice(0, -2), slice(1, -1), slice(0, -1)
    d = [(h[2][m, m, a] - h[2][m, b, a]) - (h[1][m, m, a] - h[1][b, m, a]),
         (h[0][m, a, m] - h[0][b, a, m]) - (h[2][m, a, m] - h[2][m, a, b]),
         (h[1][a, m, m] - h[1][a, m, b]) - (h[0][a, m, m] - h[0][a, b, m])]
    if eps is not None:
        d = [d[0] / eps[m, m, a], d[1] / eps[m, a, m], d[2] / eps[a, m, m]]
    p = torch.nn.functional.pad
    return [e[0] + p(0.5 * d[0], [0, 1, 1, 1, 1, 1]), e[1] + p(0.5 * d[1], [1, 1, 0, 1, 1, 1]),
            e[2] + p(0.5 * d[2], [1, 1, 1, 1, 0, 1])]


def _exact_yee(c, seed):
    f = _yee_start(c["ncell"], seed, _dt(c)).double()
    e, h, every, energy = list(f[:3]), list(f[3:]), c["energy_every"], []
    for n in range(c["steps"]):
        h2 = _h_next(e, h)
        if every and n % every == 0:
            energy.append(0.5 * sum(float((v * v).sum()) for v in e) +
                          0.5 * sum(float((v * w).sum()) for v, w in zip(h, h2)))
        h, e = h2, _e_next(e, h2)
    out = {"f": torch.stack(e + h)}
    if every:
        out["energy"] = torch.tensor(energy, dtype=torch.float64)
    return out


def _exact_yee_eps(c, seed):
    f, eps, target = (v.double() for v in _eps_inputs(c, seed))
    eps.requires_grad_(True)
    e, h = list(f[:3]), list(f[3:])
    for _ in range(c["steps"]):
        h = _h_next(e, h)
        e = _e_next(e, h, eps)
    m, a = slice(1, -1), slice(0, -1)
    J = 0.5 * sum(((v - w)[s] ** 2).sum() for v, w, s in zip(e, target, ((m, m, a), (m, a, m), (a, m, m))))
    grad, = torch.autograd.grad(J, eps)
    return {"J": J.detach(), "grad": grad}


# EMFDTD curl stencils: destination, (left field, offset), (right field,
# offset), first node and end per axis (x, y, z); the PML index
# of a term is the distance to the nearer end along the term's axis.
EM_H = [(3, (1, (0, 0, 1)), (2, (0, 1, 0)), (1, 0, 0), (0, -1, -1)),
        (4, (2, (1, 0, 0)), (0, (0, 0, 1)), (0, 1, 0), (-1, 0, -1)),
        (5, (0, (0, 1, 0)), (1, (1, 0, 0)), (0, 0, 1), (-1, -1, 0))]
EM_D = [(6, (5, (0, -1, 0)), (4, (0, 0, -1)), (0, 0, 1), (-1, 0, 0)),
        (7, (3, (0, 0, -1)), (5, (-1, 0, 0)), (1, 0, 1), (0, -1, 0)),
        (8, (4, (-1, 0, 0)), (3, (0, -1, 0)), (1, 1, 0), (0, 0, -1))]
EM_PSI = {(0, 1): 12, (0, 2): 13, (1, 0): 14, (1, 2): 15, (2, 0): 16, (2, 1): 17, (3, 1): 18, (3, 2): 19, (4, 0): 20,
          (4, 2): 21, (5, 0): 22, (5, 1): 23}


def _em_curl(f, spec, n, s, tab):
    dest, left, right, lo, end = spec
    box = tuple(slice(lo[q], n + end[q]) for q in (2, 1, 0))
    terms = []
    for src, off in (left, right):
        axis = next(q for q in range(3) if off[q])
        ax = 2 - axis
        v = torch.cat([torch.zeros_like(f[src][_sl(ax, 0, 1)]), f[src], torch.zeros_like(f[src][_sl(ax, 0, 1)])], ax)
        moved = v[_sl(ax, 1 + off[axis], n + 1 + off[axis])]
        d = (moved - f[src])[box]
        i = torch.arange(lo[axis], n + end[axis], device="cuda")
        pml = torch.minimum(i, n - 1 + end[axis] - i).clamp(max=tab[3])
        shape = [-1 if q == ax else 1 for q in range(3)]
        b, cc, ook = (tab[q][pml].reshape(shape) for q in range(3))
        psi = f[EM_PSI[(src, axis)]]
        psi[box] = b * psi[box] + cc * d
        terms.append(ook * d + psi[box])
    old = f[dest][box] + s * (terms[0] - terms[1])
    f[dest].zero_()
    f[dest][box] = old


def _exact_emfdtd(c, seed):
    f, p, n = _em_inputs(c, seed), _em_params(c), c["n"]
    tab = [torch.tensor(list(v)[:c["d"] + 1], device="cuda", dtype=torch.float64) for v in (p.b, p.c, p.ook)] + [c["d"]]
    sink = []
    for step in range(c["steps"]):
        for spec in EM_H:
            _em_curl(f, spec, n, 0.5, tab)
        for spec in EM_D:
            _em_curl(f, spec, n, -0.5, tab)
        for q in range(3):
            f[q] = f[24] * (f[6 + q] - f[9 + q])
            f[9 + q] += f[25] * f[q]
        f[2, p.src[2], p.src[1], p.src[0]] = math.exp(-0.5 * ((10.0 - step) / 4.0) ** 2)
        sink.append(float(f[2, p.sink[2], p.sink[1], p.sink[0]]))
    return {"f": f[:12], "psi": f[12:24], "sink": torch.tensor(sink, dtype=torch.float64)}


def _exact_mri(c, seed):
    t, (rho, cp, lam, rho_b, c_b, omega, t_b, q, surf) = _mri_inputs(c, seed)
    h, p = _mri_params(c)
    rc, n = rho * cp, (c["nx"], c["ny"], c["nz"])
    open_skull = surf[-1:] == 1
    ta4 = (p.t_amb + 273.15) ** 4
    for _ in range(c["steps"]):
        v = t
        for axis in range(3):
            ax = 2 - axis
            a = 2 * h[axis] / lam
            lo, hi, e, w = t[_sl(ax, 0, 1)], t[_sl(ax, -1, None)], t[_sl(ax, 1, 2)], t[_sl(ax, -2, -1)]
            al, ah = a[_sl(ax, 0, 1)], a[_sl(ax, -1, None)]
            if axis < 2:
                last = 2 * w + ah * p.q_bc - 2 * hi
            else:
                tr4 = (v[_sl(ax, -1, None)] + 273.15) ** 4
                last = torch.where(open_skull, 2 * w - ah * p.h_conv * (hi - p.t_amb) -
                                   ah * p.epsilon * p.sigma * (tr4 - ta4), 2 * w + ah * p.q_skull) - 2 * hi
            d = torch.cat([2 * e + al * p.q_bc - 2 * lo, _second(t, ax), last], ax)
            v = v + p.tau * lam / rc * d / h[axis] ** 2
        t = v + p.tau * rho_b * c_b / rc * omega * (t_b - t) + p.tau / rc * q
    return {"t": _pad(t)}


def _exact_batch2d(c, seed):
    s = _batch_inputs(c, seed)
    n, off = s["n"].long(), s["off"]
    nodes = n * n
    u_out, J, G = torch.zeros_like(s["u0"], dtype=torch.float64), [], []
    for lo in range(0, c["nprob"], 1024):  # problems padded to one edge, some at a time
        hi = min(lo + 1024, c["nprob"])
        edge, cnt = int(n[lo:hi].max()), hi - lo
        a = torch.arange(edge, device="cuda")
        valid = (a[None, :, None] < n[lo:hi, None, None]) & (a[None, None, :] < n[lo:hi, None, None])
        inner = ((a > 0)[None, :, None] & (a > 0)[None, None, :] & (a[None, :, None] < n[lo:hi, None, None] - 1) &
                 (a[None, None, :] < n[lo:hi, None, None] - 1))[:, 1:-1, 1:-1]
        part = slice(int(off[lo]), int(off[hi - 1] + nodes[hi - 1]))
        u = torch.zeros((cnt, edge, edge), device="cuda", dtype=torch.float64)
        u[valid] = s["u0"][part].double()
        h2 = 1.0 / (n[lo:hi].double() - 1) ** 2
        k = (s["tau"][lo:hi].double() * s["kappa"][lo:hi].double() / h2).reshape(-1, 1, 1)
        k = torch.where(inner, k, torch.zeros_like(k))
        for _ in range(c["steps"]):
            lap = u[:, 1:-1, :-2] + u[:, 1:-1, 2:] + u[:, :-2, 1:-1] + u[:, 2:, 1:-1] - 4 * u[:, 1:-1, 1:-1]
            u[:, 1:-1, 1:-1] += k * lap
        u_out[part] = u[valid]
        t = torch.zeros_like(u)
        t[valid] = s["target"][part].double()
        if edge < 3:
            lap = torch.zeros_like(u[:, 1:-1, 1:-1])
        r = torch.where(inner, (u - t)[:, 1:-1, 1:-1], torch.zeros_like(lap))
        J.append(0.5 * (r * r).sum((1, 2)))
        G.append(c["steps"] * s["tau"][lo:hi].double() * (r * lap).sum((1, 2)) / h2)
    return {"u": u_out, "J": torch.cat(J), "grad": torch.cat(G)} if c["gradient"] else {"u": u_out}


EXACT = {"timelin": _exact_timelin, "heat": _exact_heat, "heatvar": _exact_heatvar, "pennes": _exact_pennes,
         "pennes_grad": _exact_pennes_grad, "kappa": _exact_kappa, "yee": _exact_yee, "yee_eps": _exact_yee_eps,
         "emfdtd": _exact_emfdtd, "mri": _exact_mri, "batch2d": _exact_batch2d}


def exact(case, seed):
    return EXACT[case["kind"]](case, seed)
