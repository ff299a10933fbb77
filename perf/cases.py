"""The work that a program built on pyranda_amd has it do, as timed cases.

Two kinds of case. `op` cases are one composite of the compact operators on
resident fields, called through ParcopContext (the device-resident parcop
module): the conservative filter fbar, the Gaussian filter gbar, the LAD ring,
the Laplacian, the gradient and the divergence, over the grid sizes, boundary
kinds and storage types that simulations use. `tg` and `kh` cases are whole
time steps: the 3-D Taylor-Green Euler+LAD step and a step of an ensemble of
wall-bounded Kelvin-Helmholtz layers on uneven grids.

`exact` restates the same operators as dense line matrices in FP64 torch, from
the schemes' published coefficients, without the package.
"""
import math

import numpy as np
import torch

GAMMA_TG, GAMMA_KH = 1.4, 5.0 / 3.0
OPS_IN = {"fbar": 1, "gbar": 1, "ring": 1, "lap": 1, "grad": 1, "div": 3}
OPS_OUT = {"fbar": 1, "gbar": 1, "ring": 1, "lap": 1, "grad": 3, "div": 1}


def _op(name, what, n, bc, dtype):
    """bc: one letter per direction, p(eriodic), n(one: bounded) or s(ymmetric)."""
    return {"name": name, "kind": "op", "what": what, "nx": n[0], "ny": n[1], "nz": n[2], "bc": bc, "dtype": dtype}


def listed():
    return [
        # the conservative filter on a test-size grid: three launches of a few
        # microseconds, what a small 3-D run or a unit test pays per call
        _op("fbar_32_f64", "fbar", (32, 32, 32), "ppp", "f64"),
        # velocity-gradient tensor rows of a small FP32 run
        _op("grad_64_f32", "grad", (64, 64, 64), "ppp", "f32"),
        # flux divergence on a ragged box with a symmetry plane, periodic
        # sides and bounded ends (both kinds of antisymmetric-pair ends)
        _op("div_ragged_f64", "div", (180, 130, 75), "spn", "f64"),
        # the 2-D filter of a Richtmyer-Meshkov run: bounded along the shock,
        # periodic across it, 1024-point lines
        _op("fbar_1024x512_f64", "fbar", (1024, 512, 1), "npp", "f64"),
        # Gaussian filter on long ragged FP32 lines, not a multiple of
        # anything the launches are shaped for
        _op("gbar_ragged_f32", "gbar", (1000, 301, 53), "npp", "f32"),
        # LAD ring of an FP32 run on the headline grid
        _op("ring_256_f32", "ring", (256, 256, 256), "ppp", "f32"),
        # the filter and the gradient of an FP64 run on the headline grid
        _op("fbar_256_f64", "fbar", (256, 256, 256), "ppp", "f64"),
        _op("grad_256_f64", "grad", (256, 256, 256), "ppp", "f64"),
        # a bounded FP64 Laplacian (heat equation), every line solved by the
        # bounded solver
        _op("lap_192_f64", "lap", (192, 192, 192), "nnn", "f64"),
        # the largest field a context takes at 512 points a side
        _op("grad_512_f64", "grad", (512, 512, 512), "ppp", "f64"),
        # the headline step: 3-D Taylor-Green, five RK stages
        {"name": "tg_256_f64", "kind": "tg", "n": 256, "precision": "fp64"},
        # one step of an ensemble of wall-bounded layers, uneven grids, FP32
        {"name": "kh_group_24_f32", "kind": "kh", "members": 24, "lo": 128, "hi": 1024, "sizes_seed": 2024,
         "precision": "fp32"},
    ]


def _log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    r = rng.random()
    if r < 0.06:
        return {"kind": "tg", "n": int(_log_uniform(rng, 24, 200)), "precision": "fp64"}
    if r < 0.12:
        return {"kind": "kh", "members": rng.randint(2, 16), "lo": 96, "hi": rng.choice([256, 512, 776]),
                "sizes_seed": rng.randint(0, 10 ** 6), "precision": rng.choice(["fp32", "fp64"])}
    dims = rng.choices([1, 2, 3], [1, 5, 16])[0]
    n = [1, 1, 1]
    pts = _log_uniform(rng, *{1: (64, 1024), 2: (2 ** 12, 2 ** 20), 3: (2 ** 14, 2 ** 26)}[dims])
    side = pts ** (1.0 / dims)
    for d in range(dims):
        n[d] = int(min(max(side * _log_uniform(rng, 0.5, 2.0), 16), 1024)) if dims > 1 else int(pts)
        # solvers' own grids are often multiples of 8 or 32, users' often not
        m = rng.choice([1, 1, 8, 32])
        n[d] = max(16, n[d] // m * m)
    bc = "".join(rng.choices("pns", [60, 25, 15])[0] if n[d] > 1 else "p" for d in range(3))
    return {"kind": "op", "what": rng.choice(sorted(OPS_IN)), "nx": n[0], "ny": n[1], "nz": n[2], "bc": bc,
            "dtype": rng.choice(["f64", "f64", "f32"])}


# -- inputs --------------------------------------------------------------------
def _dtype(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _extent(n):
    """(first, last) node of each direction of a box with 2 pi periods."""
    return [(0.0, 2.0 * math.pi * (m - 1) / m if m > 1 else 1.0) for m in n]


def _fields(case, seed):
    """Turbulence-like fields: 12 product modes with a -5/3 spectrum up to a
    quarter of each direction's Nyquist wavenumber, plus 1% grid-scale noise."""
    n = (case["nx"], case["ny"], case["nz"])
    rng = np.random.default_rng(seed)
    gen = torch.Generator(device="cuda").manual_seed(seed)
    out = []
    for _ in range(OPS_IN[case["what"]]):
        f = 0.01 * torch.randn((n[2], n[1], n[0]), generator=gen, device="cuda", dtype=torch.float64)
        for _ in range(12):
            axes, k2 = [], 1.0
            for m in n:
                k = float(rng.integers(0, max(1, m // 8) + 1)) if m > 1 else 0.0
                k2 += k * k
                ph = rng.uniform(0.0, 2.0 * math.pi)
                axes.append(torch.cos(2.0 * math.pi * k * torch.arange(m, device="cuda", dtype=torch.float64) / m + ph))
            amp = k2 ** (-5.0 / 6.0)
            f += amp * axes[2][:, None, None] * axes[1][None, :, None] * axes[0][None, None, :]
        out.append(f.to(_dtype(case)).permute(2, 1, 0))
    return out


def _tg_inputs(seed):
    """Phases and amplitude of a Taylor-Green vortex at Mach 0.1."""
    rng = np.random.default_rng(seed)
    ph = rng.uniform(0.0, 2.0 * math.pi, 3)
    return [float(a) for a in ph], float(rng.uniform(0.8, 1.2))


def _kh_sizes(case):
    rng = np.random.default_rng(case["sizes_seed"])
    lo, hi = case["lo"], case["hi"]
    size = lambda: int(min(max(8 * round(_np_log_uniform(rng, lo, hi) / 8), lo), hi))  # noqa: E731
    return [(size(), size()) for _ in range(case["members"])]


def _np_log_uniform(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def _kh_inputs(seed):
    """Wavenumbers, amplitudes and phases of the interface perturbation."""
    rng = np.random.default_rng(seed)
    ks = [int(k) for k in rng.choice(np.arange(1, 9), size=6, replace=False)]
    a = rng.uniform(0.5, 1.0, 6)
    return ks, [float(x) for x in 0.1 * a / a.sum()], [float(x) for x in rng.uniform(0.0, 2.0 * math.pi, 6)]


def prepare(case, seed):
    import pyranda_amd as pr
    if case["kind"] == "op":
        from pyranda_amd.parcop import ParcopContext
        n = (case["nx"], case["ny"], case["nz"])
        ext = _extent(n)
        names = {"p": "PERI", "n": "NONE", "s": "SYMM"}
        ctx = ParcopContext(n, [e[0] for e in ext], [e[1] for e in ext], [names[b] for b in case["bc"] for _ in (0, 1)])
        call = {"fbar": ctx.sfilter, "gbar": ctx.gfilter, "ring": ctx.pring, "lap": ctx.plaplacian,
                "grad": ctx.grads, "div": ctx.divergence}[case["what"]]
        return {"kind": "op", "call": call, "fields": _fields(case, seed), "ctx": ctx}
    from pyranda_amd import workloads
    if case["kind"] == "tg":
        n = case["n"]
        (a, b, c), u0 = _tg_inputs(seed)
        dom = "(0.0, %r, %d, periodic=True)" % (2.0 * math.pi * (n - 1) / n, n)
        ss = pr.pyrandaSim("TGvortex", "xdom = %s\nydom = %s\nzdom = %s" % (dom, dom, dom), silent=True,
                           precision=case["precision"], device_scalars=True)
        ss.addPackage(pr.pyrandaTimestep(ss))
        ss.EOM(workloads.TG_EOM)
        ic = workloads.TG_IC.replace("p0 = 100.0", "p0 = %r" % (1.0 / (GAMMA_TG * 0.01))).replace("u0 = 1.0", "u0 = %r" % u0)
        # a third velocity component as large as a tenth of the others
        ic = ic.replace(":w: = 0.0*:u:", ":w: = 0.1*u0*cos(meshx/L)*cos(meshy/L)*sin(meshz/L)")
        ss.setIC(ic.replace("meshx/L", "(meshx/L + %r)" % a).replace("meshy/L", "(meshy/L + %r)" % b)
                 .replace("meshz/L", "(meshz/L + %r)" % c))
        return {"kind": "tg", "sim": ss, "time": 0.0, "dt": 0.5 * float(ss.variables["dt"].data)}
    ks, amp, ph = _kh_inputs(seed)
    pert = " + ".join("%r*sin(%r*meshx + %r)" % (amp[m], 2.0 * math.pi * ks[m], ph[m]) for m in range(len(ks)))
    ic = """
:u:   = 0.5*tanh( (meshy - 0.5)/0.025 )
:rho: = 1.5 + 0.5*tanh( (meshy - 0.5)/0.025 )
:v:   = ( PERT )*exp( -((meshy - 0.5)/0.1)**2 )
:p:   = P0 + 0.0*meshx
:Et: = :p:/( GAMMA - 1.0 ) + .5*:rho:*(:u:*:u: + :v:*:v:)
:rhou: = :rho:*:u:
:rhov: = :rho:*:v:
:cs:  = sqrt( :p: / :rho: * GAMMA )
:dt: = dt.courant(:u:,:v:,:w:,:cs:)*.1
""".replace("PERT", pert).replace("P0", repr(_KH_P0)).replace("GAMMA", repr(GAMMA_KH))
    meshes = ["xdom = (0.0, %r, %d, periodic=True)\nydom = (0.0, 1.0, %d)" % ((nx - 1.0) / nx, nx, ny)
              for nx, ny in _kh_sizes(case)]
    g = pr.pyrandaGroupSim("KH-walls", meshes, precision=case["precision"])
    g.addPackage(pr.pyrandaTimestep(g))
    g.addPackage(pr.pyrandaBC(g))
    g.EOM(workloads.KH_EOM + workloads.KH_WALL_BC, {"gamma": GAMMA_KH, "R0": 1.0, "cv": _KH_CV})
    g.setIC(ic)
    dt = g.var("dt").data
    return {"kind": "kh", "sim": g, "st": {"time": torch.zeros_like(dt), "dt": dt.clone()}}


def run(state):
    if state["kind"] == "op":
        return state["call"](*state["fields"])
    ss = state["sim"]
    if state["kind"] == "tg":
        state["time"] = ss.rk4(state["time"], state["dt"])
        out = {k: ss.variables[k].data for k in ("rho", "rhou", "rhov", "rhow", "Et")}
        out["dt"] = ss.variables["dt"].data
        return out
    from pyranda_amd.workloads import kh_advance
    kh_advance(ss, state["st"])
    # every member's points back to back (their counts are multiples of 64: no padding)
    out = {k: ss.variables[k].data for k in ("rho", "rhou", "rhov", "Et")}
    out["dt"] = state["st"]["dt"]
    return out


def work(case):
    """Each input read once and each output written once; about 20 operations
    a point for each line sweep (right-hand side and banded solve) and as many
    for the pointwise algebra that goes with it."""
    if case["kind"] == "op":
        pts = case["nx"] * case["ny"] * case["nz"]
        live = sum(case[k] > 3 for k in ("nx", "ny", "nz"))
        size = 8 if case["dtype"] == "f64" else 4
        return {"bytes": pts * size * (OPS_IN[case["what"]] + OPS_OUT[case["what"]]), "flops": 20 * live * pts}
    size = 8 if case["precision"] == "fp64" else 4
    if case["kind"] == "tg":
        # state in and out; 5 stages of 15 flux, 9 gradient, 15 filter and 12 LAD sweeps
        return {"bytes": 10 * size * case["n"] ** 3, "flops": 5 * 51 * 40 * case["n"] ** 3}
    pts = sum(nx * ny for nx, ny in _kh_sizes(case))
    # 5 stages of 8 flux, 6 gradient, 8 filter and 12 LAD sweeps
    return {"bytes": 8 * size * pts, "flops": 5 * 34 * 40 * pts}


# -- the same in FP64 torch: dense line matrices -----------------------------
# Schemes: left-hand rows (offsets -2..2), right-hand rows (-4..4), the four
# rows at a bounded end (the other end mirrors them), and the parity that maps
# an even function's ghost points on each side of the system.
def _pad(rows, width):
    out = np.zeros((len(rows), width))
    for i, r in enumerate(rows):
        k = (width - len(r)) // 2
        out[i, k:k + len(r)] = r
    return out


def _scheme(op):
    if op == "d1":
        lhs, rhs = [0.45, 4.5, 9.0, 4.5, 0.45], [-0.015, -1.515, -6.375, 0.0, 6.375, 1.515, 0.015]
        bl = [[0, 0, 4.725, 9.45, 0], [0, 1.94578125, 7.783125, 1.94578125, 0],
              [0.2964375, 4.743, 10.67175, 4.743, 0.2964375],
              [0.451390625, 4.63271875, 9.38146875, 4.63271875, 0.451390625]]
        br = [[0, 0, 0, -11.8125, 9.45, 2.3625, 0], [0, 0, -5.83734375, 0, 5.83734375, 0, 0],
              [0, -1.23515625, -7.905, 0, 7.905, 1.23515625, 0],
              [-0.015, -1.53, -6.66984375, 0, 6.66984375, 1.53, 0.015]]
        return lhs, rhs, bl, br, -1.0
    if op == "d2":
        lhs, rhs = [387.0, 6012.0, 16182.0, 6012.0, 387.0], [79.0, 4671.0, 9585.0, -28670.0, 9585.0, 4671.0, 79.0]
        bl = [[0, 0, 1, 11, 0], [0, 1, 10, 1, 0], [23, 688, 2358, 688, 23], lhs]
        br = [[0, 0, 0, 13, -27, 15, -1], [0, 0, 12, -24, 12, 0, 0], [0, 465, 1920, -4770, 1920, 465, 0], rhs]
        return lhs, rhs, bl, br, 1.0
    if op == "d8":
        lhs = [1.5, 14.0, 29.0, 14.0, 1.5]
        rhs = [60.0, -480.0, 1680.0, -3360.0, 4200.0, -3360.0, 1680.0, -480.0, 60.0]
        bl = [[0, 0, 43, 15.5, 1.5], [0, 15.5, 29, 14, 1.5], lhs, lhs]
        br = [[0, 0, 0, 0, 840, -1680, 1200, -420, 60], [0, 0, 0, -1680, 3720, -3300, 1680, -480, 60],
              [0, 0, 1200, -3300, 4200, -3360, 1680, -480, 60], [0, -420, 1680, -3360, 4200, -3360, 1680, -480, 60]]
        return lhs, rhs, bl, br, 1.0
    if op == "sf":
        lhs = [1.6688e-1, 6.6624e-1, 1.0, 6.6624e-1, 1.6688e-1]
        rhs = [-5e-6, 4e-5, 1.6674e-1, 6.6652e-1, 9.9965e-1, 6.6652e-1, 1.6674e-1, 4e-5, -5e-6]
        bl = [[0, 0, 1, 0, 0], [0, 4.997e-1, 1, 4.997e-1, 0], lhs, lhs]
        br = [[0, 0, 0, 0, 1, 0, 0, 0, 0], [0, 0, 0, 4.9985e-1, 9.997e-1, 4.9985e-1, 0, 0, 0],
              [0, 0, 1.668e-1, 6.6656e-1, 9.9952e-1, 6.6656e-1, 1.668e-1, 0, 0],
              [0, 4e-5, 1.6672e-1, 6.6652e-1, 9.9968e-1, 6.6652e-1, 1.6672e-1, 4e-5, 0]]
        return lhs, rhs, bl, br, 1.0
    a, b, c, d, e = 3565 / 10368, 3091 / 12960, 1997 / 25920, 149 / 12960, 107 / 103680
    rhs = [e, d, c, b, a, b, c, d, e]
    br = [[0, 0, 0, 0, a + b, b + c, c + d, d + e, e], [0, 0, 0, b + c, a + d, b + e, c, d, e],
          [0, 0, c + d, b + e, a, b, c, d, e], [0, d + e, c, b, a, b, c, d, e]]
    return [0, 0, 1, 0, 0], rhs, [[0, 0, 1, 0, 0]] * 4, br, 1.0


def _line_matrix(op, n, bc, anti=False):
    """The n x n matrix A^-1 B of one operator along one direction (unit spacing)."""
    lhs, rhs, bl, br, parity = _scheme(op)
    sides = []
    odd_rows = -1.0 if op == "d1" else 1.0
    for inner, rows, mirror_sign, ghost_sign in ((lhs, bl, 1.0, parity), (rhs, br, odd_rows, 1.0)):
        w = 2 if len(inner) == 5 and inner is lhs else 4
        inner, rows = _pad([inner], 2 * w + 1)[0], _pad(rows, 2 * w + 1)
        ghost = -ghost_sign if anti else ghost_sign
        m = np.zeros((n, n))
        for i in range(n):
            row = inner
            if bc == "n" and i < 4:
                row = rows[i]
            if bc == "n" and i >= n - 4:
                row = mirror_sign * rows[n - 1 - i][::-1]
            for o in range(-w, w + 1):
                c = row[o + w]
                if c == 0.0:
                    continue
                j = i + o
                if bc == "p":
                    m[i, j % n] += c
                elif j < 0:
                    m[i, -1 - j] += ghost * c
                elif j >= n:
                    m[i, 2 * n - 1 - j] += ghost * c
                else:
                    m[i, j] += c
        sides.append(m)
    if op == "gf":
        return sides[1]
    if op == "sf":  # nearly the identity: solve for what the filter changes
        return np.eye(n) + np.linalg.solve(sides[0], sides[1] - sides[0])
    return np.linalg.solve(sides[0], sides[1])


class _Plain:
    """The operators on (nz, ny, nx) FP64 tensors of one box."""

    def __init__(self, n, bc, spacing):
        self.n, self.bc, self.h = n, bc, spacing
        self.live = [d for d in range(3) if n[d] > 3]
        widest = [max(spacing[e] for e in range(3) if e != d) if n[d] == 1 else spacing[d] for d in range(3)]
        self.mesh_h, self.gridlen = widest, min(widest)
        self._m = {}

    def along(self, op, d, f, anti=False):
        key = (op, d, anti and self.bc[d] == "s")
        if key not in self._m:
            self._m[key] = torch.from_numpy(_line_matrix(op, self.n[d], self.bc[d], key[2])).to(f.device)
        m = self._m[key]
        if d == 0:
            return torch.matmul(f, m.t().contiguous())
        if d == 1:
            return torch.matmul(m, f)
        return torch.matmul(m, f.reshape(f.shape[0], -1)).reshape(f.shape)

    def d1(self, d, f, anti=False):
        return self.along("d1", d, f, anti) / self.h[d] if d in self.live else torch.zeros_like(f)

    def filt(self, op, f):
        for d in self.live:
            f = self.along(op, d, f)
        return f

    def ring(self, f):
        out = torch.zeros_like(f)
        for d in self.live:
            out = torch.maximum(out, self.along("d8", d, f).abs() * self.mesh_h[d] ** 2)
        return out

    def lap(self, f):
        return sum(self.along("d2", d, f) / self.h[d] ** 2 for d in self.live)

    def courant(self, u, v, w, c):
        h = self.mesh_h
        return 1.0 / (u.abs() / h[0] + v.abs() / h[1] + w.abs() / h[2] + c.abs() / self.gridlen).max()

    def diff(self, bulk, rho):
        return (rho * self.gridlen ** 2 / bulk.clamp(min=1e-12)).min()


_RK_A = [0.0, -6234157559845. / 12983515589748., -6194124222391. / 4410992767914.,
         -31623096876824. / 15682348800105., -12251185447671. / 11596622555746.]
_RK_B = [494393426753. / 4806282396855., 4047970641027. / 5463924506627., 9795748752853. / 13190207949281.,
         4009051133189. / 8539092990294., 1348533437543. / 7166442652324.]
_KH_P0 = (1.0 / 0.3) ** 2 / GAMMA_KH
_KH_CV = 1.0 / (1.0 - 1.0 / GAMMA_KH) - 1.0


def _rk_step(fluxes, update, U, V, dt):
    phi = {k: torch.zeros_like(a) for k, a in U.items()}
    for a, b in zip(_RK_A, _RK_B):
        F = fluxes(U, V)
        for k in U:
            phi[k] = dt * F[k] + a * phi[k]
            U[k] = U[k] + b * phi[k]
        update(U, V)


def _tg_exact(case, seed):
    n, g = case["n"], GAMMA_TG
    h = 2.0 * math.pi / n
    P = _Plain((n, n, n), "ppp", (h, h, h))
    (a, b, c), u0 = _tg_inputs(seed)
    s = torch.arange(n, device="cuda", dtype=torch.float64) * h
    X, Y, Z = s[None, None, :] + a, s[None, :, None] + b, s[:, None, None] + c
    one = torch.ones((n, n, n), device="cuda", dtype=torch.float64)
    u = u0 * torch.sin(X) * torch.cos(Y) * torch.cos(Z) * one
    v = -u0 * torch.cos(X) * torch.sin(Y) * torch.cos(Z) * one
    w = 0.1 * u0 * torch.cos(X) * torch.cos(Y) * torch.sin(Z) * one
    # the string's 2.*meshx/L holds the shifted angle too
    x2, y2, z2 = 2.0 * X, 2.0 * Y, 2.0 * Z
    p = 1.0 / (g * 0.01) + 1.0 / 16.0 * ((torch.cos(x2) + torch.cos(y2)) * (torch.cos(z2) + 2.0) - 2.0) * one
    rho = one.clone()
    U = {"rho": rho, "rhou": rho * u, "rhov": rho * v, "rhow": rho * w,
         "Et": p / (g - 1.0) + 0.5 * rho * (u * u + v * v + w * w)}
    V = {}

    def update(U, V):
        for k in U:
            U[k] = P.filt("sf", U[k])
        rho = U["rho"]
        u, v, w = U["rhou"] / rho, U["rhov"] / rho, U["rhow"] / rho
        p = (U["Et"] - .5 * rho * (u * u + v * v + w * w)) * (g - 1.0)
        ux, uy, uz = (P.d1(d, u) for d in range(3))
        vx, vy, vz = (P.d1(d, v) for d in range(3))
        wx, wy, wz = (P.d1(d, w) for d in range(3))
        div = ux + vy + wz
        S = torch.sqrt(ux * ux + vy * vy + wz * wz + .5 * ((uy + vx) ** 2 + (uz + wx) ** 2 + (vz + wy) ** 2))
        mu = P.filt("gf", P.ring(S)) * rho * 1.0e-4
        beta = P.filt("gf", P.ring(div) * rho) * 7.0e-3
        tau = (beta - 2. / 3. * mu) * div - p
        cs = torch.sqrt(p / rho * g)
        dt = torch.minimum(P.courant(u, v, w, cs), 0.2 * P.diff(beta, rho))
        V.update(u=u, v=v, w=w, xx=2.0 * mu * ux + tau, yy=2.0 * mu * vy + tau, zz=2.0 * mu * wz + tau,
                 # the reference's equation for tauyz adds wz, not wy
                 xy=mu * (uy + vx), xz=mu * (uz + wx), yz=mu * (vz + wz), dt=torch.minimum(dt, 0.2 * P.diff(mu, rho)))

    def fluxes(U, V):
        u, v, w = V["u"], V["v"], V["w"]
        xx, yy, zz, xy, xz, yz = (V[k] for k in ("xx", "yy", "zz", "xy", "xz", "yz"))
        div = lambda A, B, C: -P.d1(0, A) - P.d1(1, B) - P.d1(2, C)  # noqa: E731
        r, ru, rv, rw, E = (U[k] for k in ("rho", "rhou", "rhov", "rhow", "Et"))
        return {"rho": div(r * u, r * v, r * w),
                "rhou": div(ru * u - xx, ru * v - xy, ru * w - xz),
                "rhov": div(rv * u - xy, rv * v - yy, rv * w - yz),
                "rhow": div(rw * u - xz, rw * v - yz, rw * w - zz),
                "Et": div((E - xx) * u - xy * v - xz * w, (E - yy) * v - xy * u - yz * w,
                          (E - zz) * w - xz * u - yz * v)}

    cs = torch.sqrt(p / rho * g)
    V["dt"] = P.courant(u, v, w, cs)
    update(U, V)
    dt = 0.5 * float(V["dt"])
    _rk_step(fluxes, update, U, V, dt)
    out = {k: U[k].permute(2, 1, 0) for k in U}
    out["dt"] = V["dt"]
    return out


def _kh_exact(case, seed):
    g, cv = GAMMA_KH, _KH_CV
    ks, amp, ph = _kh_inputs(seed)
    out, dts = {}, []
    for m, (nx, ny) in enumerate(_kh_sizes(case)):
        h = (1.0 / nx, 1.0 / (ny - 1.0), 1.0)
        P = _Plain((nx, ny, 1), "pnp", h)
        x = torch.arange(nx, device="cuda", dtype=torch.float64)[None, None, :] * h[0]
        y = torch.arange(ny, device="cuda", dtype=torch.float64)[None, :, None] * h[1]
        t = torch.tanh((y - 0.5) / 0.025) + 0.0 * x
        u, rho = 0.5 * t, 1.5 + 0.5 * t
        v = sum(amp[i] * torch.sin(2.0 * math.pi * ks[i] * x + ph[i]) for i in range(len(ks))) * torch.exp(-((y - 0.5) / 0.1) ** 2)
        p = _KH_P0 + 0.0 * t
        U = {"rho": rho, "rhou": rho * u, "rhov": rho * v, "Et": p / (g - 1.0) + .5 * rho * (u * u + v * v)}
        zero = torch.zeros_like(rho)
        V = {"dt": 0.1 * P.courant(u, v, zero, torch.sqrt(p / rho * g))}

        def update(U, V):
            for k in U:
                U[k] = P.filt("sf", U[k])
            rho = U["rho"]
            u, v = U["rhou"] / rho, U["rhov"] / rho
            p = (U["Et"] - .5 * rho * (u * u + v * v)) * (g - 1.0)
            ux, uy, vx, vy = P.d1(0, u), P.d1(1, u), P.d1(0, v), P.d1(1, v)
            div = ux + vy
            mu = P.filt("gf", P.ring(torch.sqrt(ux * ux + vy * vy + .5 * (uy + vx) ** 2))) * rho * 1.0e-4
            beta = P.filt("gf", P.ring(div) * rho) * 7.0e-3
            tau = (beta - 2. / 3. * mu) * div - p
            T = p / rho
            V.update(xx=2.0 * mu * ux + tau, yy=2.0 * mu * vy + tau, xy=mu * (uy + vx), tx=P.d1(0, T), ty=P.d1(1, T),
                     kappa=P.filt("gf", P.ring(T) * rho * cv / (T * V["dt"])) * 1.0e-3)
            dt = torch.minimum(P.courant(u, v, zero, torch.sqrt(p / rho * g)), 0.2 * P.diff(beta, rho))
            V["dt"] = torch.minimum(dt, 0.2 * P.diff(mu, rho))
            # walls: extrapolated density and energy, no velocity
            for k in ("rho", "Et"):
                U[k][:, 0] = 2.0 * U[k][:, 1] - U[k][:, 2]
                U[k][:, -1] = 2.0 * U[k][:, -2] - U[k][:, -3]
            for a in (u, v):
                a[:, 0] = 0.0
                a[:, -1] = 0.0
            V.update(u=u, v=v)

        def fluxes(U, V):
            u, v, xx, yy, xy, kap = (V[k] for k in ("u", "v", "xx", "yy", "xy", "kappa"))
            r, ru, rv, E = (U[k] for k in ("rho", "rhou", "rhov", "Et"))
            return {"rho": -P.d1(0, r * u) - P.d1(1, r * v),
                    "rhou": -P.d1(0, ru * u - xx) - P.d1(1, ru * v - xy),
                    "rhov": -P.d1(0, rv * u - xy) - P.d1(1, rv * v - yy),
                    "Et": -P.d1(0, (E - xx) * u - xy * v - V["tx"] * kap)
                          - P.d1(1, (E - yy) * v - xy * u - V["ty"] * kap)}

        update(U, V)
        dt = V["dt"].clone()
        _rk_step(fluxes, update, U, V, dt)
        for k in U:
            out.setdefault(k, []).append(U[k].reshape(-1))
        dts.append(torch.clamp(torch.minimum(V["dt"], 1.1 * dt), max=1.0))
    out = {k: torch.cat(a).reshape(-1, 1, 1) for k, a in out.items()}
    out["dt"] = torch.stack(dts)
    return out


def exact(case, seed):
    """What run returns for these inputs, in FP64 (outputs in run's order)."""
    if case["kind"] == "tg":
        return _tg_exact(case, seed)
    if case["kind"] == "kh":
        return _kh_exact(case, seed)
    n = (case["nx"], case["ny"], case["nz"])
    h = [2.0 * math.pi / m if m > 1 else 1.0 for m in n]
    P = _Plain(n, case["bc"], h)
    fs = [f.permute(2, 1, 0).to(torch.float64) for f in _fields(case, seed)]
    what = case["what"]
    if what == "grad":
        return [P.d1(d, fs[0]).permute(2, 1, 0) for d in range(3)]
    r = {"fbar": lambda: P.filt("sf", fs[0]), "gbar": lambda: P.filt("gf", fs[0]), "ring": lambda: P.ring(fs[0]),
         "lap": lambda: P.lap(fs[0]), "div": lambda: sum(P.d1(d, fs[d], True) for d in range(3))}[what]()
    return r.permute(2, 1, 0)
