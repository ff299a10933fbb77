"""Device-resident replacement of pyranda's f2py module `parcop`.

pyranda reaches parcop only through pyrandaMPI (pyranda/pyrandaMPI.py:151-155
setup, :664-740 der/gfil/sfil). This shim keeps those method names and their
argument meaning, but fields are torch tensors resident on the GPU in the
reference's Fortran layout: shape (nx,ny,nz), x fastest (a permuted view of a
contiguous (nz,ny,nx) buffer). Every call enqueues HIP kernels from
libpyranda_amd.so on torch's current stream and returns a freshly allocated
output, like f2py's intent(out).

Precision: fields of dtype float64 go through the FP64 kernels; float32 fields
are solved in FP64 registers along periodic lines and, by default, in FP32 with
an FP64-residual refinement along bounded ones.
"""
import ctypes

import torch

from . import _lib


def empty_field(shape, dtype, device):
    """(nx,ny,nz) tensor with Fortran strides (x fastest)."""
    nx, ny, nz = shape
    return torch.empty_strided((nx, ny, nz), (1, nx, nx * ny), dtype=dtype, device=device)


_FIELD_TYPES = (torch.float64, torch.float32)


def is_fortran(t):
    nx, ny, nz = t.shape
    return t.stride() == (1, nx, nx * ny) or t.numel() <= 1 or _contig_equiv(t)


def _contig_equiv(t):
    nx, ny, nz = t.shape
    want = (1, nx, nx * ny)
    return all(s == w or n == 1 for s, w, n in zip(t.stride(), want, t.shape))


def _filter3(op):
    def f(ctx, v):
        a = ctx.apply(op, 0, v)
        b = ctx.apply(op, 1, a)
        return ctx.apply(op, 2, b)
    return f


def _ring(ctx, v):
    out = None
    for d in range(3):
        out = ctx.apply(_lib.OP_D8, d, v, out=out,
                        epi=_lib.EPI_ABS_SCALED if d == 0 else _lib.EPI_MAXABS_SCALED,
                        epi_scale=ctx.dmesh[d] ** 2)
    return out


def _lap(ctx, v):
    out = None
    for d in range(3):
        out = ctx.apply(_lib.OP_D2, d, v, out=out, epi=_lib.EPI_STORE if d == 0 else _lib.EPI_ADD)
    return out


def _d1(d):
    return lambda ctx, v: ctx.apply(_lib.OP_D1, d, v)


# the operator of each composite (timed launch by launch when it is timed)
_COMPOSITE_OP = {"sfilter": _lib.OP_SFILTER, "gfilter": _lib.OP_GFILTER, "pring": _lib.OP_D8,
                 "plaplacian": _lib.OP_D2, "ddx": _lib.OP_D1, "ddy": _lib.OP_D1, "ddz": _lib.OP_D1}

# the launches each composite makes, as separately timed apply() calls
_COMPOSITE = {
    "sfilter": _filter3(_lib.OP_SFILTER), "gfilter": _filter3(_lib.OP_GFILTER),
    "pring": _ring, "plaplacian": _lap, "ddx": _d1(0), "ddy": _d1(1), "ddz": _d1(2),
}


# relative gain the FP64 solve of an FP32 operator needs over the refined FP32
# solve before the autotuner picks it (the choice changes results)
SOLVE_MODE_MARGIN = 0.05

class ParcopContext:
    """One Cartesian block: parcop.setup(...) + the operator suite."""

    def __init__(self, nn, x1, xn, bcs, device="cuda"):
        self.nn = tuple(int(n) for n in nn)
        self.device = torch.device(device)
        if self.device.type == "cuda" and self.device.index is None:
            self.device = torch.device("cuda", torch.cuda.current_device())
        L = _lib.lib()
        h = ctypes.c_void_p()
        bc6 = (ctypes.c_int * 6)(*[_lib.BC[b] for b in bcs])
        self._bounded = tuple(_lib.BC[b] != _lib.BC["PERI"] for b in list(bcs)[::2])
        self._r32_solve, self._solve_tuned = "refined", {}
        _lib.check(L.pyr_setup(ctypes.byref(h), *self.nn, x1[0], xn[0], x1[1], xn[1],
                               x1[2], xn[2], bc6))
        self._h = h
        self._L = L
        self._strides = (1, self.nn[0], self.nn[0] * self.nn[1])
        dp = (ctypes.c_double * 3)()
        dm = (ctypes.c_double * 3)()
        gl = ctypes.c_double()
        _lib.check(L.pyr_mesh_scalars(h, dp, dm, ctypes.byref(gl)))
        self.dpatch = tuple(dp)
        self.dmesh = tuple(dm)
        self.gridlen = gl.value
        # optional per-launch timing: {(op, dir, dtype): [(start, end), ...]},
        # of every launch or, with timing_only a set of such keys, of those
        self.timing = None
        self.timing_only = None
        self.coords1d = []
        for ax in range(3):
            buf = (ctypes.c_double * self.nn[ax])()
            _lib.check(L.pyr_axis_coords(h, ax, buf))
            self.coords1d.append(list(buf))

    def set_r32_solve(self, name):
        """'refined' (default) or 'fp64': arithmetic of the solves on FP32 fields."""
        _lib.check(self._L.pyr_set_r32_solve(self._h, _lib.R32_SOLVE[name]))
        self._r32_solve = name

    def set_periodic_solver(self, name):
        """'circulant' (default) or 'lu': periodic implicit lines take the
        circulant solve in either setting; members of a group agree on it."""
        _lib.check(self._L.pyr_set_periodic_solver(self._h, _lib.PSOLVE[name]))

    def set_solve_tuning(self, op, direction, name=None):
        """FP32 solve arithmetic of one operator along one direction
        (pyr_set_solve_tuning): 'refined', 'fp64', or None for the context's."""
        _lib.check(self._L.pyr_set_solve_tuning(self._h, op, direction,
                                                -1 if name is None else _lib.R32_SOLVE[name]))
        self._solve_tuned[op, direction] = name

    def _two_solves(self, op, direction):
        """Whether FP32 fields have two solves to choose from here: bounded
        implicit lines (every other line is solved in FP64 in both modes)."""
        return self._bounded[direction] and op != _lib.OP_GFILTER

    def set_tuning(self, op, direction, dtype, x_lds_kb=-1, yz_pipe=-1, yz_lines=-1):
        """Per-operator knobs (pyr_set_tuning): lines per y/z workgroup
        (yz_lines) and, with yz_pipe 3 on y/z, the kernel with runtime row
        counts; x_lds_kb and the other values of yz_pipe are checked and change
        nothing; -1 = default."""
        prec = _lib.F64 if dtype == torch.float64 else _lib.R32
        _lib.check(self._L.pyr_set_tuning(self._h, op, direction, prec, int(x_lds_kb), int(yz_pipe),
                                          int(yz_lines)))

    def autotune(self, dtype, ops=None, reps=5, x_lds_kb=(8, 12, 16, 24, 40, 64, 80), seed=7, rounded=False,
                 solve_modes=False):
        """Time each operator and direction at this precision with every
        candidate (y/z: 64, 32 or 16 lines per workgroup; x lines and the
        refined FP32 solve of y/z lines have one shape, reported under the
        first of x_lds_kb and the default yz_lines, -1) on random fields and
        keep the fastest. The timed
        launches cycle through enough fields to exceed the device's 256 MB
        last-level cache, so every launch reads its input from HBM as the
        operators of a time step do. rounded: FP64
        z sweeps are timed storing the FP32 copy of their result as well (the
        last sweep of the filter of an FP32 run's FP64 state). solve_modes
        (FP32 fields): where there are two solves (bounded implicit lines) the
        candidates also range over the solve setting, refined FP32 or FP64
        (("r32_solve", 0 or 1) in the choice, 0 elsewhere); the two agree to
        the FP32 rounding of the result, so unlike the launch knobs this choice
        can change results in the last bits, and the FP64 solve is taken only
        when it is faster by SOLVE_MODE_MARGIN or more. Returns
        {(op, dir): (choice, {choice: mean ms})}."""
        ops = ops if ops is not None else (_lib.OP_D1, _lib.OP_D2, _lib.OP_D8, _lib.OP_SFILTER, _lib.OP_GFILTER)
        g = torch.Generator(device=self.device).manual_seed(seed)
        field_bytes = self.nn[0] * self.nn[1] * self.nn[2] * (8 if dtype == torch.float64 else 4)
        nfield = min(8, max(1, -(-(384 << 20) // field_bytes)))
        vs = [torch.randn(tuple(reversed(self.nn)), generator=g, device=self.device, dtype=dtype).permute(2, 1, 0)
              for _ in range(nfield)]
        v = vs[0]
        out = self._out(v)
        out32 = empty_field(self.nn, torch.float32, self.device) if rounded and dtype == torch.float64 else None
        report = {}
        for op in ops:
            for d in range(3):
                if self.nn[d] <= 3:
                    continue
                kw = {"out32": out32} if out32 is not None and d == 2 else {}
                two = dtype == torch.float32 and self._two_solves(op, d)
                if solve_modes and dtype == torch.float32:
                    solves = [((("r32_solve", m),), name) for m, name in enumerate(("refined", "fp64")[:1 + two])]
                else:
                    solves = [((), self._solve_tuned.get((op, d)) or self._r32_solve)]
                cands = []
                for pre, name in solves:
                    if d == 0:
                        shapes = [(("x_lds_kb", next(iter(x_lds_kb))), ("yz_pipe", 0))]
                    else:
                        lines = (-1,) if two and name == "refined" else (64, 32, 16)
                        shapes = [(("yz_pipe", 0), ("yz_lines", n)) for n in lines]
                    cands += [pre + c for c in shapes]
                times = {}
                for cand in cands:
                    self._set_choice(op, d, dtype, cand)
                    self.apply(op, d, v, out=out, **kw)
                    ev0 = torch.cuda.Event(enable_timing=True)
                    ev1 = torch.cuda.Event(enable_timing=True)
                    ev0.record()
                    for i in range(reps):
                        self.apply(op, d, vs[(i + 1) % nfield], out=out, **kw)
                    ev1.record()
                    torch.cuda.synchronize(self.device)
                    times[cand] = ev0.elapsed_time(ev1) / reps
                best = min(times, key=times.get)
                if solve_modes and dtype == torch.float32 and best[0] != ("r32_solve", 0):
                    # the solve arithmetic changes results: leave the refined
                    # FP32 solve only for a clear gain, so that timing noise
                    # does not decide which numerics run
                    ref = min((c for c in times if c[0] == ("r32_solve", 0)), key=times.get)
                    if times[best] > (1.0 - SOLVE_MODE_MARGIN) * times[ref]:
                        best = ref
                self._set_choice(op, d, dtype, best)
                report[(op, d)] = (best, times)
        return report

    def _set_choice(self, op, d, dtype, choice):
        kw = dict(choice)
        if "r32_solve" in kw:
            self.set_solve_tuning(op, d, ("refined", "fp64")[kw.pop("r32_solve")])
        self.set_tuning(op, d, dtype, **kw)

    def close(self):
        if getattr(self, "_h", None) is not None and self._h.value:
            self._L.pyr_destroy(self._h)
            self._h = None

    def __del__(self):
        try:
            self.close()
        except Exception:
            pass

    # -- helpers ------------------------------------------------------------
    def _prep(self, v, dtype=None):
        # a field as the kernels take it, as in nearly every call: small fields
        # are bound by this host path (with the stream handle and the strided
        # allocation: fbar on 32^3 17.1 -> 13.2 us, gradient on 64^3 22.7 -> 16.1)
        if (torch.is_tensor(v) and v.shape == self.nn and v.stride() == self._strides
                and v.dtype in _FIELD_TYPES and (dtype is None or v.dtype == dtype) and v.device == self.device):
            return v
        if not torch.is_tensor(v):
            v = torch.full(self.nn, float(v), dtype=dtype or torch.float64, device=self.device)
        if v.device != self.device:
            raise ValueError("field on %s, expected %s" % (v.device, self.device))
        if tuple(v.shape) != self.nn:
            v = v.expand(self.nn)
        if dtype is not None and v.dtype != dtype:
            v = v.to(dtype)
        if v.dtype not in (torch.float64, torch.float32):
            v = v.to(torch.float64)
        if not _contig_equiv(v):
            v = v.permute(2, 1, 0).contiguous().permute(2, 1, 0)
        return v

    def _stream(self):
        self._L.pyr_set_stream(self._h, _lib.stream_of(self.device))

    def _out(self, like):
        return torch.empty_strided(self.nn, self._strides, dtype=like.dtype, device=self.device)

    @staticmethod
    def _ptr(t):
        return ctypes.c_void_p(t.data_ptr())

    @staticmethod
    def _suffix(t):
        return "f64" if t.dtype == torch.float64 else "r32"

    def apply(self, op, direction, v, out=None, epi=_lib.EPI_STORE, epi_scale=0.0, out32=None):
        """One directional operator (compact_operators.f90:13-497). out32
        (an FP32 field; FP64 y/z sweeps with the store epilogue) also
        receives the rounding of the result."""
        v = self._prep(v)
        if out is None:
            out = self._out(v)
        prec = _lib.F64 if v.dtype == torch.float64 else _lib.R32
        if out32 is not None and (v.dtype != torch.float64 or epi != _lib.EPI_STORE
                                  or out32.dtype != torch.float32 or not _contig_equiv(out32)
                                  or tuple(out32.shape) != self.nn):
            raise ValueError("out32: an FP32 field for the store epilogue of an FP64 sweep")
        self._stream()
        tkey = self.timing is not None and self._timed(
            (op, direction, str(v.dtype) + ("+float32" if out32 is not None else ""))) or None
        if tkey is not None:
            ev0 = torch.cuda.Event(enable_timing=True)
            ev1 = torch.cuda.Event(enable_timing=True)
            ev0.record()
        if out32 is not None:
            _lib.check(self._L.pyr_apply_rounded(self._h, op, direction, self._ptr(v), self._ptr(out),
                                                 self._ptr(out32)))
        else:
            _lib.check(self._L.pyr_apply(self._h, op, direction, prec, v.data_ptr(), out.data_ptr(), epi,
                                         float(epi_scale)))
        if tkey is not None:
            ev1.record()
            self.timing.setdefault(tkey, []).append((ev0, ev1))
        return out

    def _timed(self, key):
        """key if launches of this kind are being timed, else None."""
        if self.timing is None or (self.timing_only is not None and key not in self.timing_only):
            return None
        return key

    def _split_composite(self, op):
        """Time a composite launch by launch (its operator is being timed)."""
        return self.timing is not None and (self.timing_only is None or any(k[0] == op for k in self.timing_only))

    def apply_to32(self, op, direction, v):
        """One directional operator of an FP64 field whose result is stored
        only as its FP32 rounding (pyr_apply_to_r32): the FP64 sweep reads 8
        and writes 4 bytes per point."""
        v = self._prep(v)
        if v.dtype != torch.float64:
            raise ValueError("apply_to32 sweeps FP64 fields")
        out32 = empty_field(self.nn, torch.float32, self.device)
        self._stream()
        tkey = self._timed((op, direction, "torch.float64->float32"))
        if tkey is not None:
            ev0 = torch.cuda.Event(enable_timing=True)
            ev1 = torch.cuda.Event(enable_timing=True)
            ev0.record()
        _lib.check(self._L.pyr_apply_to_r32(self._h, op, direction, self._ptr(v), self._ptr(out32)))
        if tkey is not None:
            ev1.record()
            self.timing.setdefault(tkey, []).append((ev0, ev1))
        return out32

    def timing_summary(self):
        """{(op, dir, dtype): (launches, mean ms)} of the recorded launches."""
        torch.cuda.synchronize(self.device)
        out = {}
        for key, evs in (self.timing or {}).items():
            ms = [a.elapsed_time(b) for a, b in evs]
            out[key] = (len(ms), sum(ms) / len(ms))
        return out

    def _unary(self, name, v):
        if self.timing is not None and name in _COMPOSITE and self._split_composite(_COMPOSITE_OP[name]):
            return _COMPOSITE[name](self, v)
        v = self._prep(v)
        out = self._out(v)
        self._stream()
        _lib.check(getattr(self._L, "pyr_%s_%s" % (name, self._suffix(v)))(self._h, v.data_ptr(), out.data_ptr()))
        return out

    # -- parcop names (parcop.f90:202-379) ----------------------------------
    def ddx(self, v): return self._unary("ddx", v)
    def ddy(self, v): return self._unary("ddy", v)
    def ddz(self, v): return self._unary("ddz", v)
    def dd8x(self, v): return self.apply(_lib.OP_D8, 0, v)
    def dd8y(self, v): return self.apply(_lib.OP_D8, 1, v)
    def dd8z(self, v): return self.apply(_lib.OP_D8, 2, v)
    def plaplacian(self, v): return self._unary("plaplacian", v)
    def pring(self, v): return self._unary("pring", v)
    def sfilter(self, v): return self._unary("sfilter", v)

    def sfilter_rounded(self, v):
        """fbar of an FP64 field and the FP32 rounding of the result, both
        stored by the last sweep (FP32 runs that filter an FP64 state)."""
        v = self._prep(v)
        if v.dtype != torch.float64:
            raise ValueError("sfilter_rounded filters FP64 fields")
        out32 = empty_field(self.nn, torch.float32, self.device)
        if self._split_composite(_lib.OP_SFILTER):
            a = self.apply(_lib.OP_SFILTER, 0, v)
            b = self.apply(_lib.OP_SFILTER, 1, a)
            out = self.apply(_lib.OP_SFILTER, 2, b, out32=out32)
            return out, out32
        out = self._out(v)
        self._stream()
        _lib.check(self._L.pyr_sfilter_f64_rounded(self._h, self._ptr(v), self._ptr(out), self._ptr(out32)))
        return out, out32
    def gfilter(self, v): return self._unary("gfilter", v)

    def gfilterdir(self, v, direction):
        v = self._prep(v)
        out = self._out(v)
        self._stream()
        _lib.check(getattr(self._L, "pyr_gfilterdir_%s" % self._suffix(v))(
            self._h, self._ptr(v), self._ptr(out), int(direction)))
        return out

    def pringv(self, vx, vy, vz):
        vx = self._prep(vx)
        vy = self._prep(vy, vx.dtype)
        vz = self._prep(vz, vx.dtype)
        out = self._out(vx)
        for d in range(3):
            for comp, f in enumerate((vx, vy, vz)):
                first = d == 0 and comp == 0
                # the normal component takes the antisymmetric member at SYMM
                # ends (ringx(f,..,isymX) etc., operators.f90:661-671)
                op = _lib.OP_D8 | (_lib.OP_ANTISYM if comp == d else 0)
                self.apply(op, d, f, out=out,
                           epi=_lib.EPI_ABS_SCALED if first else _lib.EPI_MAXABS_SCALED,
                           epi_scale=self.dmesh[d])
        return out

    def grads(self, v):
        v = self._prep(v)
        outs = [self._out(v) for _ in range(3)]
        self._stream()
        _lib.check(getattr(self._L, "pyr_grads_%s" % self._suffix(v))(
            self._h, v.data_ptr(), *[o.data_ptr() for o in outs]))
        return outs

    def divergence(self, fx, fy, fz):
        fx = self._prep(fx)
        fy = self._prep(fy, fx.dtype)
        fz = self._prep(fz, fx.dtype)
        out = self._out(fx)
        self._stream()
        _lib.check(getattr(self._L, "pyr_divergence_%s" % self._suffix(fx))(
            self._h, fx.data_ptr(), fy.data_ptr(), fz.data_ptr(), out.data_ptr()))
        return out
