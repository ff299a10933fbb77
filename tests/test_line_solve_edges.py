"""Line lengths and shapes where the chunked line solves can go wrong.

Chunks hold 16 rows (32 in the refined FP32 solve of bounded lines), so the
lengths sit around multiples of both, at the shortest and longest lines, and
where the number of chunks per x wave or y/z workgroup changes. Reference: the
CPU oracle, with the repository's bars (1e-12 of max|ref| in FP64, 1e-6 for
FP32 fields). Bounded FP32 lines are checked in the FP64 solve mode; the refined
mode, whose error on such rough data passes the FP32 bar, is covered on smooth
fields in test_gpu_ops.py and test_host_plan.py.
"""
import ctypes

import numpy as np
import pytest
import torch

LENGTHS = [8, 9, 15, 16, 17, 31, 32, 33, 48, 49, 65, 127, 161, 255, 256, 257, 337, 512, 513, 1000, 1023, 1024]
KINDS = ["PERI", "NONE", "SYMM"]


def _spacing(n, kind):
    return (2 * np.pi * (n - 1) / n if kind == "PERI" else 1.0)


def _oracle(po, nn, kinds):
    from meshgen import mesh
    dom = [(0.0, _spacing(n, k) if n > 1 else 1.0, n) for n, k in zip(nn, kinds)]
    _, dd = mesh(dom)
    return po.Oracle(nn, dd, [k == "PERI" for k in kinds], symmetric=[[k == "SYMM"] * 2 for k in kinds]), dom


def _rel(got, ref):
    return np.abs(got - ref).max() / max(np.abs(ref).max(), 1e-300)


@pytest.mark.parametrize("kind", KINDS)
def test_emulated_lines_match_oracle(oracle_mod, kind):
    """Every length along x, y and z (each direction splits lines its own
    way), both members of the SYMM pair, through the host emulation."""
    from pyranda_amd import _lib as amd
    L = amd.lib()
    rng = np.random.default_rng(3)
    for n in LENGTHS:
        for d in range(3):
            nn = [8, 8, 8]
            nn[d] = n
            kinds = ["PERI"] * 3
            kinds[d] = kind
            P, dom = _oracle(oracle_mod, tuple(nn), kinds)
            h = ctypes.c_void_p()
            bc6 = (ctypes.c_int * 6)(*[amd.BC[k] for k in kinds for _ in (0, 1)])
            amd.check(L.pyr_setup_host(ctypes.byref(h), *nn, *[x for lo, hi, _ in dom for x in (lo, hi)], bc6))
            amd.check(L.pyr_set_r32_solve(h, amd.R32_SOLVE["fp64"]))
            v = np.asfortranarray(rng.standard_normal(nn) + 2.0)
            v32 = np.asfortranarray(v.astype(np.float32))
            for op in range(5):
                for anti in ((0, 1) if kind == "SYMM" else (0,)):
                    ref = P.apply_sym(op, d, -1, v) if anti else P.apply(op, d, v)
                    r32 = P.apply_sym(op, d, -1, v32.astype(float)) if anti else P.apply(op, d, v32.astype(float))
                    out, o32 = np.zeros(nn, order="F"), np.zeros(nn, dtype=np.float32, order="F")
                    o = op | (amd.OP_ANTISYM if anti else 0)
                    amd.check(L.pyr_host_emulate(h, o, d, amd.F64, v.ctypes.data, out.ctypes.data))
                    amd.check(L.pyr_host_emulate(h, o, d, amd.R32, v32.ctypes.data, o32.ctypes.data))
                    assert _rel(out, ref) <= 1e-12, (n, d, op, anti)
                    assert _rel(o32.astype(float), r32) <= 1e-6, (n, d, op, anti)
            L.pyr_destroy(h)


def _ctx(nn, kinds, dom):
    from pyranda_amd.parcop import ParcopContext
    return ParcopContext(nn, [d[0] for d in dom], [d[1] for d in dom], [k for k in kinds for _ in (0, 1)])


@pytest.mark.gpu
@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("n", LENGTHS)
def test_device_lines_match_oracle(oracle_mod, n, kind):
    """Line counts that leave the last wave or workgroup partly filled, on
    fields whose first element is 16-byte aligned and on ones off by one."""
    print("lines of", n, kind, flush=True)
    rng = np.random.default_rng(n)
    for d in range(3):
        nn = [9, 11, 10]
        nn[d] = n
        kinds = ["PERI"] * 3
        kinds[d] = kind
        P, dom = _oracle(oracle_mod, tuple(nn), kinds)
        ctx = _ctx(tuple(nn), kinds, dom)
        ctx.set_r32_solve("fp64")
        v = np.asfortranarray(rng.standard_normal(nn) + 2.0)
        for dtype, tol in ((torch.float64, 1e-12), (torch.float32, 1e-6)):
            flat = torch.from_numpy(np.ascontiguousarray(v.transpose(2, 1, 0))).to(dtype).reshape(-1)
            for off in (0, 1):
                buf = torch.empty(flat.numel() + off, dtype=dtype, device="cuda")
                buf[off:] = flat.cuda()
                vd = buf[off:].view(nn[2], nn[1], nn[0]).permute(2, 1, 0)
                host = vd.cpu().double().numpy()
                for op in range(5):
                    got = ctx.apply(op, d, vd).cpu().double().numpy()
                    assert _rel(got, P.apply(op, d, np.asfortranarray(host))) <= tol, (n, d, op, dtype, off)
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["PERI", "NONE"])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_nonfinite_values_spread_over_their_line(kind, dtype):
    """A NaN or infinity makes its whole implicit line non-finite, as the
    reference's whole-line sweeps do, and leaves every other line alone."""
    n = 1024
    print("non-finite", kind, dtype, flush=True)
    for d in range(3):
        nn = [8, 9, 10]
        nn[d] = n
        kinds = ["PERI"] * 3
        kinds[d] = kind
        dom = [(0.0, 1.0, m) for m in nn]
        ctx = _ctx(tuple(nn), kinds, dom)
        g = torch.Generator(device="cuda").manual_seed(1)
        v = torch.randn(tuple(reversed(nn)), generator=g, device="cuda", dtype=dtype).permute(2, 1, 0)
        for row, bad in ((0, float("nan")), (n - 1, float("nan")), (500, float("inf"))):
            w = v.permute(2, 1, 0).clone().permute(2, 1, 0)
            idx = [3, 4, 5]
            idx[d] = row
            w[tuple(idx)] = bad
            line = [3, 4, 5]
            line[d] = slice(None)
            for op in range(4):
                a, b = ctx.apply(op, d, v), ctx.apply(op, d, w)
                assert not torch.isfinite(b[tuple(line)]).any(), (d, op, row)
                b[tuple(line)] = a[tuple(line)]
                assert torch.equal(a, b), (d, op, row)
        ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("nn", [(40, 33, 1), (40, 1, 33), (1, 33, 40), (64, 3, 2), (2, 64, 1), (1, 3, 64), (2, 1, 3)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_null_directions_of_composites(nn, dtype):
    """Filters, ring, Laplacian and divergence on grids with directions too
    short for the operators: equal to the sweeps of all three directions one
    by one (a null direction copies or adds zero), NaN and infinity included."""
    from pyranda_amd import _lib as amd
    print("null directions", nn, dtype, flush=True)
    kinds = ["PERI" if n % 2 else "NONE" for n in nn]
    ctx = _ctx(nn, kinds, [(0.0, 1.0, n) for n in nn])
    g = torch.Generator(device="cuda").manual_seed(2)
    f = [torch.randn(tuple(reversed(nn)), generator=g, device="cuda", dtype=dtype).permute(2, 1, 0) for _ in range(3)]
    bad = f[0].clone()
    bad[0, 0, 0], bad[-1, -1, -1] = float("nan"), float("inf")
    for v in (f[0], bad):
        for name, op in (("sfilter", amd.OP_SFILTER), ("gfilter", amd.OP_GFILTER)):
            ref = v
            for d in range(3):
                ref = ctx.apply(op, d, ref)
            assert torch.equal(getattr(ctx, name)(v).nan_to_num(7.0), ref.nan_to_num(7.0)), name
            if name == "sfilter" and dtype == torch.float64:
                out, out32 = ctx.sfilter_rounded(v)
                assert torch.equal(out.nan_to_num(7.0), ref.nan_to_num(7.0))
                assert torch.equal(out32.nan_to_num(7.0), ref.float().nan_to_num(7.0))
        ref = None
        for d in range(3):
            ref = ctx.apply(amd.OP_D8, d, v, out=ref, epi=amd.EPI_MAXABS_SCALED if d else amd.EPI_ABS_SCALED,
                            epi_scale=ctx.dmesh[d] ** 2)
        assert torch.equal(ctx.pring(v).nan_to_num(7.0), ref.nan_to_num(7.0)), "ring"
        for name, op, fs in (("plaplacian", amd.OP_D2, (v, v, v)), ("divergence", amd.OP_D1, (v, f[1], f[2]))):
            ref = None
            for d in range(3):
                ref = ctx.apply(op, d, fs[d], out=ref, epi=amd.EPI_ADD if d else amd.EPI_STORE)
            got = ctx.plaplacian(v) if name == "plaplacian" else ctx.divergence(*fs)
            assert torch.equal(got.nan_to_num(7.0), ref.nan_to_num(7.0)), name
    # the refusals of the whole call hold for a direction that is not swept
    for call in ("pyr_plaplacian_f64", "pyr_sfilter_f64", "pyr_pring_f64"):
        p = ctypes.c_void_p(f[0].data_ptr())
        assert getattr(ctx._L, call)(ctx._h, p, p) != 0, call
    ctx.close()


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["PERI", "NONE"])
@pytest.mark.parametrize("n", [64, 71])
def test_every_epilogue_of_every_operator(n, kind):
    """Each operator and direction with each epilogue and with the FP32 copy,
    whole and ragged chunks: the epilogue of the stored result, to one rounding
    of the stored type (the fused forms round the result once, not twice)."""
    from pyranda_amd import _lib as amd
    print("epilogues", n, kind, flush=True)
    nn = (n, n, n)
    ctx = _ctx(nn, [kind] * 3, [(0.0, 1.0, n)] * 3)
    g = torch.Generator(device="cuda").manual_seed(4)
    for dtype in (torch.float64, torch.float32):
        eps = torch.finfo(dtype).eps
        v, old = [torch.randn(nn, generator=g, device="cuda", dtype=dtype).permute(2, 1, 0) for _ in range(2)]
        for op in range(5):
            for d in range(3):
                y = ctx.apply(op, d, v)
                for epi, want in ((amd.EPI_ADD, old.double() + y.double()),
                                  (amd.EPI_ABS_SCALED, 0.75 * y.double().abs()),
                                  (amd.EPI_MAXABS_SCALED, torch.maximum(old.double(), 0.75 * y.double().abs()))):
                    out = old.permute(2, 1, 0).clone().permute(2, 1, 0)
                    got = ctx.apply(op, d, v, out=out, epi=epi, epi_scale=0.75).double()
                    bar = 2 * eps * (old.double().abs() + y.double().abs())
                    assert ((got - want).abs() <= bar).all(), (op, d, epi, dtype)
                if dtype == torch.float64:
                    o32 = torch.empty(nn, device="cuda", dtype=torch.float32).permute(2, 1, 0)
                    assert torch.equal(ctx.apply(op, d, v, out32=o32), y) and torch.equal(o32, y.float()), (op, d)
                    assert torch.equal(ctx.apply_to32(op, d, v), y.float()), (op, d)
    ctx.close()
