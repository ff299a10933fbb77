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
