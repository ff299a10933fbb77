"""Bounded lines in the default solve modes: the refined FP32 solve at the
lengths where its chunks of up to 32 rows split in every way, and the autotuner's
choice of launch shapes and solve modes."""
import ctypes

import numpy as np
import pytest
import torch

from test_line_solve_edges import LENGTHS

FACES = [("NONE", "NONE"), ("SYMM", "SYMM"), ("NONE", "SYMM"), ("SYMM", "NONE")]


def _bounded(oracle_mod, run, others, faces, lengths, dtype):
    """Each implicit operator on smooth fields with 5% noise, against the oracle
    on the same values: the repository's bars, 1e-12 of max|ref| in FP64 and 1e-6
    for FP32 fields. The antisymmetric member gets fields that are odd about the
    faces."""
    bar = 1e-12 if dtype == np.float64 else 1e-6
    from meshgen import mesh
    rng = np.random.default_rng(8)
    for n in lengths:
        for d in range(3):
            nn = list(others)
            nn[d] = n
            dom = [(0.0, 1.0, m) for m in nn]
            _, dd = mesh(dom)
            P = oracle_mod.Oracle(tuple(nn), dd, [e != d for e in range(3)],
                                  symmetric=[[e == d and k == "SYMM" for k in faces] for e in range(3)])
            s = [((np.arange(m) + 0.5) / m).reshape([-1 if e == i else 1 for i in range(3)]) for e, m in enumerate(nn)]
            noise = 0.05 * rng.standard_normal(nn)
            cross = np.cos(s[(d + 1) % 3] + 2.0 * s[(d + 2) % 3])
            even = (2.0 + np.cos(3.0 * s[d]) * cross + noise).astype(dtype)
            odd = (np.sin(2.0 * np.pi * s[d]) * (cross + noise)).astype(dtype)
            kinds = ["PERI"] * 6
            kinds[2 * d:2 * d + 2] = faces
            apply, close = run(tuple(nn), kinds, d)
            for op in range(4):
                for anti in ((0, 1) if "SYMM" in faces else (0,)):
                    v = np.asfortranarray(odd if anti else even)
                    w = np.asfortranarray(v.astype(np.float64))
                    ref = P.apply_sym(op, d, -1, w) if anti else P.apply(op, d, w)
                    got = apply(op | (0x10 if anti else 0), v)
                    assert np.abs(got - ref).max() <= bar * np.abs(ref).max(), (n, d, op, anti)
            close()


@pytest.mark.parametrize("faces", FACES)
def test_emulated_refined_lines_match_oracle(oracle_mod, faces):
    from pyranda_amd import _lib as amd
    L = amd.lib()

    def run(nn, kinds, d):
        h = ctypes.c_void_p()
        bc6 = (ctypes.c_int * 6)(*[amd.BC[k] for k in kinds])
        amd.check(L.pyr_setup_host(ctypes.byref(h), *nn, 0.0, 1.0, 0.0, 1.0, 0.0, 1.0, bc6))

        def apply(op, v):
            out = np.zeros(nn, dtype=np.float32, order="F")
            amd.check(L.pyr_host_emulate(h, op, d, amd.R32, v.ctypes.data, out.ctypes.data))
            return out
        return apply, lambda: L.pyr_destroy(h)
    _bounded(oracle_mod, run, (2, 3, 2), faces, LENGTHS, np.float32)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("n", LENGTHS)
def test_device_bounded_lines_match_oracle(oracle_mod, n, dtype):
    """Line counts that leave the last wave or workgroup partly filled, on
    fields whose first element is 16-byte aligned and on ones off by one, which
    give the same bits."""
    from pyranda_amd.parcop import ParcopContext
    print("bounded lines of", n, dtype, flush=True)

    def run(nn, kinds, d):
        ctx = ParcopContext(nn, (0.0,) * 3, (1.0,) * 3, kinds)

        def apply(op, v):
            flat = torch.from_numpy(np.ascontiguousarray(v.transpose(2, 1, 0))).reshape(-1).cuda()
            got = []
            for off in (0, 1):
                buf, out = [torch.empty(flat.numel() + off, dtype=flat.dtype, device="cuda") for _ in range(2)]
                buf[off:] = flat
                vd, od = [b[off:].view(nn[2], nn[1], nn[0]).permute(2, 1, 0) for b in (buf, out)]
                got.append(ctx.apply(op, d, vd, out=od))
            assert torch.equal(*got), (nn, d, op)
            return got[0].cpu().numpy()
        return apply, ctx.close
    for faces in FACES:
        _bounded(oracle_mod, run, (9, 11, 10), faces, [n], dtype)


def _ctx(nn, kinds):
    from pyranda_amd.parcop import ParcopContext
    return ParcopContext(nn, (0.0,) * 3, (1.0,) * 3, [k for k in kinds for _ in (0, 1)])


@pytest.mark.gpu
@pytest.mark.parametrize("mode", ["refined", "fp64"])
def test_autotune_of_bounded_fp32_lines(mode):
    """One candidate where one launch exists (the refined solve), which leaves
    the FP64 solve's lines per workgroup at their default; results unchanged."""
    from pyranda_amd import _lib
    print("autotune of bounded lines", mode, flush=True)
    ctx = _ctx((40, 48, 33), ("PERI", "NONE", "SYMM"))
    ctx.set_r32_solve(mode)
    v = torch.rand((33, 48, 40), device="cuda", dtype=torch.float32).permute(2, 1, 0)
    before = {(op, d): ctx.apply(op, d, v) for op in range(5) for d in range(3)}
    rep = ctx.autotune(torch.float32, reps=2)
    for (op, d), (best, times) in rep.items():
        one = d == 0 or (mode == "refined" and op != _lib.OP_GFILTER)
        assert len(times) == (1 if one else 3) and best in times, (op, d)
        assert torch.equal(ctx.apply(op, d, v), before[op, d]), (op, d)
    ctx.close()


@pytest.mark.gpu
def test_autotune_solve_modes_of_bounded_lines():
    """Bounded implicit lines range over both solves, every other line keeps
    the one it has; each result is that of a context in the chosen mode."""
    from pyranda_amd import _lib
    print("autotune of solve modes", flush=True)
    nn, kinds = (40, 48, 33), ("NONE", "NONE", "PERI")
    ctx, ref = _ctx(nn, kinds), [_ctx(nn, kinds) for _ in range(2)]
    ref[1].set_r32_solve("fp64")
    v = torch.rand(tuple(reversed(nn)), device="cuda", dtype=torch.float32).permute(2, 1, 0)
    rep = ctx.autotune(torch.float32, reps=2, solve_modes=True)
    for (op, d), (best, times) in rep.items():
        modes = {c[0] for c in times}
        both = d < 2 and op != _lib.OP_GFILTER
        assert modes == {("r32_solve", m) for m in range(1 + both)}, (op, d)
        assert torch.equal(ctx.apply(op, d, v), ref[best[0][1]].apply(op, d, v)), (op, d)
    for c in [ctx] + ref:
        c.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
@pytest.mark.parametrize("kinds", [("PERI", "PERI", "PERI"), ("NONE", "NONE", "PERI"), ("PERI", "NONE", "NONE")])
def test_grouped_launches_equal_single_ones(kinds, dtype):
    """Members of very different line lengths, a null direction and starts that
    are not 16-byte aligned among them, in one launch: each member's result is
    its own sweep's, bit for bit, for every operator and epilogue, and nothing
    between the members is written."""
    from pyranda_amd import _lib
    print("grouped launches", kinds, dtype, flush=True)
    sizes = [(8, 9, 10), (64, 40, 16), (1000, 12, 8), (33, 1024, 1), (17, 31, 129), (256, 16, 3), (9, 700, 8)]
    ctxs = [_ctx(n, kinds) for n in sizes]
    offs, at = [], 0
    for i, n in enumerate(sizes):
        offs.append(at)
        at += n[0] * n[1] * n[2] + (16, 1, 3)[i % 3]
    L, h = _lib.lib(), ctypes.c_void_p()
    _lib.check(L.pyr_group_create(ctypes.byref(h), len(ctxs), (ctypes.c_void_p * len(ctxs))(*[c._h.value for c in ctxs]),
                                  (ctypes.c_longlong * len(ctxs))(*offs)))
    _lib.check(L.pyr_group_set_stream(h, _lib.stream_of(torch.device("cuda", torch.cuda.current_device()))))
    g = torch.Generator(device="cuda").manual_seed(9)
    src, old = [torch.randn(at, generator=g, device="cuda", dtype=dtype) for _ in range(2)]
    prec = _lib.F64 if dtype == torch.float64 else _lib.R32
    for op in range(5):
        for d in range(3):
            for epi in (_lib.EPI_STORE, _lib.EPI_ADD, _lib.EPI_ABS_SCALED, _lib.EPI_MAXABS_SCALED):
                got, want = old.clone(), old.clone()
                _lib.check(L.pyr_group_apply(h, op, d, prec, src.data_ptr(), got.data_ptr(), epi, 0.75, 2))
                for c, n, o in zip(ctxs, sizes, offs):
                    v, w = [t[o:o + n[0] * n[1] * n[2]].view(n[2], n[1], n[0]).permute(2, 1, 0) for t in (src, want)]
                    c.apply(op, d, v, out=w, epi=epi, epi_scale=0.75 * c.dmesh[d] ** 2)
                assert torch.equal(got, want), (op, d, epi)
    _lib.check(L.pyr_group_destroy(h))
    for c in ctxs:
        c.close()
