"""Line operators on values near the ends of the number formats."""
import ctypes

import numpy as np
import pytest
import torch

BOUNDED = [("NONE", "NONE"), ("SYMM", "SYMM"), ("NONE", "SYMM")]
# whole and ragged chunks of up to 16 and 32 rows, one of them and several
LENGTHS = [8, 9, 16, 31, 32, 33, 37, 48, 64, 65, 100, 257]


class Host:
    """The kernels' arithmetic along direction d on host arrays."""

    def __init__(self, nn, d, faces):
        from pyranda_amd import _lib as amd
        self.amd, self.L, self.d = amd, amd.lib(), d
        self.h = ctypes.c_void_p()
        kinds = ["PERI"] * 6
        kinds[2 * d:2 * d + 2] = faces
        bc6 = (ctypes.c_int * 6)(*[amd.BC[k] for k in kinds])
        amd.check(self.L.pyr_setup_host(ctypes.byref(self.h), *nn, 0.0, 1.0, 0.0, 1.0, 0.0, 1.0, bc6))

    def __call__(self, op, v):
        out = np.full(v.shape, 7.0, dtype=v.dtype, order="F")
        prec = self.amd.F64 if v.dtype == np.float64 else self.amd.R32
        self.amd.check(self.L.pyr_host_emulate(self.h, op, self.d, prec, v.ctypes.data, out.ctypes.data))
        return out

    def close(self):
        self.L.pyr_destroy(self.h)


class Device:
    """The same through the kernels."""

    def __init__(self, nn, d, faces):
        from pyranda_amd.parcop import ParcopContext
        kinds = ["PERI"] * 6
        kinds[2 * d:2 * d + 2] = faces
        self.d, self.ctx = d, ParcopContext(nn, (0.0,) * 3, (1.0,) * 3, kinds)

    def __call__(self, op, v):
        vd = torch.from_numpy(np.ascontiguousarray(v.transpose(2, 1, 0))).cuda().permute(2, 1, 0)
        return self.ctx.apply(op, self.d, vd).cpu().numpy()

    def close(self):
        self.ctx.close()


def _dims(n, d):
    nn = [2, 3, 2]
    nn[d] = n
    return tuple(nn)


def _each(run, lengths, faces):
    for n in lengths:
        for d in range(3):
            f = run(_dims(n, d), d, faces)
            yield n, d, f
            f.close()


def _constants_of_any_size(run, faces):
    # rows are sums of differences of the field's values: a derivative of a
    # constant is 0 and a filter returns the constant, whatever its size
    for n, d, f in _each(run, LENGTHS, faces):
        for c in (1.0, 1e36, 3.4e38):
            v = np.full(_dims(n, d), c, dtype=np.float32, order="F")
            for op in range(5):
                want = v if op > 2 else np.zeros_like(v)
                assert np.array_equal(f(op, v), want), (n, d, op, c)


@pytest.mark.parametrize("faces", BOUNDED)
def test_emulated_constants_of_any_size(faces):
    _constants_of_any_size(Host, faces)


@pytest.mark.gpu
@pytest.mark.parametrize("faces", BOUNDED)
def test_device_constants_of_any_size(faces):
    print("constants", faces, flush=True)
    _constants_of_any_size(Device, faces)


def _explicit_filter_of_infinities(run, faces, oracle_mod):
    # a row next to an infinity is that infinity, the infinity's own row is NaN
    # and no other row is touched, rows at the ends and their antisymmetric
    # variants included; finite values to a few roundings of the largest one
    rng = np.random.default_rng(5)
    with np.errstate(invalid="ignore"):
        for n, d, f in _each(run, LENGTHS, faces):
            nn = _dims(n, d)
            P = oracle_mod.Oracle(nn, (1.0,) * 3, [faces[0] == "PERI" if e == d else True for e in range(3)],
                                  symmetric=[[e == d and k == "SYMM" for k in faces] for e in range(3)])
            v0 = rng.standard_normal(nn)
            for dtype in (np.float64, np.float32):
                for row in sorted({0, 1, 3, 4, n // 2, n - 5, n - 4, n - 1}):
                    for bad in (np.inf, -np.inf):
                        v = np.asfortranarray(v0.astype(dtype))
                        idx = [1, 1, 1]
                        idx[d] = row
                        v[tuple(idx)] = bad
                        w = np.asfortranarray(v.astype(np.float64))
                        for anti in ((0, 1) if "SYMM" in faces else (0,)):
                            want = P.apply_sym(4, d, -1, w) if anti else P.apply(4, d, w)
                            got = f(4 | (0x10 if anti else 0), v)
                            where = (n, d, dtype, row, bad, anti)
                            for kind in (np.isnan, np.isposinf, np.isneginf):
                                assert np.array_equal(kind(got), kind(want)), where
                            ok = np.isfinite(want)
                            assert np.abs(got[ok] - want[ok]).max() <= 8 * np.finfo(dtype).eps * np.abs(w[np.isfinite(w)]).max(), where


@pytest.mark.parametrize("faces", BOUNDED + [("PERI", "PERI")])
def test_emulated_explicit_filter_of_infinities(oracle_mod, faces):
    _explicit_filter_of_infinities(Host, faces, oracle_mod)


@pytest.mark.gpu
@pytest.mark.parametrize("faces", BOUNDED + [("PERI", "PERI")])
def test_device_explicit_filter_of_infinities(oracle_mod, faces):
    print("explicit filter of infinities", faces, flush=True)
    _explicit_filter_of_infinities(Device, faces, oracle_mod)


# bounds on the right-hand side's partial sums, in units of the largest value
RHS_GAIN = (16.0, 57400.0, 11200.0, 4.0, 4.0)


def _fields_near_overflow(run, faces):
    # a field times a power of two gives the result times that power, up to
    # where the result or a row's right-hand side leaves the FP64 range
    rng = np.random.default_rng(6)
    for n, d, f in _each(run, LENGTHS, faces):
        v = np.asfortranarray(rng.uniform(-1.0, 1.0, _dims(n, d)))
        for op in range(5):
            for anti in ((0, 0x10) if "SYMM" in faces else (0,)):
                out = f(op | anti, v)
                top = max(np.abs(out).max(), RHS_GAIN[op])
                s = 2.0 ** np.floor(np.log2(np.finfo(float).max / top) - 2.0)
                assert np.array_equal(f(op | anti, np.asfortranarray(v * s)), out * s), (n, d, op, anti)


@pytest.mark.parametrize("faces", BOUNDED)
def test_emulated_fields_near_overflow(faces):
    _fields_near_overflow(Host, faces)


@pytest.mark.gpu
@pytest.mark.parametrize("faces", BOUNDED)
def test_device_fields_near_overflow(faces):
    print("fields near overflow", faces, flush=True)
    _fields_near_overflow(Device, faces)


@pytest.mark.parametrize("faces", BOUNDED + [("PERI", "PERI")])
def test_emulated_nonfinite_values_spread_over_their_line(faces):
    # as in the kernels (test_line_solve_edges.py)
    rng = np.random.default_rng(7)
    with np.errstate(invalid="ignore"):
        for n, d, f in _each(Host, [9, 65, 257, 1000], faces):
            for dtype in (np.float64, np.float32):
                for row, bad in ((0, np.nan), (n - 1, -np.inf), (n // 2, np.inf)):
                    v = np.asfortranarray(rng.standard_normal(_dims(n, d)).astype(dtype))
                    line = [1, 1, 1]
                    line[d] = slice(None)
                    clean = [f(op, v) for op in range(4)]
                    line[d] = row
                    v[tuple(line)] = bad
                    line[d] = slice(None)
                    for op in range(4):
                        got = f(op, v)
                        assert not np.isfinite(got[tuple(line)]).any(), (n, d, op, dtype, row)
                        got[tuple(line)] = clean[op][tuple(line)]
                        assert np.array_equal(got, clean[op]), (n, d, op, dtype, row)
