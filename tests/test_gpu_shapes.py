"""Kernels whose threads and radices were chosen per role and length (column_shapes.py): every listed length
against the FP64 oracle (rel-L2 2e-6), on counts that leave the last tile partly empty and, for columns,
strides that do not fall on whole 128-byte lines."""
import importlib.util
import os

import numpy as np
import pytest

import oracle
import sip_amd as S
from fftcase import FWD, INV, c2c, c2r, make, r2c, report, sign_of

pytestmark = pytest.mark.gpu
TOL = 2e-6


def _shapes(module):
    path = os.path.join(S.HERE, "csrc", "kernels", module + ".py")
    spec = importlib.util.spec_from_file_location(module, path)
    mod = importlib.util.module_from_spec(spec)
    spec.loader.exec_module(mod)
    return mod


COLS = _shapes("column_shapes")


def _vertical(n, b, direction):
    x = oracle.uniform_complex((n, b), 0x5EED0E00 + n)
    y = c2c(x.reshape(n, b), [n], direction, S.ASCEND_FFT_VERTICAL)
    want = oracle.c2c(np.ascontiguousarray(x.T), sign_of(direction)).T
    rel, _ = report(f"columns {n} x {b}", y, want)
    assert rel <= TOL


@pytest.mark.parametrize("n", sorted(COLS.COLUMN_SHAPES) + [20, 24, 45])
def test_column_shapes(torch_cuda, n):
    _vertical(n, 37, INV if n % 3 else FWD)


@pytest.mark.parametrize("n", sorted(COLS.LONG_COLUMN_SHAPES))
def test_long_column_shapes(torch_cuda, n):
    """One pass from 128 tiles up (an odd count: 2051 columns), two below; both checked."""
    h = make([n], S.ASCEND_FFT_C2C, FWD, 2051, S.ASCEND_FFT_VERTICAL)
    assert h.describe()["fused"][0]["note"] == f"columns {n}"
    h.destroy()
    _vertical(n, 2051, FWD if n % 2 else INV)
    _vertical(n, 19, INV)


@pytest.mark.parametrize("n", sorted(COLS.COLUMN_TW_SHAPES))
def test_column_shapes_with_twiddle(torch_cuda, monkeypatch, n):
    """First four-step stage of length n (forced factor), second stage the shortest smooth leaf that makes the
    length one that no single launch takes."""
    m = next(v for v in S.smooth_lengths(33, 1024) if v * n > 32768)
    monkeypatch.setenv("SIP_FFT_SPLIT_L1", str(n))
    d = INV if n % 3 else FWD
    x = oracle.uniform_complex((3, n * m), 0x5EED0F00 + n)
    h = make([n * m], S.ASCEND_FFT_C2C, d, 3)
    st = h.describe()["stages"][0]
    assert st["L"] == n and st["tw4"] == n * m and st["T"] == COLS.COLUMN_TW_SHAPES[n][0]
    h.destroy()
    y = c2c(x, [n * m], d)
    rel, _ = report(f"four-step {n} x {m}", y, oracle.c2c(x, sign_of(d)))
    assert rel <= TOL


def test_streaming_input_of_several_launches(torch_cuda):
    """A plan of several launches that touches more than 128 MiB loads its input nontemporally."""
    h = make([1 << 20], S.ASCEND_FFT_C2C, FWD, 8)
    assert [s["nt_in"] for s in h.describe()["stages"]] == [1, 0]
    h.destroy()
    h = make([1 << 20], S.ASCEND_FFT_C2C, FWD, 5)
    assert [s["nt_in"] for s in h.describe()["stages"]] == [0, 0]
    h.destroy()


ROWS = _shapes("row_shapes")


@pytest.mark.parametrize("n", sorted(ROWS.ROW_SHAPES) + [25, 27, 35, 64, 66, 104, 117, 128, 16200])
def test_row_shapes(torch_cuda, n):
    b = max(3, min(75, (1 << 19) // n))
    d = INV if n % 3 else FWD
    h = make([n], S.ASCEND_FFT_C2C, d, b)
    st = h.describe()["stages"][0]
    h.destroy()
    assert st["split_lds"] == st["direct_in"] == st["direct_out"] == 1
    if n in ROWS.ROW_SHAPES:
        assert st["T"] == ROWS.ROW_SHAPES[n][0] and st["radices"] == ROWS.ROW_SHAPES[n][1]
    x = oracle.uniform_complex((b, n), 0x5EED1000 + n)
    rel, _ = report(f"rows {n} x {b}", c2c(x, [n], d), oracle.c2c(x, sign_of(d)))
    assert rel <= TOL


@pytest.mark.parametrize("n", [2, 3, 7, 8, 11, 13, 16, 20, 22, 24, 25, 26, 30, 33, 39, 40, 45, 48, 50, 52, 54, 56, 64, 65, 66, 81,
                               100, 104, 200,
                               243, 300, 1000, 1200, 3600, 4096, 15000, 15625, 16384])
@pytest.mark.parametrize("direction", [FWD, INV])
def test_split_plane_rows(torch_cuda, n, direction):
    """Rows in two planes on both sides of the line-order limit (48), one to several tiles with the last one
    partly empty, out of place and in place."""
    import torch
    for b in sorted({1, max(2, min(131, (1 << 18) // n))}):
        x = oracle.uniform_complex((b, n), 0x5EED1100 + n + b)
        xs = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x.real, x.imag)]
        ys = [torch.empty_like(v) for v in xs]
        h = S.FftHandle()
        assert h.make_plan_1d(n, S.ASCEND_FFT_C2C_SEP, direction, b) == S.ACL_SUCCESS
        h.use_current_torch_stream()
        assert h.workspace_size() == 0
        assert h.exec_c2c_separated(*xs, *ys) == S.ACL_SUCCESS
        assert h.exec_c2c_separated(*xs, *xs) == S.ACL_SUCCESS
        assert h.synchronize() == S.ACL_SUCCESS
        h.destroy()
        got = ys[0].cpu().numpy() + 1j * ys[1].cpu().numpy().astype(np.float64)
        rel, _ = report(f"planes {n} x {b}", got, oracle.c2c(x, sign_of(direction)))
        assert rel <= TOL
        assert torch.equal(xs[0], ys[0]) and torch.equal(xs[1], ys[1])


REAL = _shapes("real_shapes")


def _real(n, b):
    x = oracle.uniform(n * b, 0x5EED1200 + n).reshape(b, n)
    rel, _ = report(f"r2c {n} x {b}", r2c(x, [n]), oracle.r2c(x))
    assert rel <= TOL
    X = oracle.uniform_complex((b, n // 2 + 1), 0x5EED1300 + n)  # imaginary parts of the end bins are dropped
    rel, _ = report(f"c2r {n} x {b}", c2r(X, [n]), oracle.c2r(X, n))
    assert rel <= TOL


@pytest.mark.parametrize("L", sorted(REAL.REAL_SHAPES) + [32, 35, 64, 104, 128, 256])
def test_real_shapes(torch_cuda, L):
    b = max(3, min(75, (1 << 18) // L))
    h = make([2 * L], S.ASCEND_FFT_R2C, FWD, b)
    st = h.describe()["stages"][0]
    h.destroy()
    assert st["split_lds"] == 1 and (L not in REAL.REAL_SHAPES or st["T"] == REAL.REAL_SHAPES[L][0])
    _real(2 * L, b)


@pytest.mark.parametrize("n", [9, 15, 25, 27, 35, 45, 63, 75, 81, 99, 117, 225, 243, 375, 625, 585, 1215, 2025, 3125, 3375,
                               3645, 6561, 9375, 10125, 15625])
def test_real_odd_lengths(torch_cuda, n):
    """Odd lengths, both directions of both transforms."""
    b = max(3, min(75, (1 << 18) // n))
    _real(n, b)
    x = oracle.uniform(n * b, 77 + n).reshape(b, n)
    rel, _ = report(f"r2c {n} inverse", r2c(x, [n], INV), oracle.r2c(x, oracle.INVERSE))
    assert rel <= TOL
    X = oracle.uniform_complex((b, n // 2 + 1), 78 + n)
    rel, _ = report(f"c2r {n} forward", c2r(X, [n], FWD), oracle.c2r(X, n, oracle.FORWARD))
    assert rel <= TOL


@pytest.mark.parametrize("n", sorted(REAL.ROWS_COLS_SHAPES))
def test_rows_cols_shapes(torch_cuda, monkeypatch, n):
    """Second four-step stage of length n (the first factor forced)."""
    m = next(v for v in S.smooth_lengths(33, 1024) if v * n > 32768)
    monkeypatch.setenv("SIP_FFT_SPLIT_L1", str(m))
    d = INV if n % 3 else FWD
    h = make([n * m], S.ASCEND_FFT_C2C, d, 3)
    st = h.describe()["stages"][1]
    h.destroy()
    assert st["L"] == n and st["rc"] == 1 and st["T"] == REAL.ROWS_COLS_SHAPES[n][0]
    x = oracle.uniform_complex((3, n * m), 0x5EED1400 + n)
    rel, _ = report(f"four-step {m} x {n}", c2c(x, [n * m], d), oracle.c2c(x, sign_of(d)))
    assert rel <= TOL


@pytest.mark.parametrize("n, factors", [(243000, [675, 360]), (327680, [640, 512]), (777600, [960, 810]),
                                        (65536, [256, 256])])
def test_four_step_splits_by_measured_rates(torch_cuda, n, factors):
    """Splits that the stage rates choose (split_rates.py) and one that they leave alone."""
    for d in (FWD, INV):
        h = make([n], S.ASCEND_FFT_C2C, d, 2)
        assert [s["L"] for s in h.describe()["stages"]] == factors
        h.destroy()
        x = oracle.uniform_complex((2, n), 0x5EED1100 + n)
        rel, _ = report(f"split {n}", c2c(x, [n], d), oracle.c2c(x, sign_of(d)))
        assert rel <= TOL
