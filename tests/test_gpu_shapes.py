"""Kernels whose threads and radices were chosen per role and length (column_shapes.py, row_shapes.py,
real_shapes.py): every listed length against the FP64 oracle (rel-L2 2e-6), on counts that leave the last
tile partly empty and, for columns, strides that do not fall on whole 128-byte lines. Columns and split
stages run at two counts: few transforms (8-wide tiles, or the two-plane leaf where a shape needs many) and
many (16-wide tiles, the listed shape)."""
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


def _many(start):
    """Columns that make more than 128 tiles of 16, and `start` of them, with a partly empty last one."""
    return 16 * max(128, start) + 3


def _check_role(st, n, shapes, start, few):
    """The stage runs the listed shape (or the leaf where few transforms keep it) on the expected tile width."""
    shape = shapes.get(n)
    leaf = few and start > 0
    assert st["L"] == n and st["split_lds"] == (0 if leaf else 1)
    if shape and not leaf:
        assert st["T"] == shape[0] and st["radices"] == shape[1]
    if st["T"] >= 8:
        assert st["F"] == 8 if few else (st["F"] % 16 == 0 or st["T"] > 64)


@pytest.mark.parametrize("n", sorted(COLS.COLUMN_SHAPES) + [20, 24, 45, 400, 512, 1024])
def test_column_shapes(torch_cuda, n):
    start = COLS.COLUMN_FROM.get(n, 0)
    for b, few in ((37, True), (_many(start), False)):
        h = make([n], S.ASCEND_FFT_C2C, FWD, b, S.ASCEND_FFT_VERTICAL)
        _check_role(h.describe()["stages"][0], n, COLS.COLUMN_SHAPES, start, few)
        h.destroy()
        _vertical(n, b, INV if n % 3 else FWD)


@pytest.mark.parametrize("n", sorted(COLS.LONG_COLUMN_SHAPES))
def test_long_column_shapes(torch_cuda, n):
    """One pass from 128 tiles up, for some lengths later (an odd count, the last tile partly empty), two
    below; both checked."""
    width = COLS.LONG_COLUMN_SHAPES[n][3]
    b = max(2051, width * COLS.LONG_COLUMN_FROM.get(n, 128) + 3)
    h = make([n], S.ASCEND_FFT_C2C, FWD, b, S.ASCEND_FFT_VERTICAL)
    f = h.describe()["fused"][0]
    assert f["note"] == f"columns {n}" and f["F"] == width
    h.destroy()
    _vertical(n, b, FWD if n % 2 else INV)
    _vertical(n, 19, INV)


def _split(n, first):
    """The other factor: the shortest smooth leaf that makes a length which no single launch takes."""
    m = next(v for v in S.smooth_lengths(33, 1024) if v * n > 32768)
    return (n, m) if first else (m, n)


@pytest.mark.parametrize("n", sorted(COLS.COLUMN_TW_SHAPES))
def test_column_shapes_with_twiddle(torch_cuda, monkeypatch, n):
    """First four-step stage of length n (forced factor)."""
    _, m = _split(n, True)
    monkeypatch.setenv("SIP_FFT_SPLIT_L1", str(n))
    d = INV if n % 3 else FWD
    start = COLS.COLUMN_TW_FROM.get(n, 0)
    for b, few in ((3, True), (_many(start) // m + 1, False)):
        x = oracle.uniform_complex((b, n * m), 0x5EED0F00 + n)
        h = make([n * m], S.ASCEND_FFT_C2C, d, b)
        st = h.describe()["stages"][0]
        h.destroy()
        assert st["tw4"] == n * m
        _check_role(st, n, COLS.COLUMN_TW_SHAPES, start, few and b * m <= 2048)
        y = c2c(x, [n * m], d)
        rel, _ = report(f"four-step {n} x {m} x {b}", y, oracle.c2c(x, sign_of(d)))
        assert rel <= TOL


def test_streaming_input_of_several_launches(torch_cuda):
    """A first stage of long whole-line columns in a plan that touches more than 128 MiB loads its input nontemporally."""
    h = make([1 << 20], S.ASCEND_FFT_C2C, FWD, 8)
    assert [s["nt_in"] for s in h.describe()["stages"]] == [1, 0]
    h.destroy()
    h = make([1 << 20], S.ASCEND_FFT_C2C, FWD, 5)
    assert [s["nt_in"] for s in h.describe()["stages"]] == [0, 0]
    h.destroy()


ROWS = _shapes("row_shapes")


@pytest.mark.parametrize("n", sorted(ROWS.ROW_SHAPES) + [25, 27, 35, 64, 66, 104, 117, 128, 16200])
def test_row_shapes(torch_cuda, n):
    b = ROWS.ROW_FROM.get(n, max(3, min(75, (1 << 19) // n)))
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


@pytest.mark.parametrize("n", sorted(_shapes("gen_instances").ROWS_POINTS))
def test_short_rows_of_many(torch_cuda, n):
    """On both sides of the count from which short rows go through LDS in line order."""
    points = _shapes("gen_instances").ROWS_POINTS[n]
    for b in (points // n, points // n + 1):
        x = oracle.uniform_complex((b, n), 0x5EED1600 + n)
        rel, _ = report(f"rows {n} x {b}", c2c(x, [n], INV if n % 2 else FWD), oracle.c2c(x, sign_of(INV if n % 2 else FWD)))
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


@pytest.mark.parametrize("L", sorted(REAL.REAL_SHAPES) + [32, 35, 64, 104, 128, 256, 162, 375])
def test_real_shapes(torch_cuda, L):
    """162 and 375: leaves of 16 to 31 threads, on one plane from 48 MiB."""
    b = (6 << 20) // L + 1 if L in (162, 375) else max(3, min(75, (1 << 18) // L))
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
    m, _ = _split(n, False)
    monkeypatch.setenv("SIP_FFT_SPLIT_L1", str(m))
    d = INV if n % 3 else FWD
    start = REAL.ROWS_COLS_FROM.get(n, 0)
    for b, few in ((3, True), (_many(start) // m + 1, False)):
        h = make([n * m], S.ASCEND_FFT_C2C, d, b)
        st = h.describe()["stages"][1]
        h.destroy()
        assert st["L"] == n and st["rc"] == (0 if few and start else 1)
        if not (few and start):
            assert st["T"] == REAL.ROWS_COLS_SHAPES[n][0]
        x = oracle.uniform_complex((b, n * m), 0x5EED1400 + n)
        rel, _ = report(f"four-step {m} x {n} x {b}", c2c(x, [n * m], d), oracle.c2c(x, sign_of(d)))
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
