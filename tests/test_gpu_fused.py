"""Launches that stand for several stages of a plan (one-launch Bluestein, one-launch ISTFT): each
against the FP64 oracle (rel-L2 5e-6 for Bluestein lengths, 2e-6 otherwise) and against the stages run
one by one (SIP_FFT_FUSE=0 at plan time). Both ways round a result a few times per pass of log2 M
levels, each within 4e-7 of the exact one, so they agree to 1e-6.
"""
import numpy as np
import pytest

import oracle
import sip_amd as S
from fftcase import FWD, INV, c2c, make, report, sign_of

pytestmark = pytest.mark.gpu
AGREE = 1e-6


def _run(make, execute, fuse, monkeypatch):
    monkeypatch.setenv("SIP_FFT_FUSE", "1" if fuse else "0")
    h = S.FftHandle()
    try:
        make(h)
        h.alloc_workspace()
        h.use_current_torch_stream()
        fused = h.describe()["fused"]
        assert len(fused) == (1 if fuse else 0), fused
        out = execute(h)
        assert h.synchronize() == S.ACL_SUCCESS
        return out
    finally:
        h.destroy()


def _both(make, execute, monkeypatch):
    return [_run(make, execute, f, monkeypatch) for f in (True, False)]


def _agree(name, got, staged, want, tol):
    rel, _ = report(name, got, want)
    assert rel <= tol
    scale = np.linalg.norm(want)
    assert np.linalg.norm(got.astype(np.complex128) - staged) <= AGREE * scale


def _prime_at_most(n):
    while n > 17 and any(n % p == 0 for p in range(2, int(n ** 0.5) + 1)):
        n -= 1
    return n


# the largest prime of every convolution length, and the first of the next (padding near nothing / most)
EDGES = sorted({_prime_at_most((m + 1) // 2) for m in (
    48, 64, 80, 96, 128, 160, 192, 256, 320, 384, 512, 640, 768, 1024, 1280, 1536, 2048, 2560, 3072, 4096, 5120, 6144,
    8192, 10240, 12288, 16384, 20480, 24576, 32768)} | {17, 521, 2053, 4099, 12289})


@pytest.mark.parametrize("n", EDGES)
def test_bluestein_rows(torch_cuda, monkeypatch, n):
    import torch
    b = max(1, min(37, (1 << 17) // n))
    d = INV if n % 4 == 1 else FWD
    x = oracle.uniform_complex((b, n), 0x5EED0B00 + n)
    xd = torch.from_numpy(x).cuda()
    y = torch.empty_like(xd)

    def execute(h):
        assert h.exec_c2c(xd, y) == S.ACL_SUCCESS
        torch.cuda.synchronize()
        return y.cpu().numpy()

    got, staged = _both(lambda h: h.make_plan_1d(n, S.ASCEND_FFT_C2C, d, b), execute, monkeypatch)
    _agree(f"bluestein {n} x {b}", got, staged, oracle.c2c(x, sign_of(d)), 5e-6)


@pytest.mark.parametrize("n,b", [(17, 5), (127, 33), (1009, 40), (2039, 3), (6007, 2), (16381, 2)])
def test_bluestein_vertical(torch_cuda, monkeypatch, n, b):
    """Columns of an (n, b) array: tiles of adjacent transforms, partly empty, down to one wide."""
    import torch
    x = oracle.uniform_complex((n, b), 0x5EED0C00 + n)
    xd = torch.from_numpy(x).cuda()
    y = torch.empty_like(xd)

    def execute(h):
        assert h.exec_c2c(xd, y) == S.ACL_SUCCESS
        torch.cuda.synchronize()
        return y.cpu().numpy()

    got, staged = _both(lambda h: h.make_plan_1d(n, S.ASCEND_FFT_C2C, FWD, b, S.ASCEND_FFT_VERTICAL), execute,
                        monkeypatch)
    want = oracle.c2c(np.ascontiguousarray(x.T), sign_of(FWD)).T
    _agree(f"bluestein vertical {n} x {b}", got, staged, want, 5e-6)


@pytest.mark.parametrize("n,b", [(19, 70), (509, 9), (2003, 3)])
def test_bluestein_split_planes(torch_cuda, monkeypatch, n, b):
    import torch
    x = oracle.uniform_complex((b, n), 0x5EED0D00 + n)
    xs = [torch.from_numpy(np.ascontiguousarray(v)).cuda() for v in (x.real, x.imag)]
    ys = [torch.empty_like(v) for v in xs]

    def execute(h):
        assert h.exec_c2c_separated(*xs, *ys) == S.ACL_SUCCESS
        torch.cuda.synchronize()
        return ys[0].cpu().numpy() + 1j * ys[1].cpu().numpy().astype(np.float64)

    got, staged = _both(lambda h: h.make_plan_1d(n, S.ASCEND_FFT_C2C_SEP, INV, b), execute, monkeypatch)
    _agree(f"bluestein split {n} x {b}", got, staged, oracle.c2c(x, sign_of(INV)), 5e-6)


# one frame more than a tile holds, fewer frames than the halo, hops that divide the frame and that do
# not, no overlap at all, odd lengths, the shortest hop that is still one launch (n / 8 with 16 frames), tiles
# of few frames
@pytest.mark.parametrize("ch,n,hop,frames", [(1, 24, 6, 65), (2, 27, 10, 40), (3, 256, 64, 2), (2, 256, 256, 70),
                                             (2, 400, 160, 131), (1, 625, 125, 9), (2, 1024, 256, 17),
                                             (1, 1024, 128, 33), (2, 1080, 270, 20), (1, 1458, 365, 12),
                                             (1, 1440, 720, 164), (1, 1440, 360, 165), (4, 640, 320, 103),
                                             (16, 1200, 600, 90), (1, 960, 960, 31)])
def test_istft_one_launch(torch_cuda, monkeypatch, ch, n, hop, frames):
    import torch
    rng = np.random.default_rng(n * 7 + hop)
    x = (rng.standard_normal((ch, n, frames)) + 1j * rng.standard_normal((ch, n, frames))).astype(np.complex64)
    w = (np.hanning(n + 2)[1:-1] + 0.05).astype(np.float32)
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    y = torch.empty((ch, oracle.istft_out_len(n, hop, frames)), dtype=torch.complex64, device="cuda")

    def execute(h):
        assert h.exec_istft(xd, wd, y) == S.ACL_SUCCESS
        torch.cuda.synchronize()
        return y.cpu().numpy()

    got, staged = _both(lambda h: h.istft_make_plan(xd, n, hop, n), execute, monkeypatch)
    _agree(f"istft ch={ch} n={n} hop={hop} frames={frames}", got, staged, oracle.istft(x, n, hop, w), 2e-6)


@pytest.mark.parametrize("n", [40, 45, 60, 160, 180, 192, 240, 320, 400, 640, 800])
def test_istft_lengths_off_the_register_limit(torch_cuda, monkeypatch, n):
    test_istft_one_launch(torch_cuda, monkeypatch, 2, n, n // 4, 90)


@pytest.mark.parametrize("ch,n,hop,frames,fused", [(1, 24, 24, 64, 0), (1, 400, 400, 64, 0), (4, 640, 640, 200, 0),
                                                   (2, 160, 160, 2049, 1), (4, 80, 40, 200, 0), (4, 128, 64, 200, 1),
                                                   (1, 1000, 125, 2, 0), (1, 1000, 125, 9, 1), (8, 1024, 256, 40, 1)])
def test_istft_route(torch_cuda, monkeypatch, ch, n, hop, frames, fused):
    """Where the stages are faster the plan keeps them."""
    import torch
    monkeypatch.delenv("SIP_FFT_FUSE", raising=False)
    h = S.FftHandle()
    x = torch.empty(ch, n, frames, dtype=torch.complex64, device="cuda")
    assert h.istft_make_plan(x, n, hop, n) == S.ACL_SUCCESS
    assert len(h.describe()["fused"]) == fused
    h.destroy()


@pytest.mark.parametrize("mode", [S.PREC_F16_SPLIT, S.PREC_BF16_SPLIT3])
@pytest.mark.parametrize("a, b, batch", [(2048, 525, 4), (1536, 1050, 2)])
def test_precision_long_columns(torch_cuda, monkeypatch, a, b, batch, mode):
    """An axis whose four-step stages are FP32 in the precision form too runs as one FP32 column pass there
    (counts that leave the last tile partly empty); both agree with the oracle as FP32 does."""
    x = oracle.uniform_complex((batch, a, b), 0x5EED1500 + a)
    want = oracle.c2c_nd(x, 2, sign_of(INV))
    for fuse in ("1", "0"):
        monkeypatch.setenv("SIP_FFT_FUSE", fuse)
        h = make([a, b], S.ASCEND_FFT_C2C, INV, batch, precision=mode)
        assert len(h.describe()["fused"]) == int(fuse)
        h.destroy()
        rel, _ = report(f"{a} x {b} fuse={fuse}", c2c(x, [a, b], INV, precision=mode), want)
        assert rel <= 2e-6
