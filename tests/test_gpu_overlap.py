"""Input and output in one allocation. A launch that stands for several stages stores outputs while other
workgroups still read inputs, so where the caller's buffers overlap the input is copied into the workspace
first; a C2C transform of an array into itself needs no copy. Against the FP64 oracle at the plain parity
tolerances (rel-L2 2e-6, Bluestein lengths 5e-6)."""
import numpy as np
import pytest

import oracle
import sip_amd as S
from fftcase import FWD, INV, make, report, sign_of

pytestmark = pytest.mark.gpu


def _views(torch, x, shift):
    """x and an output of its size, `shift` elements apart in one allocation (either may come first)."""
    n, a = x.size, abs(shift)
    pool = torch.zeros(n + a, dtype=torch.complex64, device="cuda")
    src, dst = (pool[a:], pool[:n]) if shift < 0 else (pool[:n], pool[a:a + n])
    src.copy_(torch.from_numpy(x.reshape(-1)))
    return src.view(x.shape), dst.view(x.shape)


CASES = [([1009], 40, S.ASCEND_FFT_HORIZONTAL, 5e-6), ([1009], 40, S.ASCEND_FFT_VERTICAL, 5e-6),
         ([17], 3000, S.ASCEND_FFT_HORIZONTAL, 5e-6), ([33, 509], 3, S.ASCEND_FFT_HORIZONTAL, 5e-6),
         ([1080], 2051, S.ASCEND_FFT_VERTICAL, 2e-6)]


@pytest.mark.parametrize("dims,b,dim,tol", CASES)
@pytest.mark.parametrize("shift", [0, 1, -1, 1000, -777])
def test_c2c(torch_cuda, monkeypatch, dims, b, dim, tol, shift):
    torch = torch_cuda
    monkeypatch.delenv("SIP_FFT_FUSE", raising=False)
    vertical = dim == S.ASCEND_FFT_VERTICAL
    shape = (dims[0], b) if vertical else (b, *dims)
    x = oracle.uniform_complex(shape, 0x5EED1700 + dims[0])
    h = make(dims, S.ASCEND_FFT_C2C, INV, b, dim)
    assert len(h.describe()["fused"]) >= 1
    src, dst = _views(torch, x, shift)
    assert h.exec_c2c(src, dst) == S.ACL_SUCCESS and h.synchronize() == S.ACL_SUCCESS
    h.destroy()
    if vertical:
        want = oracle.c2c(np.ascontiguousarray(x.T), sign_of(INV)).T
    else:
        want = oracle.c2c_nd(x, len(dims), sign_of(INV))
    rel, _ = report(f"{dims} x {b} shift {shift}", dst.cpu().numpy(), want)
    assert rel <= tol


@pytest.mark.parametrize("swap", [False, True])
@pytest.mark.parametrize("shift", [0, 5])
def test_split_planes(torch_cuda, swap, shift):
    """Planes transformed into themselves, into each other, and into planes that begin a few values later."""
    torch = torch_cuda
    n, b = 509, 60
    x = oracle.uniform_complex((b, n), 0x5EED1800)
    pools = [torch.zeros(b * n + 5, device="cuda") for _ in range(2)]
    src = [p[:b * n].view(b, n) for p in pools]
    for s, v in zip(src, (x.real, x.imag)):
        s.copy_(torch.from_numpy(np.ascontiguousarray(v)))
    dst = [p[shift:shift + b * n].view(b, n) for p in (pools[::-1] if swap else pools)]
    h = make([n], S.ASCEND_FFT_C2C_SEP, FWD, b)
    assert len(h.describe()["fused"]) == 1
    assert h.exec_c2c_separated(*src, *dst) == S.ACL_SUCCESS and h.synchronize() == S.ACL_SUCCESS
    h.destroy()
    got = dst[0].cpu().numpy() + 1j * dst[1].cpu().numpy().astype(np.float64)
    rel, _ = report(f"planes swap={swap} shift={shift}", got, oracle.c2c(x, sign_of(FWD)))
    assert rel <= 5e-6


@pytest.mark.parametrize("ch,n,hop,frames,at", [(4, 256, 64, 300, 0), (4, 256, 64, 300, 12345), (2, 1024, 256, 90, 0),
                                                (2, 1200, 300, 90, 1)])
def test_istft(torch_cuda, monkeypatch, ch, n, hop, frames, at):
    """Samples over the spectra that they come from."""
    torch = torch_cuda
    monkeypatch.delenv("SIP_FFT_FUSE", raising=False)
    rng = np.random.default_rng(n + at)
    x = (rng.standard_normal((ch, n, frames)) + 1j * rng.standard_normal((ch, n, frames))).astype(np.complex64)
    w = (np.hanning(n + 2)[1:-1] + 0.05).astype(np.float32)
    xd, wd = torch.from_numpy(x).cuda(), torch.from_numpy(w).cuda()
    out = oracle.istft_out_len(n, hop, frames)
    y = xd.view(-1)[at:at + ch * out].view(ch, out)
    h = S.FftHandle()
    assert h.istft_make_plan(xd, n, hop, n) == S.ACL_SUCCESS
    assert len(h.describe()["fused"]) == 1
    h.alloc_workspace()
    h.use_current_torch_stream()
    assert h.exec_istft(xd, wd, y) == S.ACL_SUCCESS and h.synchronize() == S.ACL_SUCCESS
    h.destroy()
    rel, _ = report(f"istft {ch} x {n} over its input", y.cpu().numpy(), oracle.istft(x, n, hop, w))
    assert rel <= 2e-6


@pytest.mark.parametrize("graph", [0, S.BATCH_GRAPH])
def test_batch_problems_that_swap_buffers(torch_cuda, graph):
    """Two problems of one Bluestein length, each into the other's input."""
    torch = torch_cuda
    n, rows = 1009, (30, 30)
    hs = [oracle.uniform_complex((r, n), 0x5EED1900 + i) for i, r in enumerate(rows)]
    xs = [torch.from_numpy(v).cuda() for v in hs]
    b = S.BatchHandle()
    assert b.make_plan([n, n], list(rows), [x.data_ptr() for x in xs], [x.data_ptr() for x in xs[::-1]], FWD, graph) == S.ACL_SUCCESS
    b.alloc_workspace()
    assert b.exec() == S.ACL_SUCCESS
    torch.cuda.synchronize()
    for i in range(2):
        rel, _ = report(f"swapped problem {i}", xs[1 - i].cpu().numpy(), oracle.c2c(hs[i]))
        assert rel <= 5e-6
    b.destroy()
