"""Performance cases of the FFT library: what a program has it do, through the public handles.

A case is a dict of plain values. `listed()` names the standing ones, `draw(rng)` makes another of the
same ranges, `prepare(case, seed)` makes inputs, plan and workspace on the GPU as a program keeps them
across calls, `run(state)` is one pass (it only enqueues), `exact(case, seed)` the same outputs in
64-bit arithmetic by torch on the CPU, and `work(case)` the bytes and operations of one pass that no
implementation can do without.

Kinds of cases:
  c2c     complex transforms in 1-3 dimensions ("dims", e.g. "1024x1024"), either direction;
          layout "rows" or "vertical" (1D transforms down the columns of an (n, batch) array);
          planes "interleaved" or "split" (real and imaginary parts in arrays of their own);
          precision "fp32" or one of the matrix-core modes
  r2c     real to half spectrum, c2r half spectrum to real (1D and 2D)
  istft   inverse short-time transform with overlap-add
  uneven  many 1D problems of uneven 2,3,5-smooth lengths bound into one launch
"""
import math
import random

import torch

import sip_amd as S

PRECISION = {"fp32": S.PREC_FP32, "f16x2": S.PREC_F16_SPLIT, "bf16x3": S.PREC_BF16_SPLIT3}


def _case(kind, dims="", batch=1, **kw):
    c = {"kind": kind, "dims": dims, "batch": batch}
    if kind == "c2c":
        c.update(inverse=False, layout="rows", planes="interleaved", precision="fp32")
    c.update(kw)
    return c


def listed():
    return [
        # one short call on a small batch: latency (a filter bank's or a detector's frame)
        _case("c2c", "1024", 256, name="c2c_1024x256"),
        # the benchmark's headline: a large batch of power-of-two rows
        _case("c2c", "4096", 16384, name="c2c_4096x16384"),
        # mixed radices (2^4 5^3), inverse: sampling rates are rarely powers of two
        _case("c2c", "2000", 8192, inverse=True, name="c2c_2000x8192_inverse"),
        # a record length nobody chose: a large prime factor
        _case("c2c", "1009", 4096, name="c2c_1009x4096_prime"),
        # few long records: spectra of whole captures
        _case("c2c", "1048576", 8, name="c2c_1048576x8_long"),
        # real signals to half spectra, rows
        _case("r2c", "8192", 4096, inverse=False, name="r2c_8192x4096"),
        # split planes at the longest of the entry point's documented lengths (2..256)
        _case("c2c", "256", 32768, planes="split", name="c2c_256x32768_split"),
        # 2D on the matrix cores (FP16 hi + lo operands)
        _case("c2c", "1024x1024", 8, precision="f16x2", name="c2c_1024x1024x8_f16x2"),
        # 3D volumes (plain form)
        _case("c2c", "128x128x128", 4, name="c2c_128x128x128x4"),
        # images back from their half spectra (full-HD frames, ragged in both axes)
        _case("c2r", "1080x1920", 8, inverse=True, name="c2r_1080x1920x8"),
        # audio: inverse short-time transform, 75 % overlap
        _case("istft", "1024", 8, hop=256, frames=2049, name="istft_1024_hop256"),
        # uneven lengths in one launch
        _case("uneven", "", 256, lo=64, hi=65536, max_batch=64, mix=4, name="uneven_256"),
    ]


# ---------------------------------------------------------------------------------------- drawn cases

def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


_SMOOTH = S.smooth_lengths(16, 1 << 20)


def _smooth(rng, lo, hi):
    x = _log(rng, lo, hi)
    return min((v for v in _SMOOTH if lo <= v <= hi), key=lambda v: abs(math.log(v / x)))


def _pow2(rng, lo, hi):
    return 1 << rng.randint(lo.bit_length() - 1, hi.bit_length() - 1)


def _batch(rng, per, lo, hi):
    """A batch so that the points of the call are log-uniform in [lo, hi]."""
    return max(1, int(_log(rng, lo, hi) / per))


def draw(rng: random.Random):
    kind = rng.choice(["c2c1", "c2c1", "c2c1", "any", "vertical", "split", "c2c2", "c2c3", "precision", "r2c", "c2r",
                       "real2", "istft", "uneven"])
    inv = rng.random() < 0.5
    if kind == "c2c1":
        n = _pow2(rng, 16, 1 << 20) if rng.random() < 0.4 else _smooth(rng, 16, 1 << 20)
        return _case("c2c", str(n), _batch(rng, n, 1 << 17, 1 << 25), inverse=inv)
    if kind == "any":  # whatever length: most of these have a large prime factor
        n = int(_log(rng, 17, 20000))
        return _case("c2c", str(n), _batch(rng, n, 1 << 16, 1 << 22), inverse=inv)
    if kind == "vertical":
        n = _smooth(rng, 32, 4096)
        return _case("c2c", str(n), max(2, _batch(rng, n, 1 << 17, 1 << 24)), inverse=inv, layout="vertical")
    if kind == "split":
        n = _smooth(rng, 16, 4096)
        return _case("c2c", str(n), _batch(rng, n, 1 << 17, 1 << 24), inverse=inv, planes="split")
    if kind == "c2c2":
        a, b = _smooth(rng, 32, 2048), _smooth(rng, 32, 2048)
        return _case("c2c", "%dx%d" % (a, b), _batch(rng, a * b, 1 << 17, 1 << 24), inverse=inv)
    if kind == "c2c3":
        a, b, c = (_smooth(rng, 24, 160) for _ in range(3))
        return _case("c2c", "%dx%dx%d" % (a, b, c), _batch(rng, a * b * c, 1 << 17, 1 << 24), inverse=inv)
    if kind == "precision":
        p = rng.choice(["f16x2", "bf16x3"])
        if rng.random() < 0.5:
            n = _pow2(rng, 128, 4096)
            return _case("c2c", str(n), _batch(rng, n, 1 << 18, 1 << 24), inverse=inv, precision=p)
        a, b = _pow2(rng, 128, 2048), _pow2(rng, 128, 2048)
        return _case("c2c", "%dx%d" % (a, b), _batch(rng, a * b, 1 << 18, 1 << 24), inverse=inv, precision=p)
    if kind in ("r2c", "c2r"):
        if rng.random() < 0.25:  # odd lengths
            n = rng.choice([v for v in _SMOOTH if v % 2 and v <= 16384])
        else:
            n = 2 * (_pow2(rng, 16, 32768) if rng.random() < 0.4 else _smooth(rng, 16, 32768))
        return _case(kind, str(n), _batch(rng, n, 1 << 17, 1 << 25), inverse=kind == "c2r")
    if kind == "real2":
        a, b = _smooth(rng, 32, 2048), 2 * _smooth(rng, 16, 1024)
        k = rng.choice(["r2c", "c2r"])
        return _case(k, "%dx%d" % (a, b), _batch(rng, a * b, 1 << 17, 1 << 24), inverse=k == "c2r")
    if kind == "istft":
        n = _smooth(rng, 128, 1499)  # the entry point's longest frame
        hop = max(1, n // rng.choice([2, 4, 4, 8]))
        ch = rng.randint(1, 16)
        return _case("istft", str(n), ch, hop=hop, frames=max(8, _batch(rng, n * ch, 1 << 17, 1 << 24)))
    return _case("uneven", "", int(_log(rng, 24, 256)), lo=64, hi=rng.choice([4096, 16384, 65536]), max_batch=64,
                 mix=rng.randint(1, 1 << 30))


# ---------------------------------------------------------------------------------------- preparing

def _dims(case):
    return [int(v) for v in case["dims"].split("x")]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) * 7919 + 17)


def _uniform_complex(g, shape):
    x = torch.empty(*shape, 2, device="cuda").uniform_(-1.0, 1.0, generator=g)
    return torch.view_as_complex(x)


def _tones(g, seed, batch, dims):
    """Gaussian noise and three pure tones of amplitude 1e3 at random bins: a dynamic range that the
    matrix-core modes have to keep."""
    x = torch.view_as_complex(torch.empty(batch, *dims, 2, device="cuda").normal_(generator=g))
    rng = random.Random(int(seed))
    for _ in range(3):
        phase = torch.zeros((), dtype=torch.float64, device="cuda")
        for ax, n in enumerate(dims):
            shape = [1] * len(dims)
            shape[ax] = n
            k = rng.randrange(n)
            phase = phase + (torch.arange(n, device="cuda").mul(k).remainder(n).double() / n).view(shape)
        x += torch.polar(torch.full_like(phase, 1e3), 2 * math.pi * phase).to(torch.complex64)
    return x


def _input(case, seed):
    g = _gen(seed)
    kind, B = case["kind"], case["batch"]
    if kind == "uneven":
        lengths, batches = _uneven(case)
        return _uniform_complex(g, (sum(n * b for n, b in zip(lengths, batches)),))
    dims = _dims(case)
    if kind == "istft":
        x = torch.empty(B, dims[0], case["frames"], 2, device="cuda").normal_(generator=g)
        return torch.view_as_complex(x)
    if kind == "r2c":
        return torch.empty(B, *dims, device="cuda").uniform_(-1.0, 1.0, generator=g)
    if kind == "c2r":
        return _uniform_complex(g, (B, *dims[:-1], dims[-1] // 2 + 1))
    if case["precision"] != "fp32":
        return _tones(g, seed, B, dims)
    if case["layout"] == "vertical":
        return _uniform_complex(g, (dims[0], B))
    return _uniform_complex(g, (B, *dims))


def _uneven(case):
    return S.batching_workload(case["batch"], case["mix"], case["lo"], case["hi"], case["max_batch"])


def _window(n):
    """Periodic Hann."""
    return 0.5 - 0.5 * torch.cos(2 * math.pi * torch.arange(n, dtype=torch.float64) / n)


def _ok(status):
    if status != S.ACL_SUCCESS:
        raise RuntimeError("status %d" % status)


def prepare(case, seed):
    x = _input(case, seed)
    kind, B = case["kind"], case["batch"]
    if kind == "uneven":
        lengths, batches = _uneven(case)
        y = torch.empty_like(x)
        offs = [0]
        for n, b in zip(lengths, batches):
            offs.append(offs[-1] + 8 * n * b)
        h = S.BatchHandle()
        _ok(h.make_plan(lengths, batches, [x.data_ptr() + o for o in offs[:-1]], [y.data_ptr() + o for o in offs[:-1]],
                        S.ASCEND_FFT_FORWARD, S.BATCH_GRAPH | S.BATCH_PERSIST))
        h.alloc_workspace()
        stream = torch.cuda.current_stream().cuda_stream
        if stream:
            _ok(h.set_stream(stream))
        return {"kind": kind, "h": h, "x": x, "y": y}
    h = S.FftHandle()
    dims = _dims(case)
    if kind == "istft":
        n, hop, frames = dims[0], case["hop"], case["frames"]
        _ok(h.istft_make_plan(x, n, hop, n))
        y = torch.empty(B, n + hop * (frames - 1) - 2 * (n // 2), dtype=torch.complex64, device="cuda")
        w = _window(n).float().cuda()
        state = {"kind": kind, "h": h, "x": x, "y": y, "w": w}
    else:
        split = kind == "c2c" and case["planes"] == "split"
        ftype = {"r2c": S.ASCEND_FFT_R2C, "c2r": S.ASCEND_FFT_C2R}.get(
            kind, S.ASCEND_FFT_C2C_SEP if split else S.ASCEND_FFT_C2C)
        direction = S.ASCEND_FFT_INVERSE if case["inverse"] else S.ASCEND_FFT_FORWARD
        if kind == "c2c" and case["precision"] != "fp32":
            _ok(h.set_precision(PRECISION[case["precision"]]))
        if len(dims) == 1:
            dim_type = S.ASCEND_FFT_VERTICAL if case.get("layout") == "vertical" else S.ASCEND_FFT_HORIZONTAL
            _ok(h.make_plan_1d(dims[0], ftype, direction, B, dim_type))
        elif len(dims) == 2:
            _ok(h.make_plan_2d(*dims, ftype, direction, B))
        else:
            _ok(h.make_plan_3d(*dims, ftype, direction, B))
        if split:
            xs = (x.real.contiguous(), x.imag.contiguous())
            ys = tuple(torch.empty_like(v) for v in xs)
            state = {"kind": "split", "h": h, "x": xs, "y": ys}
        elif kind == "r2c":
            y = torch.empty(B, *dims[:-1], dims[-1] // 2 + 1, dtype=torch.complex64, device="cuda")
            state = {"kind": kind, "h": h, "x": x, "y": y}
        elif kind == "c2r":
            state = {"kind": kind, "h": h, "x": x, "y": torch.empty(B, *dims, device="cuda")}
        else:
            state = {"kind": kind, "h": h, "x": x, "y": torch.empty_like(x)}
    h.alloc_workspace()
    h.use_current_torch_stream()
    return state


# ---------------------------------------------------------------------------------------- one pass

def run(state):
    kind, h, x, y = state["kind"], state["h"], state["x"], state["y"]
    if kind == "c2c":
        st = h.exec_c2c(x, y)
    elif kind == "split":
        st = h.exec_c2c_separated(*x, *y)
    elif kind == "r2c":
        st = h.exec_r2c(x, y)
    elif kind == "c2r":
        st = h.exec_c2r(x, y)
    elif kind == "istft":
        st = h.exec_istft(x, state["w"], y)
    else:
        st = h.exec()
    _ok(st)
    return y


# ---------------------------------------------------------------------------------------- 64-bit results

def _c2c64(x, dim, inverse):
    return torch.fft.ifftn(x, dim=dim, norm="forward") if inverse else torch.fft.fftn(x, dim=dim)


def exact(case, seed):
    """Transforms are not normalised in either direction."""
    x = _input(case, seed).cpu()
    kind = case["kind"]
    if kind == "uneven":
        lengths, batches = _uneven(case)
        out, o = torch.empty(x.shape, dtype=torch.complex128), 0
        for n, b in zip(lengths, batches):
            out[o:o + n * b] = torch.fft.fft(x[o:o + n * b].view(b, n).to(torch.complex128)).reshape(-1)
            o += n * b
        return out
    dims = _dims(case)
    axes = tuple(range(-len(dims), 0))
    if kind == "istft":
        n, hop, frames = dims[0], case["hop"], case["frames"]
        w = _window(n).float().double()
        f = torch.fft.ifft(x.to(torch.complex128), dim=1) * w.view(1, n, 1)
        at = (torch.arange(n).view(n, 1) + hop * torch.arange(frames).view(1, frames)).reshape(-1)
        span = n + hop * (frames - 1)
        y = torch.zeros(x.shape[0], span, dtype=torch.complex128).index_add_(1, at, f.reshape(x.shape[0], -1))
        env = torch.zeros(span, dtype=torch.float64).index_add_(0, at, (w * w).view(n, 1).expand(n, frames).reshape(-1))
        return (y / env)[:, n // 2:span - n // 2].contiguous()
    if kind == "r2c":
        return torch.fft.rfftn(x.double(), dim=axes)
    if kind == "c2r":
        x = x.to(torch.complex128)
        if len(dims) > 1:
            x = _c2c64(x, axes[:-1], True)
        # the imaginary parts of the zero bin and, for even lengths, of the last one are dropped
        x[..., 0].imag.zero_()
        if dims[-1] % 2 == 0:
            x[..., -1].imag.zero_()
        return torch.fft.irfft(x, n=dims[-1], norm="forward")
    x = x.to(torch.complex128)
    if case["layout"] == "vertical":
        return _c2c64(x, (0,), case["inverse"])
    y = _c2c64(x, axes, case["inverse"])
    if case["planes"] == "split":
        return y.real.contiguous(), y.imag.contiguous()
    return y


# ---------------------------------------------------------------------------------------- work

def work(case):
    """Each input read once and each output written once; 5 n log2 n operations a complex transform of
    n points (half of that for real data)."""
    kind, B = case["kind"], case["batch"]
    if kind == "uneven":
        lengths, batches = _uneven(case)
        return {"bytes": sum(16 * n * b for n, b in zip(lengths, batches)),
                "flops": sum(5 * n * math.log2(n) * b for n, b in zip(lengths, batches))}
    dims = _dims(case)
    n = math.prod(dims)
    if kind == "istft":
        frames, hop = case["frames"], case["hop"]
        out = n + hop * (frames - 1) - 2 * (n // 2)
        return {"bytes": 8 * B * (n * frames + out) + 4 * n,
                "flops": B * frames * (5 * n * math.log2(n) + 4 * n)}
    half = math.prod(dims[:-1]) * (dims[-1] // 2 + 1)
    if kind in ("r2c", "c2r"):
        return {"bytes": B * (4 * n + 8 * half), "flops": B * 2.5 * n * math.log2(n)}
    return {"bytes": 16 * B * n, "flops": 5 * B * n * math.log2(n)}
