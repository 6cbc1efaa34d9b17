"""Performance cases of the transform library: what a program that uses it runs.

A case names a transform kind, its sizes and its precision:

  c2c     complexForward and complexInverse(scale) of a 1D/2D/3D plan
  real    realForward and realInverse(scale) in the packed layout
  full    realForwardFull (the only real transform of 2D/3D sizes that are no
          powers of two)
  dct, dst, dht   forward and inverse, scaled, of a 1D/2D/3D plan
  batch   many lines of one length (FFTBatch1D), both directions
  ragged  many transforms of unequal lengths (RaggedBatch1D), both directions

A program that keeps its plans transforms in place, in both directions.  A
state therefore holds two arrays: a pass transforms one forward and the other
back, and the next pass exchanges their roles, so that values keep their size
however often it runs.  `host` cases hand numpy arrays to the same methods,
as a program does that has its data in host memory.
"""
import math

import numpy as np
import torch

import jtransforms_amd as jt
from jtransforms_amd.workloads import ragged_lengths

PRECISION = {"f64": (torch.float64, "Double", 8), "f32": (torch.float32, "Float", 4)}


def _case(kind, dims, dtype, host=False, **more):
    """dims: the lengths of the axes, as a text like "1080x1920"."""
    return {"kind": kind, "dims": "x".join(str(d) for d in dims), "dtype": dtype, "host": host, **more}


def _dims(case):
    return [int(d) for d in case["dims"].split("x")]


def listed():
    return [
        # one short signal: the call's latency is what counts
        dict(_case("c2c", [1024], "f64"), name="c2c_1d_1024_f64"),
        # one real signal of an ordinary, not power-of-two length
        dict(_case("real", [6000], "f32"), name="real_1d_6000_f32"),
        # a length with a large prime factor (2 * 3 * 1693), as data has that nobody padded
        dict(_case("c2c", [10158], "f64"), name="c2c_1d_10158_f64"),
        # one long record (3 * 2^22 points)
        dict(_case("c2c", [3 << 22], "f64"), name="c2c_1d_12582912_f64"),
        # a large batch of equal lines: channels, traces, frames
        dict(_case("batch", [4096], "f32", batch=16384), name="batch_16384x4096_f32"),
        # records of unequal lengths, 16 to 65536 points, in one call
        dict(_case("ragged", [65536], "f64", batch=4000), name="ragged_4000_f64"),
        # a large padded image or field, double precision
        dict(_case("c2c", [4096, 4096], "f64"), name="c2c_2d_4096x4096_f64"),
        # a video frame at its own size
        dict(_case("c2c", [1080, 1920], "f32"), name="c2c_2d_1080x1920_f32"),
        # a real image in the packed layout
        dict(_case("real", [2048, 2048], "f32"), name="real_2d_2048x2048_f32"),
        # a volume at its own size
        dict(_case("c2c", [180, 180, 180], "f64"), name="c2c_3d_180_f64"),
        # a spectral solver's grid, cosine basis
        dict(_case("dct", [512, 512, 512], "f64"), name="dct_3d_512_f64"),
        # a sine basis on a grid with an odd and an even axis
        dict(_case("dst", [999, 1000], "f64"), name="dst_2d_999x1000_f64"),
    ]


def _smooth(n):
    for p in (2, 3, 5, 7):
        while n % p == 0:
            n //= p
    return n == 1


def _length(rng, style, lo, hi):
    """One length in [lo, hi], spread over its logarithm: a power of two, a
    product of 2, 3, 5 and 7, or any number."""
    n = int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    if style == "pow2":
        return min(1 << round(math.log2(n)), 1 << int(math.log2(hi)))
    if style == "smooth":
        while not _smooth(n):
            n -= 1
    return n


def draw(rng):
    dtype = rng.choice(["f64", "f32"])
    kind = rng.choice(["c2c", "c2c", "real", "full", "dct", "dst", "dht", "batch", "ragged"])
    if kind == "ragged":
        return _case(kind, [65536], dtype, batch=int(math.exp(rng.uniform(math.log(100), math.log(4000)))),
                     lengths=rng.randrange(1 << 20))
    style = rng.choice(["pow2", "smooth", "smooth", "any"])
    if kind == "batch":
        n = _length(rng, style, 16, 8192)
        return _case(kind, [n], dtype, batch=int(math.exp(rng.uniform(math.log(4), math.log((1 << 24) / n)))))
    nd = rng.choice([1, 2, 2, 3])
    if kind == "real" and nd > 1:
        style = "pow2"  # what the packed layout of 2D and 3D is defined for
    top = {"pow2": 1 << 23, "smooth": 1 << 23, "any": 1 << 15 if nd == 1 else 1 << 20}[style]
    host = rng.random() < 0.1
    if host:
        top = min(top, 1 << 20)
    lo, hi = {1: (16, top), 2: (16, 4096), 3: (8, 512)}[nd]
    while True:
        dims = [_length(rng, style, lo, hi) for _ in range(nd)]
        if math.prod(dims) <= top:
            return _case(kind, dims, dtype, host)


def _inputs(case, seed):
    """The two arrays of a state on the GPU, flat: gaussian signals, and
    spectra of the size that such signals have."""
    d = _dims(case)
    dt = PRECISION[case["dtype"]][0]
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    if case["kind"] == "ragged":
        n = 2 * int(_lengths(case).sum())
        return [torch.randn(n, dtype=dt, device="cuda", generator=g) for _ in range(2)]
    tot = math.prod(d) * case.get("batch", 1)
    if case["kind"] == "full":
        return [torch.randn(tot, dtype=dt, device="cuda", generator=g)]
    n = 2 * tot if case["kind"] in ("c2c", "batch") else tot
    a = torch.randn(n, dtype=dt, device="cuda", generator=g)
    b = torch.randn(n, dtype=dt, device="cuda", generator=g)
    if case["kind"] in ("c2c", "batch", "real", "dht"):
        b *= math.sqrt(math.prod(d))
    return [a, b]


def _lengths(case):
    return ragged_lengths(case["batch"], seed=20110602 + case.get("lengths", 0))


def _plan(case):
    d, kind, name = _dims(case), case["kind"], PRECISION[case["dtype"]][1]
    if kind == "ragged":
        return jt.RaggedBatch1D(_lengths(case), precision=case["dtype"])
    if kind == "batch":
        return jt.FFTBatch1D(d[0], case["batch"], precision=case["dtype"])
    family = {"dct": "DCT", "dst": "DST", "dht": "DHT"}.get(kind, "FFT")
    return getattr(jt, "%s%s_%dD" % (name, family, len(d)))(*d)


def prepare(case, seed):
    arrays = _inputs(case, seed)
    if case["kind"] == "full":
        arrays.append(torch.zeros(2 * arrays[0].numel(), dtype=arrays[0].dtype, device="cuda"))
    if case["host"]:
        arrays = [a.cpu().numpy() for a in arrays]
    return {"kind": case["kind"], "plan": _plan(case), "arrays": arrays, "turn": 0}


def run(state):
    p, kind, (a, b) = state["plan"], state["kind"], state["arrays"]
    if kind == "full":
        # the samples arrive in the first half of the array that gets the spectrum
        b[: len(a)] = a
        p.realForwardFull(b)
        return [b]
    if state["turn"]:
        a, b = b, a
    state["turn"] ^= 1
    if kind in ("c2c", "batch", "ragged"):
        p.complexForward(a)
        p.complexInverse(b, True)
    elif kind == "real":
        p.realForward(a)
        p.realInverse(b, True)
    elif kind == "dht":
        p.forward(a)
        p.inverse(b, True)
    else:
        p.forward(a, True)
        p.inverse(b, True)
    return state["arrays"]


def work(case):
    d, kind, size = _dims(case), case["kind"], PRECISION[case["dtype"]][2]
    if kind == "ragged":
        ns = _lengths(case).astype(np.float64)
        return {"bytes": 8 * size * float(ns.sum()), "flops": 10 * float((ns * np.log2(ns)).sum())}
    tot, lines = math.prod(d), case.get("batch", 1)
    flops = 5 * tot * lines * math.log2(tot)
    if kind in ("c2c", "batch"):
        return {"bytes": 8 * size * tot * lines, "flops": 2 * flops}
    if kind == "full":
        return {"bytes": 3 * size * tot, "flops": flops / 2}
    return {"bytes": 4 * size * tot, "flops": flops}


def tolerance(case):
    # about four times the distance from the 64-bit results that was measured
    # over these ranges (8e-16 and 2.4e-7)
    return {"rel": 4e-15} if case["dtype"] == "f64" else {"rel": 1e-6}


# ---------------------------------------------------------------------------
# the same transforms in 64 bits, from their definitions
# ---------------------------------------------------------------------------
def _phase(n, like, sign):
    k = torch.arange(n, dtype=torch.float64, device=like.device) * (sign * math.pi / (2 * n))
    return torch.polar(torch.ones_like(k), k)


def _dct2(x, axis):
    """Orthonormal DCT-II along one axis (Makhoul's n-point form)."""
    x = x.movedim(axis, -1)
    n = x.shape[-1]
    v = torch.cat([x[..., 0::2], x[..., 1::2].flip(-1)], -1)
    c = (torch.fft.fft(v) * _phase(n, x, -1)).real * math.sqrt(2.0 / n)
    c[..., 0] *= math.sqrt(0.5)
    return c.movedim(-1, axis)


def _dct3(y, axis):
    """The inverse of _dct2."""
    y = y.movedim(axis, -1)
    n = y.shape[-1]
    c = y * math.sqrt(n / 2.0)
    c[..., 0] *= math.sqrt(2.0)
    m = torch.cat([torch.zeros_like(c[..., :1]), c[..., 1:].flip(-1)], -1)
    v = torch.fft.ifft(torch.complex(c, -m) * _phase(n, y, 1)).real
    x = torch.empty_like(y)
    x[..., 0::2] = v[..., : (n + 1) // 2]
    x[..., 1::2] = v[..., (n + 1) // 2:].flip(-1)
    return x.movedim(-1, axis)


def _odd_sign(x, axis):
    s = torch.ones(x.shape[axis], dtype=x.dtype, device=x.device)
    s[1::2] = -1
    return x * s.reshape([-1 if i == axis else 1 for i in range(x.dim())])


def _pairs(shape, device):
    """Over the axes before the last: which places of the packed plane pair
    hold the zero-frequency plane, which the other one, the rest both."""
    first = torch.zeros(shape, dtype=torch.bool, device=device)
    if shape:
        idx = torch.meshgrid(*[torch.arange(s, device=device) for s in shape], indexing="ij")
        r, k = shape[-1], idx[-1]
        first = (k > 0) & (k < r // 2)
        if len(shape) == 2:
            first |= ((k == 0) | (k == r // 2)) & (idx[0] > 0) & (idx[0] < shape[0] // 2)
    return first, _mirror(first)


def _mirror(x):
    for axis in range(x.dim()):
        x = x.flip(axis).roll(1, axis)
    return x


def _pack(x):
    """realForward: the spectrum of real x in the packed layout."""
    f = torch.fft.rfftn(x)
    n = x.shape[-1]
    out = torch.empty_like(x)
    if n % 2:
        out[..., 0] = f[..., 0].real
        out[..., 2::2] = f[..., 1:].real
        out[..., 3::2] = f[..., 1:-1].imag
        out[..., 1] = f[..., -1].imag
        return out
    out[..., 2::2] = f[..., 1:-1].real
    out[..., 3::2] = f[..., 1:-1].imag
    lo, hi = f[..., 0], f[..., -1]
    first, second = _pairs(list(x.shape[:-1]), x.device)
    out[..., 0] = torch.where(second, hi.imag, lo.real)
    out[..., 1] = torch.where(first, lo.imag, hi.real)
    return out


def _unpack(a):
    """realInverse(scale): the real data of a packed spectrum."""
    n = a.shape[-1]
    f = torch.zeros(list(a.shape[:-1]) + [n // 2 + 1], dtype=torch.complex128, device=a.device)
    if n % 2:
        f[..., 0] = a[..., 0].to(torch.complex128)
        f[..., 1:-1] = torch.complex(a[..., 2:-1:2], a[..., 3::2])
        f[..., -1] = torch.complex(a[..., -1], a[..., 1])
        return torch.fft.irfft(f, n)
    f[..., 1:-1] = torch.complex(a[..., 2::2].contiguous(), a[..., 3::2].contiguous())
    first, second = _pairs(list(a.shape[:-1]), a.device)
    p, q = a[..., 0], a[..., 1]
    zero = torch.zeros_like(p)
    lo = torch.complex(torch.where(second, zero, p), torch.where(first, q, zero))
    hi = torch.complex(torch.where(first, zero, q), torch.where(second, p, zero))
    f[..., 0] = torch.where(second, _mirror(lo).conj(), lo)
    f[..., -1] = torch.where(first, _mirror(hi).conj(), hi)
    return torch.fft.irfftn(f, s=list(a.shape))


def exact(case, seed):
    d, kind = _dims(case), case["kind"]
    big = kind != "ragged" and math.prod(d) * case.get("batch", 1) >= 1 << 22
    xs = [a.to("cuda" if big else "cpu", torch.float64) for a in _inputs(case, seed)]
    if kind == "ragged":
        out, at = [[], []], 0
        for n in _lengths(case):
            for k, f in enumerate((torch.fft.fft, torch.fft.ifft)):
                z = torch.view_as_complex(xs[k][at:at + 2 * n].reshape(-1, 2))
                out[k].append(torch.view_as_real(f(z)).reshape(-1))
            at += 2 * n
        return [torch.cat(o) for o in out]
    if kind in ("c2c", "batch"):
        shape = ([case["batch"]] if kind == "batch" else []) + d
        axes = list(range(len(shape) - len(d), len(shape)))
        z = [torch.view_as_complex(x.reshape(shape + [2])) for x in xs]
        y = [torch.fft.fftn(z[0], dim=axes), torch.fft.ifftn(z[1], dim=axes)]
        return [torch.view_as_real(v).reshape(-1) for v in y]
    xs = [x.reshape(d) for x in xs]
    if kind == "full":
        return [torch.view_as_real(torch.fft.fftn(xs[0])).reshape(-1)]
    if kind == "real":
        return [_pack(xs[0]).reshape(-1), _unpack(xs[1]).reshape(-1)]
    if kind == "dht":
        f = [torch.fft.fftn(x) for x in xs]
        return [(f[0].real - f[0].imag).reshape(-1), ((f[1].real - f[1].imag) / math.prod(d)).reshape(-1)]
    a, b = xs
    for axis in range(len(d)):
        if kind == "dct":
            a, b = _dct2(a, axis), _dct3(b, axis)
        else:
            a = _dct2(_odd_sign(a, axis), axis).flip(axis)
            b = _odd_sign(_dct3(b.flip(axis), axis), axis)
    return [a.reshape(-1), b.reshape(-1)]
