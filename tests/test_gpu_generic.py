"""The runtime-radix kernel (lengths without a compile-time kernel) at the
edges of its shapes: every radix alone and as the first, an inner and the last
stage, the longest lengths, one line, and line counts that leave the last
workgroup partly filled, over rows (batches) and columns (first axis of a 2D
transform).  Tolerances as in test_gpu_fft: FP64 rel-l2 <= 1e-13 * log2(N),
FP32 <= 2e-7 * log2(N) + 1e-6, against the FP64 oracle."""
import math

import numpy as np
import pytest

import jtransforms_amd as jt

pytestmark = pytest.mark.gpu

DT = {"f64": np.float64, "f32": np.float32}
FFT2 = {"f64": jt.DoubleFFT_2D, "f32": jt.FloatFFT_2D}

# one stage; two; three and more (2197 = 13^3, 3125 = 5^5, 3993 = 3 * 11^3); the limits
LENGTHS = [2, 3, 5, 6, 7, 9, 10, 11, 12, 13, 14, 15, 18, 33, 91, 98, 132, 143, 180, 225, 1000, 1331, 2197, 3125, 3993,
           4095]
LENGTHS_F32 = [5000, 6655, 7203, 7290, 8192]


def tol(n, prec):
    lg = max(1.0, math.log2(max(n, 2)))
    return 1e-13 * lg if prec == "f64" else 2e-7 * lg + 1e-6


def rel(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


CASES = [(n, p) for p in ("f64", "f32") for n in LENGTHS] + [(n, "f32") for n in LENGTHS_F32]


@pytest.mark.parametrize("n,prec", CASES)
def test_rows(orc, n, prec):
    for lines in (1, 3, 65, 1030):
        if n * lines > 1 << 20:
            continue
        x = orc.jrandom_doubles(n + lines, 2 * n * lines).astype(DT[prec])
        p = jt.FFTBatch1D(n, lines, precision=prec)
        a = x.copy()
        p.complexForward(a)
        for b in {0, lines // 2, lines - 1}:
            seg = slice(2 * n * b, 2 * n * (b + 1))
            assert rel(a[seg], orc.complex_forward(n, x[seg].astype(np.float64))) <= tol(n, prec), (n, lines, b)
        p.complexInverse(a, True)
        assert rel(a, x) <= 2 * tol(n, prec), (n, lines)


@pytest.mark.parametrize("n,prec", CASES)
def test_columns(orc, n, prec):
    for cols in (3, 17, 250):
        if n * cols > 1 << 18:
            continue
        x = orc.jrandom_doubles(n + cols, 2 * n * cols).astype(DT[prec])
        p = FFT2[prec](n, cols)
        a = x.copy()
        p.complexForward(a)
        e = rel(a, orc.fftnd_complex([n, cols], x.astype(np.float64), -1))
        assert e <= tol(n * cols, prec), (n, cols, e)
        p.complexInverse(a, True)
        assert rel(a, x) <= 2 * tol(n * cols, prec), (n, cols)


R2R2 = {"dct": (jt.DoubleDCT_2D, jt.FloatDCT_2D), "dst": (jt.DoubleDST_2D, jt.FloatDST_2D),
        "dht": (jt.DoubleDHT_2D, jt.FloatDHT_2D)}


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["dct", "dst", "dht"])
@pytest.mark.parametrize("dims", [(4, 6), (6, 4), (8, 10), (10, 14), (18, 512), (1024, 6), (30, 32), (64, 22)])
def test_r2r_quads(orc, kind, dims, prec):
    """The real transforms read and write four elements at a time: half
    lengths that are odd leave a pair, with contiguous and strided lines."""
    x = orc.jrandom_doubles(dims[0], dims[0] * dims[1]).astype(DT[prec])
    p = R2R2[kind][prec == "f32"](*dims)
    for fwd in (True, False):
        scale = kind != "dht" or not fwd
        a = x.copy()
        if fwd:
            p.forward(a, *([True] if kind != "dht" else []))
        else:
            p.inverse(a, True)
        e = rel(a, orc.realnd(kind, list(dims), x.astype(np.float64), fwd, scale))
        assert e <= tol(x.size, prec), (fwd, e)


# convolution lengths just inside and outside one workgroup's LDS (4096 points
# in FP64, 8192 in FP32), short ones, and a two-level one
BLUE = [(n, p) for p in ("f64", "f32") for n in (17, 19, 34, 67, 519, 1021, 2047, 2051, 4079, 4103)] + [(20011, "f64")]


@pytest.mark.parametrize("n,prec", BLUE)
def test_bluestein(orc, n, prec):
    """Bluestein lengths as rows of a batch and as columns, both directions."""
    cls = FFT2[prec]
    for lines in (1, 3, 70):
        if n * lines > 1 << 18:
            continue
        x = orc.jrandom_doubles(n + lines, 2 * n * lines).astype(DT[prec])
        rows = jt.FFTBatch1D(n, lines, precision=prec)
        a = x.copy()
        rows.complexForward(a)
        seg = slice(2 * n * (lines - 1), 2 * n * lines)
        assert rel(a[seg], orc.complex_forward(n, x[seg].astype(np.float64))) <= tol(n, prec), (n, lines)
        rows.complexInverse(a, True)
        assert rel(a, x) <= 2 * tol(n, prec), (n, lines)
    x = orc.jrandom_doubles(n, 2 * n * 6).astype(DT[prec])
    a = x.copy()
    p = cls(n, 6)
    p.complexForward(a)
    assert rel(a, orc.fftnd_complex([n, 6], x.astype(np.float64), -1)) <= tol(6 * n, prec)
    p.complexInverse(a, True)
    assert rel(a, x) <= 2 * tol(6 * n, prec)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [8400, 13125, 16875, 27000, 33075, 78125, 192000])
def test_four_step_few_lines(orc, n, prec):
    """One line and a few of two passes of runtime-radix columns: up to one
    thread per two points, with partly filled last workgroups."""
    for lines in (1, 3):
        x = orc.jrandom_doubles(n + lines, 2 * n * lines).astype(DT[prec])
        p = jt.FFTBatch1D(n, lines, precision=prec)
        a = x.copy()
        p.complexForward(a)
        for b in range(lines):
            s = slice(2 * n * b, 2 * n * (b + 1))
            assert rel(a[s], orc.complex_forward(n, x[s].astype(np.float64))) <= tol(n, prec), (lines, b)
        p.complexInverse(a, True)
        assert rel(a, x) <= 2 * tol(n, prec), lines


# odd lengths (one launch; Bluestein in one launch; several launches), 2, and
# even ones whose half has a large prime factor
PAIR = [2, 3, 9, 37, 74, 225, 999, 1021, 2047, 4095, 4103, 10158]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind", ["dct", "dst", "dht"])
@pytest.mark.parametrize("n", PAIR)
def test_line_pairs(orc, kind, n, prec):
    """Two real lines as one complex transform: contiguous and strided lines,
    an odd number of them (the last pair has one line), both directions."""
    for dims in ((3, n), (n, 5)):
        x = orc.jrandom_doubles(n, n * dims[0 if dims[1] == n else 1]).astype(DT[prec])
        p = R2R2[kind][prec == "f32"](*dims)
        for fwd in (True, False):
            a = x.copy()
            if fwd:
                p.forward(a, *([True] if kind != "dht" else []))
            else:
                p.inverse(a, True)
            e = rel(a, orc.realnd(kind, list(dims), x.astype(np.float64), fwd, kind != "dht" or not fwd))
            assert e <= tol(x.size, prec), (dims, fwd, e)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 9, 37, 225, 1021, 4095, 4103, 33075])
def test_odd_packed_batch(orc, n, prec):
    """realForward / realInverse of odd lengths on a batch with a last single line."""
    lines = 3
    x = orc.jrandom_doubles(n, n * lines).astype(DT[prec])
    p = jt.FFTBatch1D(n, lines, precision=prec)
    a = x.copy()
    p.realForward(a)
    for b in range(lines):
        s = slice(b * n, (b + 1) * n)
        assert rel(a[s], orc.real_forward(n, x[s].astype(np.float64))) <= tol(n, prec), b
    for scale in (True, False):
        c = x.copy()
        p.realInverse(c, scale)
        for b in range(lines):
            s = slice(b * n, (b + 1) * n)
            assert rel(c[s], orc.real_inverse(n, x[s].astype(np.float64), scale)) <= 2 * tol(n, prec), (b, scale)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 9, 37, 225, 1021, 4095, 4103, 33075, 74, 1000, 2042, 4096, 20000])
def test_packed_batch_lines_are_independent(orc, n, prec):
    """The lines of a batch are signals of their own: a line 10^16 times as
    loud as another, or one with a NaN or an infinity, leaves the others what
    they are alone, to the last bit."""
    lines, amp = 5, [1.0, 1e-8, 1e8, 1e-8, 1.0]
    x = orc.jrandom_doubles(n + 1, n * lines).astype(DT[prec]).reshape(lines, n)
    x *= np.array(amp, DT[prec])[:, None]
    p = jt.FFTBatch1D(n, lines, precision=prec)
    ops = {"forward": (lambda a: p.realForward(a), orc.real_forward, ()),
           "inverse": (lambda a: p.realInverse(a, True), orc.real_inverse, (True,))}
    for op, (call, ref, more) in ops.items():
        a = x.reshape(-1).copy()
        call(a)
        a = a.reshape(lines, n)
        for b in range(lines):
            e = rel(a[b], ref(n, x[b].astype(np.float64), *more))
            assert e <= 2 * tol(n, prec), (op, b, e)
        y = x.copy()
        y[1, n // 2], y[2, 0] = np.nan, np.inf
        y = y.reshape(-1)
        call(y)
        y = y.reshape(lines, n)
        for b in (0, 3, 4):
            assert np.array_equal(y[b], a[b]), (op, b)
        assert not np.isfinite(y[1]).all() and not np.isfinite(y[2]).all(), op


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("n", [3, 225, 4095, 33075])
def test_odd_packed_large_values(orc, n, prec):
    """A sum of 0.6 times the type's largest value is a result, not an overflow."""
    x = orc.jrandom_doubles(n, n) + 2.0  # positive: the first value is the largest
    want = orc.real_forward(n, x)
    top = 0.6 * float(np.finfo(DT[prec]).max) / np.abs(want).max()
    a = (x * top).astype(DT[prec])
    jt.FFTBatch1D(n, 1, precision=prec).realForward(a)
    assert np.isfinite(a).all()
    assert rel(a.astype(np.float64) / top, want) <= tol(n, prec)


# line pairs of one launch and of several, half-length forms; (kind, n, forward, scale)
LARGE = ([("dht", n, True, False) for n in (3, 225, 1021, 2042, 4103, 16875, 65536)]
         + [("dct", n, True, False) for n in (3, 225, 1021, 4103, 10158)]
         + [("dct", 3, False, True), ("dst", 3, False, True), ("dct", 65536, False, False),
            ("dst", 65536, False, False)])


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind,n,fwd,scale", LARGE)
def test_r2r_large_values(orc, kind, n, fwd, scale, prec):
    """Results and inputs of up to 0.6 times the type's largest value."""
    cls = {"dct": (jt.DoubleDCT_1D, jt.FloatDCT_1D), "dst": (jt.DoubleDST_1D, jt.FloatDST_1D),
           "dht": (jt.DoubleDHT_1D, jt.FloatDHT_1D)}[kind][prec == "f32"]
    x = orc.jrandom_doubles(n, n)
    want = orc.realnd(kind, [n], x, fwd, scale)
    top = 0.6 * float(np.finfo(DT[prec]).max) / max(np.abs(want).max(), np.abs(x).max())
    a = (x * top).astype(DT[prec])
    p = cls(n)
    if fwd:
        p.forward(a, *([scale] if kind != "dht" else []))
    else:
        p.inverse(a, scale)
    assert np.isfinite(a).all()
    assert rel(a.astype(np.float64) / top, want) <= tol(n, prec)


# single-launch, Bluestein and several-launch plans on each axis
FULL = [(2,), (16,), (37,), (360,), (4096,), (2047,), (4103,), (10158,), (2, 2), (9, 37), (37, 16), (64, 225),
        (4103, 3), (3, 4103), (5, 6, 7), (16, 37, 9), (3, 4, 10158)]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("dims", FULL)
def test_real_full(orc, dims, prec):
    """realForwardFull / realInverseFull(scale) where the row pass reads the
    reals, and where it cannot."""
    tot = int(np.prod(dims))
    x = orc.jrandom_doubles(tot, tot).astype(DT[prec])
    src = np.concatenate([x, np.zeros_like(x)])
    cls = [{"f64": jt.DoubleFFT_1D, "f32": jt.FloatFFT_1D}, FFT2, {"f64": jt.DoubleFFT_3D, "f32": jt.FloatFFT_3D}]
    p = cls[len(dims) - 1][prec](*dims)
    z = (x.astype(np.float64) + 0j).reshape(dims)
    for fwd in (True, False):
        a = src.copy()
        if fwd:
            p.realForwardFull(a)
        else:
            p.realInverseFull(a, True)
        want = np.fft.fftn(z) if fwd else np.fft.ifftn(z)
        e = rel(a, np.ascontiguousarray(want).view(np.float64))
        assert e <= tol(tot, prec), (fwd, e)


@pytest.mark.parametrize("first", [True, False])
def test_device_calls_refused(first):
    """What a plan's calls on device tensors refuse, its first call or a later one."""
    import torch
    n = 600
    good = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
    bad = [(TypeError, good.float()), (TypeError, good.cpu()), (TypeError, good.reshape(2, n)),
           (TypeError, torch.zeros(4 * n, dtype=torch.float64, device="cuda")[::2]), (IndexError, good[:-1]),
           (IndexError, good, 1), (ValueError, good, -1)]
    for err, *args in bad:
        p = jt.DoubleFFT_1D(n)
        if not first:
            p.complexForward(good)
        with pytest.raises(err):
            p.complexForward(*args)
        p.complexForward(good)
    with pytest.raises(ValueError):
        jt.DoubleDCT_1D(n)._run(jt.COMPLEX_FORWARD, good)  # an op that the plan does not have


def test_device_calls_after_the_first(orc):
    """Calls of a plan on flat device tensors take a short path: the same
    results, streams, offsets and refusals from the first call on."""
    import torch
    n = 600
    x = orc.jrandom_doubles(n, 2 * n + 3)
    p = jt.DoubleFFT_1D(n)
    want = orc.complex_forward(n, x[:2 * n])
    for rep in range(3):
        t = torch.from_numpy(x.copy()).cuda()
        torch.cuda.synchronize()
        p.complexForward(t)
        y = t.cpu().numpy()
        assert rel(y[:2 * n], want) <= tol(n, "f64") and np.array_equal(y[2 * n:], x[2 * n:])
    # on a stream of the caller's: the input arrives there, behind work that
    # takes milliseconds, so that a call on any other stream would transform
    # what is in t before and then be overwritten
    s = torch.cuda.Stream()
    src = torch.from_numpy(x.copy()).cuda()
    t = torch.zeros_like(src)
    m = torch.ones(4096, 4096, device="cuda")
    torch.mm(m, m)
    torch.cuda.synchronize()
    with torch.cuda.stream(s):
        assert jt._raw_stream(torch, torch.cuda.current_device()) == s.cuda_stream
        for _ in range(20):
            torch.mm(m, m)
        t.copy_(src)
        p.complexForward(t)
        y = t.to("cpu", non_blocking=False).numpy()
    assert rel(y[:2 * n], want) <= tol(n, "f64")
    assert jt._raw_stream(torch, torch.cuda.current_device()) == torch.cuda.current_stream().cuda_stream
    t = torch.from_numpy(x.copy()).cuda()
    p.complexForward(t, 3)  # misaligned pairs
    assert rel(t.cpu().numpy()[3:], orc.complex_forward(n, x[3:])) <= tol(n, "f64")
    good = torch.zeros(2 * n, dtype=torch.float64, device="cuda")
    with pytest.raises(TypeError):
        p.complexForward(good.float())
    with pytest.raises(TypeError):
        p.complexForward(good.cpu())
    with pytest.raises(TypeError):
        p.complexForward(torch.zeros(4 * n, dtype=torch.float64, device="cuda")[::2])
    with pytest.raises(TypeError):
        p.complexForward(good.reshape(2, n))
    with pytest.raises(IndexError):
        p.complexForward(good[:-1])
    with pytest.raises(IndexError):
        p.complexForward(good, 1)
    with pytest.raises(ValueError):
        p.complexForward(good, -1)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("rows,cols", [(256, 3), (256, 1030), (512, 520), (1024, 515), (1024, 1030), (2048, 129),
                                       (4096, 65), (2048, 1024)])
def test_narrow_column_groups(orc, rows, cols, prec):
    """Compile-time columns in groups of full, half and quarter width, with a
    partly filled last group; the packed real form where cols allows."""
    x = orc.jrandom_doubles(rows + cols, 2 * rows * cols).astype(DT[prec])
    p = FFT2[prec](rows, cols)
    a = x.copy()
    p.complexForward(a)
    assert rel(a, orc.fftnd_complex([rows, cols], x.astype(np.float64), -1)) <= tol(rows * cols, prec)
    p.complexInverse(a, True)
    assert rel(a, x) <= 2 * tol(rows * cols, prec)
    if cols & (cols - 1) == 0:
        r = x[:rows * cols].copy()
        p.realForward(r)
        assert rel(r, orc.fft2d_real_forward(rows, cols, x[:rows * cols].astype(np.float64))) <= tol(rows * cols, prec)
        p.realInverse(r, True)
        assert rel(r, x[:rows * cols]) <= 2 * tol(rows * cols, prec)
