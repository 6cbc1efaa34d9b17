"""One plan shared by several host threads and streams.

The reference's 1D plans keep read-only tables and allocate their scratch per
call (fft/DoubleFFT_1D.java:1922 Bluestein `ak`, :6639 mixed-radix `ch`;
fft/DoubleFFT_2D.java:2644 column `t`), so one plan object serves concurrent
callers.  Here the plan owns one device buffer (workspace and staging);
calls that use it are serialised by the library.  Every result is checked
against the oracle (FP64 rel-l2 <= 1e-13*log2 n).
"""
import math
import threading

import numpy as np
import pytest

import jtransforms_amd as jt

pytestmark = pytest.mark.gpu


def tol(n):
    return 1e-13 * max(1.0, math.log2(n))


def rel(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("n", [4096, 10007])  # one-pass kernel; Bluestein (workspace)
def test_host_threads_share_one_plan(orc, n):
    plan = jt.DoubleFFT_1D(n)
    inputs = [orc.jrandom_doubles(9000 + s, 2 * n) for s in range(8)]
    want = [orc.complex_forward(n, x) for x in inputs]
    errors = []

    def worker(tid):
        try:
            for c in range(50):
                k = (tid * 3 + c) % len(inputs)
                a = inputs[k].copy()
                plan.complexForward(a)
                e = rel(a, want[k])
                if e > tol(n):
                    errors.append((tid, c, k, e))
        except Exception as ex:  # reported below
            errors.append((tid, repr(ex)))

    threads = [threading.Thread(target=worker, args=(t,)) for t in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    print(f"n={n}: 4 threads x 50 host calls, failures: {errors[:3]}", flush=True)
    assert not errors


@pytest.mark.parametrize("n,offa", [(4096, 0), (65536, 0), (10007, 0), (4096, 1)])
def test_two_streams_share_one_plan(orc, n, offa):
    """Calls alternate between two streams on distinct buffers; 65536 runs
    four-step and 10007 Bluestein through the plan's workspace, offset 1
    misaligns the complex pairs so every call runs through the staging
    area."""
    import torch
    plan = jt.DoubleFFT_1D(n)
    xs = [orc.jrandom_doubles(7000 + s, 2 * n + offa) for s in range(12)]
    bufs = [torch.from_numpy(x.copy()).cuda() for x in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for rep in range(2):
        for i, b in enumerate(bufs):
            with torch.cuda.stream(streams[i % 2]):
                if rep == 0:
                    plan.complexForward(b, offa)
                else:
                    plan.complexInverse(b, offa, True)
        if rep == 0:
            for s in streams:
                s.synchronize()
            for i, b in enumerate(bufs):
                got = b.cpu().numpy()[offa:]
                e = rel(got, orc.complex_forward(n, xs[i][offa:]))
                assert e <= tol(n), (i, e)
                if offa:
                    assert got.size == 2 * n and b[0].item() == xs[i][0]
    for s in streams:
        s.synchronize()
    for i, b in enumerate(bufs):
        assert rel(b.cpu().numpy(), xs[i]) <= 2 * tol(n), i


# forms that use the plan's workspace and forms that do not, neighbours of the
# line between them: Bluestein in one launch and in three, odd and half-length
# real transforms of one launch and of several, the expanded real transforms
SHARED = [("c2c", (1021,)), ("c2c", (4103,)), ("c2c", (37, 1021)), ("c2c", (6, 10007)), ("real", (999,)),
          ("real", (1021,)), ("real", (33075,)), ("real", (2042,)), ("real", (20000,)), ("real", (64, 128)),
          ("full", (360,)), ("full", (10158,)), ("full", (64, 225)), ("full", (5, 6, 7)), ("full", (3, 10007)),
          ("dct", (4103,)), ("dct", (1021,)), ("dct", (20014,)), ("dct", (9, 10, 11)), ("dst", (999, 1000)),
          ("dht", (33075,)), ("dht", (101, 6))]


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("kind,dims", SHARED)
def test_two_streams_share_one_plan_forms(kind, dims, prec):
    """Calls of one plan on distinct buffers alternate between two streams,
    several deep; every result is to the last bit what the call gives alone."""
    import torch
    family = {"dct": "DCT", "dst": "DST", "dht": "DHT"}.get(kind, "FFT")
    plan = getattr(jt, "%s%s_%dD" % ("Double" if prec == "f64" else "Float", family, len(dims)))(*dims)
    names = {"c2c": ("complexForward", "complexInverse"), "real": ("realForward", "realInverse"),
             "full": ("realForwardFull", "realInverseFull")}.get(kind, ("forward", "inverse"))
    fwd, inv = (getattr(plan, m) for m in names)
    if kind in ("dct", "dst"):
        fwd = lambda a: plan.forward(a, True)  # noqa: E731
    n = math.prod(dims) * (2 if kind in ("c2c", "full") else 1)
    g = torch.Generator(device="cuda")
    g.manual_seed(n)
    dt = torch.float64 if prec == "f64" else torch.float32
    src = [torch.randn(n, dtype=dt, device="cuda", generator=g) for _ in range(8)]
    want = []
    for i, x in enumerate(src):
        y = x.clone()
        inv(y, True) if i % 4 > 1 else fwd(y)
        torch.cuda.synchronize()
        want.append(y)
    assert all(torch.isfinite(w).all() for w in want)
    streams = [torch.cuda.Stream(), torch.cuda.Stream()]
    for rep in range(3):
        bufs = [x.clone() for x in src]
        torch.cuda.synchronize()
        for i, b in enumerate(bufs):
            with torch.cuda.stream(streams[i % 2]):
                inv(b, True) if i % 4 > 1 else fwd(b)
        torch.cuda.synchronize()
        for i, b in enumerate(bufs):
            assert torch.equal(b, want[i]), (rep, i)


def test_threads_and_streams_mixed(orc):
    """Host-array calls from two threads while a third thread drives device
    calls on its own stream, all on one four-step plan."""
    import torch
    n = 65536
    plan = jt.DoubleFFT_1D(n)
    x = orc.jrandom_doubles(4242, 2 * n)
    want = orc.complex_forward(n, x)
    errors = []

    def host_worker():
        try:
            for _ in range(20):
                a = x.copy()
                plan.complexForward(a)
                if rel(a, want) > tol(n):
                    errors.append("host")
        except Exception as ex:
            errors.append(repr(ex))

    def device_worker():
        try:
            s = torch.cuda.Stream()
            bufs = [torch.from_numpy(x.copy()).cuda() for _ in range(20)]
            with torch.cuda.stream(s):
                for b in bufs:
                    plan.complexForward(b)
            s.synchronize()
            for b in bufs:
                if rel(b.cpu().numpy(), want) > tol(n):
                    errors.append("device")
        except Exception as ex:
            errors.append(repr(ex))

    ts = [threading.Thread(target=host_worker), threading.Thread(target=host_worker),
          threading.Thread(target=device_worker)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not errors, errors[:3]
