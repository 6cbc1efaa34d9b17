"""Ragged batches as one launch per pass (batches of 2^17 points and more)
against the oracle: the line limits of one workgroup, lines that need the
wide launch (FP32 above 4096 points), groups of equal lengths with a partly
filled last workgroup, lengths 1 and 2, both directions.  Tolerances as for
single transforms."""
import math

import numpy as np
import pytest

import jtransforms_amd as jt

pytestmark = pytest.mark.gpu

DT = {"f64": np.float64, "f32": np.float32}
LENS = ([1, 2, 4096, 4095, 4097, 4100, 8192, 8190, 7290, 6561, 2047, 2049, 4079, 4103, 65521, 65536, 46875, 12800]
        + [17] * 129 + [16] * 65 + [1] * 65 + [360] * 23 + [37] * 40 + [12800, 10007, 10007])


def tol(n, prec):
    lg = max(1.0, math.log2(max(n, 2)))
    return 1e-13 * lg if prec == "f64" else 2e-7 * lg + 1e-6


def rel(a, b):
    a = np.asarray(a, np.float64).ravel()
    b = np.asarray(b, np.float64).ravel()
    return float(np.linalg.norm(a - b) / np.linalg.norm(b))


@pytest.mark.parametrize("prec", ["f64", "f32"])
def test_passes(orc, prec):
    import torch
    lens = np.random.default_rng(5).permutation(np.array(LENS, dtype=np.int64))
    p = jt.RaggedBatch1D(lens, precision=prec)
    assert "form=launches" in p.describe(), p.describe()
    x = orc.jrandom_doubles(20110609, int(2 * lens.sum())).astype(DT[prec])
    t = torch.from_numpy(x.copy()).cuda()
    p.complexForward(t)
    y = t.cpu().numpy()
    p.sync_status()
    seg = [slice(int(p.offsets[i]), int(p.offsets[i + 1])) for i in range(len(lens))]
    for i, n in enumerate(lens):
        e = rel(y[seg[i]], orc.complex_forward(int(n), x[seg[i]].astype(np.float64)))
        assert e <= tol(n, prec), (i, n, e)
    p.complexInverse(t, True)
    z = t.cpu().numpy()
    t.copy_(torch.from_numpy(y))
    p.complexInverse(t, False)
    w = t.cpu().numpy()
    for i, n in enumerate(lens):
        assert rel(z[seg[i]], x[seg[i]]) <= 2 * tol(n, prec), (i, n)
        assert rel(w[seg[i]], float(n) * x[seg[i]].astype(np.float64)) <= 2 * tol(n, prec), (i, n)


@pytest.mark.parametrize("prec", ["f64", "f32"])
@pytest.mark.parametrize("form", ["persistent", "launches"])
@pytest.mark.parametrize("big", [False, True])
def test_described_schedule_is_accepted(orc, form, big, prec, monkeypatch):
    """JT_RAGGED_SCHEDULE takes what describe() prints, of either form, and
    gives the same schedule for batches on both sides of the default's line;
    tuned plans describe theirs the same way."""
    import torch
    lens = np.array([12800, 10007, 17, 17, 360, 4096] + ([65536, 65521] if big else []), dtype=np.int64)
    monkeypatch.setenv("JT_RAGGED_SCHEDULE", "form=" + form)
    first = jt.RaggedBatch1D(lens, precision=prec).describe()
    assert "form=" + form in first, first
    sched = first.split("schedule ")[1].split()[0]
    monkeypatch.setenv("JT_RAGGED_SCHEDULE", sched)
    p = jt.RaggedBatch1D(lens, precision=prec)
    assert p.describe() == first
    x = orc.jrandom_doubles(20110630, int(2 * lens.sum())).astype(DT[prec])
    t = torch.from_numpy(x.copy()).cuda()
    p.complexForward(t)
    y = t.cpu().numpy()
    p.sync_status()
    for i, n in enumerate(lens):
        s = slice(int(p.offsets[i]), int(p.offsets[i + 1]))
        assert rel(y[s], orc.complex_forward(int(n), x[s].astype(np.float64))) <= tol(n, prec), (i, n)
    if form == "launches" and not big:
        monkeypatch.delenv("JT_RAGGED_SCHEDULE")
        tuned = jt.RaggedBatch1D(lens, precision=prec, autotune=True).describe()
        sched = tuned.split("schedule ")[1].split()[0]
        monkeypatch.setenv("JT_RAGGED_SCHEDULE", sched)
        assert jt.RaggedBatch1D(lens, precision=prec).describe().split("schedule ")[1].split()[0] == sched
