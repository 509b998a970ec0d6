"""Time-domain PCC1 / PCC-v where the tiled kernel can go wrong: lag blocks of up to 224
and 480 lags (bands of 32), chunks of 512 samples, split and unsplit
launches, and the records that decide between its two ways of summing PCC1's terms; and
the kernel of one lag a thread at its edges."""
import ctypes

import numpy as np
import pytest

from fastpcc_amd import _lib, api

pytestmark = pytest.mark.gpu
# A term is in [-2, 2]; its half-angle phasors are rounded to 2^-25 of each component,
# products of them are exact in three bf16 parts and summed in FP32 (a few 2^-23 of a
# term), a dropped correction is at most 2^-24, and the FP32 analytic signal moves a
# phasor by about 3e-7 / |z|, which averages out: 1e-6 over 400 terms and more.  Short
# overlaps can hold single phasors of small |z| (1e-5, as the other tests).
TOL, TOL_SHORT, LONG = 1e-6, 1e-5, 400


def _records(S, W, N, seed, what):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((S, W, N)).astype(np.float32)
    n = np.arange(N)
    if what == "event":  # a decaying event far above the noise: large regulariser differences
        x[:, 0] += (300 * np.exp(-n / 40.0) * np.sin(0.7 * n)).astype(np.float32)
    elif what == "silent":
        x[1, -1] = 0
        x[0, 0, : N // 2] = 0
    elif what == "antiphase":  # one modulated tone and its negative: |a+b| = |d| at every sample
        tone = ((1.5 + np.sin(2 * np.pi * 3 * n / N)) * np.sin(0.9 * n)).astype(np.float32)
        x[0] = tone
        x[1:] = -tone
    return x.reshape(S, W * N)


def _check(y, yr, N, lag1, lag2, tol=TOL):
    long_ = N - np.abs(np.arange(lag1, lag2 + 1)) >= LONG
    d = np.abs(y - yr)
    err = [float(d[..., m].max()) if m.any() else 0.0 for m in (long_, ~long_)]
    print(f"  max|gpu-fp64| {err[0]:.2e} (overlap >= {LONG}), {err[1]:.2e}")
    assert err[0] <= tol and err[1] <= TOL_SHORT


@pytest.mark.parametrize("S,W,N,lag1,lag2,stack", [
    (2, 1, 511, 0, 0, "none"), (2, 1, 512, -16, 15, "none"), (2, 1, 513, -16, 16, "none"),
    (3, 2, 1025, -112, 111, "none"), (3, 2, 1024, -112, 112, "plain"), (2, 5, 1600, -240, 239, "plain"),
    (2, 1, 5003, -240, 240, "none"), (4, 8, 1700, 37, 690, "plain"), (12, 12, 700, -240, 240, "plain"),
    (12, 8, 900, -480, 480, "plain")])
@pytest.mark.parametrize("kind,v", [("pcc1", 1.0), ("pccv", 2.0), ("pccv", 1.5)])
def test_tile_edges(fp, orc, launched, S, W, N, lag1, lag2, stack, kind, v):
    x = _records(S, W, N, S * N + W, "noise")
    y, names = launched(lambda: fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack, v=v))
    assert kind + "_time" in names and kind + "_direct" not in names
    yr = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True, v=v)
    _check(y, yr, N, lag1, lag2)


# one lag a thread: blocks of 256 lags in waves of 64, chunks of 256 samples in runs of 64
@pytest.mark.parametrize("S,W,N,lag1,lag2,stack", [
    (2, 1, 2, -1, 1, "none"), (40, 24, 64, -31, 31, "none"), (40, 24, 64, -63, 63, "plain"),
    (30, 9, 65, -64, 64, "none"), (30, 9, 255, 0, 0, "none"), (24, 8, 256, -32, 31, "none"),
    (24, 8, 257, -128, 127, "none"), (24, 8, 257, -128, 128, "none"), (24, 8, 320, 5, 261, "none"),
    (30, 9, 513, -100, -60, "none"), (12, 12, 700, -320, 161, "none")])
@pytest.mark.parametrize("kind,v", [("pcc1", 1.0), ("pccv", 2.0), ("pccv", 1.5)])
def test_one_lag_a_thread(fp, orc, launched, S, W, N, lag1, lag2, stack, kind, v):
    x = _records(S, W, N, S * N + W, "noise")
    y, names = launched(lambda: fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack, v=v))
    assert kind + "_direct" in names and kind + "_time" not in names
    yr = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True, v=v)
    _check(y, yr, N, lag1, lag2)


@pytest.mark.parametrize("what", ["event", "silent", "antiphase"])
@pytest.mark.parametrize("kind,v", [("pcc1", 1.0), ("pccv", 1.5)])
def test_records_one_lag_a_thread(fp, orc, launched, what, kind, v):
    S, W, N = 24, 6, 600
    x = _records(S, W, N, 7, what)
    y, names = launched(lambda: fp.allpairs(x, W, N, -100, 100, kind=kind, stack="none", v=v))
    assert kind + "_direct" in names
    yr = orc.allpairs(kind, x, W, N, -100, 100, stacked=False, f64=True, v=v)
    _check(y, yr, N, -100, 100, tol=TOL if what == "antiphase" else TOL_SHORT)  # as test_records_on_both_ways


@pytest.mark.parametrize("what", ["event", "silent", "antiphase"])
@pytest.mark.parametrize("kind,v", [("pcc1", 1.0), ("pccv", 1.5)])
def test_records_on_both_ways(fp, orc, what, kind, v):
    S, W, N = 4, 3, 1800
    x = _records(S, W, N, 7, what)
    y = fp.allpairs(x, W, N, -300, 300, kind=kind, stack="none", v=v)
    yr = orc.allpairs(kind, x, W, N, -300, 300, stacked=False, f64=True, v=v)
    # the FP32 transform's error is 3e-7 of the window's rms: half of a silent record holds
    # the Hilbert transform's tail of the other half, |z| about 0.05 of the rms, and the
    # event's window is noise of 0.05 of the rms too, so its phasors are off by 6e-6
    _check(y, yr, N, -300, 300, tol=TOL if what == "antiphase" else TOL_SHORT)


@pytest.mark.parametrize("stack", ["none", "plain"])
def test_workspace_without_the_split_scratch(fp, hip, stack):
    """A workspace that holds the phasors alone runs unsplit; sums in another order."""
    S, W, N = 3, 4, 1500
    x = _records(S, W, N, 3, "noise")
    job = api.make_job("pcc1", S, W, N, -200, 200, stack)
    lib, jp = _lib.lib(), ctypes.byref(job)
    total, need = lib.fpcc_workspace_size(jp), -(-S * W * N * 8 // 256) * 256
    assert total > need
    nout = lib.fpcc_output_len(jp)
    dx, dy, ws = hip.alloc(x.nbytes), hip.alloc(4 * nout), hip.alloc(total)
    hip.h2d(dx, x)

    def run(size):
        y = np.full(nout, np.nan, dtype=np.float32)
        hip.h2d(dy, y)
        r = lib.fpcc_allpairs_device(jp, ctypes.c_void_p(dx), ctypes.c_void_p(dy), ctypes.c_void_p(ws), size, None)
        hip.d2h(y, dy)
        return r, y

    (r0, full), (r1, small) = run(total), run(need)
    assert r0 == 0 and r1 == 0
    # FP64 sums of the same FP32 partial sums of at most 64 terms, cut at other samples
    assert np.abs(small - full).max() <= 2e-8
    assert run(need - 256)[0] == -1


def _phasors(x, W, N):
    """FP64 phasors [S][W][N] and a bound of the FP32 station stage's error in each: a window
    of any length takes up to four transforms of 2048 points and more, 2^-24 sqrt(log2 n)
    of the window's rms each, 4e-7 together, and no sample is off by more than three
    times that over |z|; 1e-7 for the half-angle phasor's rounding."""
    X = np.fft.fft(x.reshape(-1, W, N).astype(np.float64), axis=-1)
    k = np.arange(N)
    X[..., (k > 0) & (2 * k < N)] *= 2
    X[..., 2 * k > N] = 0
    z = np.fft.ifft(X, axis=-1)
    mag = np.abs(z)
    rms = np.sqrt((mag ** 2).mean(axis=-1, keepdims=True))
    return z / (mag + 1e-6 * mag.max(axis=-1, keepdims=True)), 1.2e-6 * rms / mag + 1e-7


@pytest.mark.parametrize("S,W,N,lag1,lag2,stack", [
    (3, 1, 100, 7, 40, "none"), (3, 2, 100, -99, 99, "plain"), (2, 1, 512, -256, 255, "none"),
    (2, 3, 1001, -300, 20, "none"), (4, 2, 777, 5, 520, "plain"), (2, 1, 9001, -3, 3, "none")])
@pytest.mark.parametrize("v", [-0.5, -1.5, 0.0])
def test_powers_that_are_not_positive(fp, orc, S, W, N, lag1, lag2, stack, v):
    """Terms of samples outside the windows would be infinite, and the terms inside grow
    without bound where two phasors are nearly equal or opposite."""
    x = _records(S, W, N, 3 * N + W, "noise")
    y = fp.allpairs(x, W, N, lag1, lag2, kind="pccv", stack=stack, v=v)
    yr = orc.allpairs("pccv", x, W, N, lag1, lag2, stacked=stack != "none", f64=True, v=v)
    assert np.isfinite(y).all()
    # first-order bound of a term's error: |v| r^(v-1) times the phasors' error e, and the
    # rounding of the terms and their sums (2^-21 of each); r kept from below by 2 e
    ph, er = _phasors(x, W, N)
    tol = np.zeros(y.shape).reshape(-1, W if stack == "none" else 1, y.shape[-1])
    for p, (i, j) in enumerate((i, j) for i in range(S) for j in range(i + 1, S)):
        for w in range(W):
            for l, lag in enumerate(range(lag1, lag2 + 1)):
                a, b = slice(max(0, lag), min(N, N + lag)), slice(max(0, -lag), min(N, N - lag))
                e = er[j, w, a] + er[i, w, b]
                for r in (np.abs(ph[j, w, a] + ph[i, w, b]), np.abs(ph[j, w, a] - ph[i, w, b])):
                    r = np.maximum(r - e, e)
                    t = (abs(v) * r ** (v - 1) * e + 2.0 ** -21 * r ** v).sum() / (2 ** (v / 2) * (N - abs(lag)))
                    tol[p, w if stack == "none" else 0, l] += t if stack == "none" else t / W
    err = np.abs(y - yr).reshape(tol.shape)
    print(f"v {v} N {N}: max|gpu-fp64| {err.max():.2e}, at most {(err / tol).max():.2f} of the bound", flush=True)
    assert (err <= tol).all()


def test_equal_and_opposite_records_at_a_negative_power(fp, orc):
    """0^v: the terms of equal records at lag 0 are -inf, of opposite ones +inf."""
    W, N, v = 2, 333, -0.5
    x = _records(3, W, N, 5, "noise")
    x[1], x[2] = x[0], -x[0]
    for stack in ("none", "plain"):
        y = fp.allpairs(x, W, N, -4, 4, kind="pccv", stack=stack, v=v)
        yr = orc.allpairs("pccv", x, W, N, -4, 4, stacked=stack != "none", f64=True, v=v)
        inf = np.isinf(yr)
        assert inf.any() and (np.isinf(y) == inf).all() and (y[inf] == yr[inf]).all()
        assert np.isfinite(y[~inf]).all()


def test_host_entry_at_a_negative_power(fp):
    """pcc_set runs the same kernels."""
    W, N, v = 3, 450, -1.0
    x = _records(2, W, N, 9, "noise")
    y = fp.pcc_set(*x.reshape(2, W, N), v, -30, 200)
    assert np.isfinite(y).all()
    assert np.array_equal(y, fp.allpairs(x, W, N, -30, 200, kind="pccv", stack="none", v=v)[0])


# more than 2^32 threads: the rows of one launch at a time
@pytest.mark.parametrize("kind,lag1,lag2", [("pcc1", 0, 0), ("pccv", -2, 1)])
def test_more_rows_than_one_launch(fp, kind, lag1, lag2):
    S, W, N = 2000, 10, 8
    x = np.random.default_rng(2).standard_normal((S, W * N)).astype(np.float32)
    y = fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack="none", v=1.5)
    # the pairs of the first three and of the last four stations
    first = fp.allpairs(x[:3], W, N, lag1, lag2, kind=kind, stack="none", v=1.5)
    last = fp.allpairs(x[-4:], W, N, lag1, lag2, kind=kind, stack="none", v=1.5)
    tol = 2.0 ** -22  # FP32 terms summed in another order
    assert np.abs(y[[0, 1, S - 1]] - first).max() <= tol and np.abs(y[-6:] - last).max() <= tol
    # every row is written: a correlation of 6 and more noise samples is not exactly 0
    assert (np.abs(y).max(axis=-1) > 0).all()

