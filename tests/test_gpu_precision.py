"""Errors against 64 bits that the FP32 stages are built to keep: 2-norm of the difference
over 2-norm of the result, on records of noise with a common source."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu


def _error(fp, orc, kind, stack, S, W, N, lag1, lag2, x=None, **kw):
    if x is None:
        x, _ = synth.make_stations(S, W * N, 100, seed=N + S)
    y = fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack, **kw).astype(np.float64)
    r = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True, **kw)
    e = float(np.linalg.norm(y - r) / np.linalg.norm(r))
    print(f"{kind}/{stack} S={S} W={W} N={N}: {e:.2e}", flush=True)
    return e


@pytest.mark.parametrize("N", [450, 900, 1800, 3600])
def test_mean_of_many_windows(fp, orc, N):
    """One source in every window: its spectra add up coherently, and a sum of 2000 of them
    in FP32 would be off by 2^-25 sqrt(2000 / 3) = 8e-7 of itself; in FP64 what is left is
    the inverse of nearly one value, under 2^-24."""
    W = 2000
    x = np.repeat(np.random.default_rng(N).standard_normal(W * N).astype(np.float32)[None], 2, axis=0)
    x[1] += 0.3 * np.random.default_rng(1).standard_normal(W * N).astype(np.float32)
    assert _error(fp, orc, "cc1b", "plain", 2, W, N, -50, 50, x=x) <= 2.0 ** -24


# limits between the two ways' errors on these records: 2.3 .. 3.9e-7 with the window as
# real part, 2.9 .. 4.9e-7 with the transforms' (each about 0.78 of the other)
@pytest.mark.parametrize("kind,stack,N,limit", [
    ("pcc2", "none", 3600, 4.4e-7), ("pcc2", "plain", 3600, 2.6e-7), ("pcc2", "plain", 1800, 2.55e-7),
    ("pcc2", "plain", 900, 3.0e-7), ("pcc1", "none", 1500, 3.8e-7), ("pccv", "none", 1500, 3.6e-7)])
def test_real_part_of_the_analytic_signal(fp, orc, kind, stack, N, limit):
    """The window itself, so that the transforms' error moves a phasor through the Hilbert
    transform alone and not through both components."""
    W = 12
    kw = dict(v=1.5) if kind == "pccv" else {}
    rng = np.random.default_rng(N)
    src = rng.standard_normal(W * N + 64)
    x = rng.standard_normal((8, W * N))
    for s in range(8):
        x[s] += 0.5 * src[8 * s:8 * s + W * N]
    assert _error(fp, orc, kind, stack, 8, W, N, -200, 200, x=x.astype(np.float32), **kw) <= limit


# limits between the errors with twiddles formed in FP64 (1.7 .. 2.4e-7 on these records) and
# in FP32 (2.0 .. 2.6e-7)
@pytest.mark.parametrize("kind,stack,S,W,N,limit", [
    ("cc1b", "plain", 6, 1, 86400, 2.0e-7), ("gncc", "plain", 6, 1, 86400, 1.85e-7),
    ("gncc", "none", 8, 6, 12000, 2.53e-7), ("cc1b", "gram", 12, 3, 12000, 2.18e-7)])
def test_long_pair_stage(fp, orc, launched, kind, stack, S, W, N, limit):
    e, names = launched(lambda: _error(fp, orc, kind, stack, S, W, N, -2000, 2000))
    assert "pair_long" in names and e <= limit
