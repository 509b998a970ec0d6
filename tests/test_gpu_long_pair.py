"""Pair stage of long windows (one kernel from the spectra to the few outputs the lag
window reads) at its edges: each row length, the smallest and largest lag windows it
takes and the first it leaves to the two-pass inverse, one-sided windows, each source
(spectra of phasors, of real signals, Gram rows) and the sums over windows."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu
# FP32 transforms of 2^14 .. 2^19 points: each value carries about log2(n) roundings of
# 2^-24 of the transform's rms, and correlations are normalised to full scale 1: 1e-6
TOL = 1e-6


def _case(fp, orc, kind, stack, S, W, N, lag1, lag2, **kw):
    x, _ = synth.make_stations(S, W * N, 100, seed=N % 1000 + S)
    y = fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack, **kw)
    yr = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True, **kw)
    err = np.abs(y - yr).max()
    print(f"{kind}/{stack} S={S} W={W} N={N} lags {lag1}..{lag2}: max|gpu-fp64| {err:.2e}", flush=True)
    assert y.shape == yr.shape and err <= TOL


# row lengths 512 (2^14 .. 2^17), 1024 (2^18), 2048 (2^19); outputs at n1 = 0, -1, +-12 H
@pytest.mark.parametrize("N,lag1,lag2", [
    (10000, 0, 0), (10000, -1, 1), (9001, -6144, 6143), (9001, -6145, 6144), (10000, 6000, 6143), (10000, -6144, -6100),
    (24000, -511, 512), (50000, -512, 511), (120000, -2048, 2047), (200000, -1024, 1023), (200000, -6144, 6143),
    (300000, -2048, 2048)])
def test_pcc2_lag_windows(fp, orc, N, lag1, lag2):
    _case(fp, orc, "pcc2", "plain", 3, 1, N, lag1, lag2)


@pytest.mark.parametrize("kind", ["pcc2", "gncc", "cc1b"])
@pytest.mark.parametrize("stack", ["none", "plain"])
def test_kinds_and_windows(fp, orc, kind, stack):
    _case(fp, orc, kind, stack, 4, 3, 9000, -700, 1500)


@pytest.mark.parametrize("kind,stack", [("pcc2", "gram"), ("pcc2", "gram16"), ("cc1b", "gram")])
@pytest.mark.parametrize("lag1,lag2", [(-300, 900), (-6144, 6143)])
def test_gram_rows(fp, orc, kind, stack, lag1, lag2):
    _case(fp, orc, kind, stack, 5, 4, 9000, lag1, lag2)


def test_many_items_share_less(fp, orc):
    """Enough pair-windows that a workgroup takes several units of row pairs."""
    _case(fp, orc, "pcc2", "none", 12, 20, 12000, -100, 100)


# every lag of the window: those of short overlap are exact sums over the record's ends,
# normalised like the others (1-bit values are multiples of 1/overlap)
@pytest.mark.parametrize("W", [1, 3])
@pytest.mark.parametrize("stack", ["gram", "gram16"])
def test_gram_rows_to_the_last_lag(fp, orc, stack, W):
    _case(fp, orc, "cc1b", stack, 12, W, 5000, -4990, 4990)
