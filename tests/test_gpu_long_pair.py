"""Pair stage of long windows (one kernel from the spectra to the few outputs the lag
window reads) at its edges: each row length, the smallest and largest lag windows it
takes and the first it leaves to the two-pass inverse, one-sided windows, each source
(spectra of phasors, of real signals, Gram rows) and the sums over windows.  Every case
holds the pairs that the kernel asks for (items x units of 8 row pairs: 2 at 2^14, 4 at
2^15, .. 16 at 2^17, 32 at 2^18, 64 at 2^19; 128, or 512 where windows are summed) and says
which way it takes."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu
# FP32 transforms of 2^14 .. 2^19 points: each value carries about log2(n) roundings of
# 2^-24 of the transform's rms, and correlations are normalised to full scale 1: 1e-6
TOL = 1e-6
LONG, PASSES = "pair_long", {"pair_cross_rows", "pair_inv_rows"}


def _case(fp, orc, launched, kind, stack, S, W, N, lag1, lag2, long_=True, tol=TOL, **kw):
    x, _ = synth.make_stations(S, W * N, 100, seed=N % 1000 + S)
    y, names = launched(lambda: fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack, **kw))
    assert (LONG in names) == long_ and bool(PASSES & names) != long_
    yr = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True, **kw)
    err = np.abs(y - yr).max()
    print(f"{kind}/{stack} S={S} W={W} N={N} lags {lag1}..{lag2}: max|gpu-fp64| {err:.2e}", flush=True)
    assert y.shape == yr.shape and err <= tol


# row lengths 512 (2^14 .. 2^17), 1024 (2^18), 2048 (2^19); outputs at n1 = 0, -1, +-12 H, and
# each bound of the kept sums (2048, 4096 and 6144 lags)
@pytest.mark.parametrize("S,N,lag1,lag2", [
    (12, 10000, 0, 0), (12, 10000, -1, 1), (12, 9001, -6144, 6143), (12, 10000, 6000, 6143), (12, 10000, -6144, -6100),
    (9, 24000, -511, 512), (9, 24000, -4096, 4095), (7, 50000, -512, 511), (5, 120000, -2048, 2047),
    (4, 200000, -1024, 1023), (4, 200000, -4096, 4095), (4, 200000, -6144, 6143), (3, 300000, -2048, 2047),
    (3, 300000, -4096, 4095), (3, 300000, -6144, 6143)])
def test_pcc2_lag_windows(fp, orc, launched, S, N, lag1, lag2):
    _case(fp, orc, launched, "pcc2", "plain", S, 1, N, lag1, lag2)


# past the widest lag window, and one pair short of the work it asks for
@pytest.mark.parametrize("S,W,N,lag1,lag2", [(12, 1, 9001, -6145, 6144), (11, 1, 10000, -100, 100),
                                             (23, 2, 10000, -100, 100)])
def test_left_to_two_passes(fp, orc, launched, S, W, N, lag1, lag2):
    _case(fp, orc, launched, "pcc2", "plain", S, W, N, lag1, lag2, long_=False)


@pytest.mark.parametrize("kind", ["pcc2", "gncc", "cc1b"])
@pytest.mark.parametrize("stack,S,W", [("none", 8, 3), ("plain", 24, 3)])
@pytest.mark.parametrize("lag1,lag2", [(-700, 1500), (-3000, 4000), (-6000, 100)])
def test_kinds_and_windows(fp, orc, launched, kind, stack, S, W, lag1, lag2):
    _case(fp, orc, launched, kind, stack, S, W, 9000, lag1, lag2)


# rows of 1024 and 2048 bins, windows summed, each bound of the kept sums
@pytest.mark.parametrize("kind", ["pcc2", "gncc", "cc1b"])
@pytest.mark.parametrize("S,W,N,lag1,lag2", [(7, 2, 150000, -900, 900), (7, 2, 150000, -300, 4000),
                                             (7, 2, 150000, -6000, 6000), (5, 2, 300000, -1500, 1500),
                                             (5, 2, 300000, -4000, 300), (5, 2, 300000, -6000, 6000)])
def test_longer_rows(fp, orc, launched, kind, S, W, N, lag1, lag2):
    _case(fp, orc, launched, kind, "plain", S, W, N, lag1, lag2)


@pytest.mark.parametrize("kind,stack", [("pcc2", "gram"), ("pcc2", "gram16"), ("cc1b", "gram")])
@pytest.mark.parametrize("S,W,N,lag1,lag2", [
    (12, 4, 9000, -300, 900), (12, 4, 9000, -3000, 900), (12, 4, 9000, -6144, 6143), (4, 2, 150000, -900, 900),
    (4, 2, 150000, -4000, 4000), (4, 2, 150000, -6000, 6000), (3, 2, 300000, -1500, 1500), (3, 2, 300000, -4000, 300),
    (3, 2, 300000, -6000, 6000)])
def test_gram_rows(fp, orc, launched, kind, stack, S, W, N, lag1, lag2):
    _case(fp, orc, launched, kind, stack, S, W, N, lag1, lag2)


def test_many_items_share_less(fp, orc, launched):
    """2640 pair-windows, more than 2048: a workgroup takes both units of its row pairs."""
    _case(fp, orc, launched, "pcc2", "none", 12, 40, 12000, -100, 100)


# every lag of the window: those of short overlap are exact sums over the record's ends,
# normalised like the others (1-bit values are multiples of 1/overlap)
@pytest.mark.parametrize("W", [1, 3])
@pytest.mark.parametrize("stack", ["gram", "gram16"])
def test_gram_rows_to_the_last_lag(fp, orc, launched, stack, W):
    _case(fp, orc, launched, "cc1b", stack, 12, W, 5000, -4990, 4990)


@pytest.mark.parametrize("kind,stack,S,W", [("cc1b", "none", 12, 1), ("cc1b", "plain", 24, 2), ("gncc", "none", 12, 1),
                                            ("gncc", "plain", 12, 2)])
def test_real_spectra_to_the_last_lag(fp, orc, launched, kind, stack, S, W):
    _case(fp, orc, launched, kind, stack, S, W, 5000, -4990, 4990, tol=TOL if kind == "cc1b" else 1e-5)


def test_wavelet_rows(fp, orc, launched):
    """Wavelet PCC's Gram rows, 10 pairs of 2^17 points."""
    S, N, kw = 5, 66000, dict(pmin=4.0, pmax=16.0, V=2)
    x, _ = synth.make_stations(S, N, 50, seed=3)
    y, names = launched(lambda: fp.allpairs(x, 1, N, -300, 300, kind="wpcc", stack="plain", **kw))
    assert "wpcc_pair_long" in names
    yr = orc.allpairs("wpcc", x, 1, N, -300, 300, stacked=True, f64=True, **kw)
    assert np.abs(y - yr[..., : y.shape[-1]]).max() <= TOL
