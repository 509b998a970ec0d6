"""Pair stages of Nz 512 .. 8192 on compile-time inverses: every length, numbers of
transforms that leave a workgroup partly empty, few pairs with many windows (split over
the chip) and one window, full lag ranges (exact short overlaps of 1-bit), each source."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu
# FP32 transforms of at most 8192 points: about log2(n) roundings of 2^-24 of full scale;
# at short overlaps 1-bit sums are exact and PCC2's divisor stays N
TOL = 1e-6


def _check(fp, orc, kind, stack, S, W, N, lag1, lag2):
    x, _ = synth.make_stations(S, W * N, 20, seed=S * 100 + N)
    y = fp.allpairs(x, W, N, lag1, lag2, kind=kind, stack=stack)
    yr = orc.allpairs(kind, x, W, N, lag1, lag2, stacked=stack != "none", f64=True)
    err = np.abs(y - yr).max()
    print(f"{kind}/{stack} S={S} W={W} N={N} lags {lag1}..{lag2}: max|gpu-fp64| {err:.2e}", flush=True)
    assert y.shape == yr.shape and err <= TOL


# zero-pad lengths 512, 1024, 2048, 4096, 8192 (and 256 on the runtime plan); 3, 10 and 21
# pairs leave workgroups of 8, 4 and 2 transforms partly empty
@pytest.mark.parametrize("N,lag", [(200, 50), (400, 100), (700, 300), (1500, 500), (2500, 1500), (4096, 4000)])
@pytest.mark.parametrize("S,W", [(3, 1), (5, 3), (7, 2)])
@pytest.mark.parametrize("kind", ["pcc2", "cc1b"])
@pytest.mark.parametrize("stack", ["none", "plain"])
def test_lengths(fp, orc, kind, stack, S, W, N, lag):
    _check(fp, orc, kind, stack, S, W, N, -lag, lag)


@pytest.mark.parametrize("N", [360, 900, 1800])
@pytest.mark.parametrize("kind,stack", [("cc1b", "none"), ("cc1b", "plain"), ("cc1b", "gram"), ("pcc2", "plain"),
                                        ("pcc2", "gram"), ("pcc2", "gram16")])
def test_every_lag(fp, orc, kind, stack, N):
    _check(fp, orc, kind, stack, 4, 4, N, -(N - 1), N - 1)


@pytest.mark.parametrize("S,W", [(2, 31), (3, 40), (24, 2), (40, 3)])
@pytest.mark.parametrize("stack", ["none", "plain", "zsum"])
def test_windows_over_the_chip(fp, orc, S, W, stack):
    """Nz 8192: one pair's windows in as many units as there are, and more pairs than run at once."""
    _check(fp, orc, "pcc2", stack, S, W, 2100, -700, 20)


def test_one_sided(fp, orc):
    _check(fp, orc, "pcc2", "none", 5, 2, 1500, 37, 38)
    _check(fp, orc, "cc1b", "plain", 5, 2, 1500, -1400, -1399)


@pytest.mark.parametrize("kind", ["pcc2", "gncc", "cc1b"])
def test_more_pair_windows_than_one_launch(fp, kind):
    """20 million pair-windows, a workgroup of 512 threads each: more than 2^32 threads."""
    S, W, N = 2000, 10, 8
    x = np.random.default_rng(2).standard_normal((S, W * N)).astype(np.float32)
    y = fp.allpairs(x, W, N, -1, 2, kind=kind, stack="none")
    first, last = (fp.allpairs(v, W, N, -1, 2, kind=kind, stack="none") for v in (x[:3], x[-4:]))
    assert np.array_equal(y[[0, 1, S - 1]], first) and np.array_equal(y[-6:], last)
    if kind != "cc1b":  # 6 and more samples of noise: never 0 at every lag
        assert (np.abs(y).max(axis=-1) > 0).all()


@pytest.mark.parametrize("kind,stacks", [("pcc2", ("plain", "zsum", "gram", "gram16")), ("cc1b", ("plain", "gram", "gram16")),
                                         ("gncc", ("plain",))])
@pytest.mark.parametrize("S,W,N,lag", [(7, 5, 3600, 800), (40, 24, 1200, 300), (5, 3, 200, 60), (12, 4, 12000, 900)])
def test_stacks_against_the_mean_of_the_windows(fp, kind, stacks, S, W, N, lag):
    """The means are formed from summed spectra; every window inverted on its own and averaged
    in FP64 is the same by linearity (each within 5e-7 of 64 bits, 2e-7 rms of full scale 1)."""
    x, _ = synth.make_stations(S, W * N, 50, seed=N)
    mean = fp.allpairs(x, W, N, -lag, lag, kind=kind, stack="none").astype(np.float64).mean(axis=1)
    for stack in stacks:
        y = fp.allpairs(x, W, N, -lag, lag, kind=kind, stack=stack)
        assert np.abs(y - mean).max() <= 1e-6, stack
