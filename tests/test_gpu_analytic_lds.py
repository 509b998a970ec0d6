"""Station stage of long windows: analytic signals in one workgroup's LDS at the edges
of its range (every radix, its smallest and largest lengths, the first lengths past
it, rows that start on odd samples, special windows), and the column passes of each
compile-time length, Bluestein's middle pass included."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu
TOL = 1e-6  # FP32 transforms of 2^14 .. 2^18 points on unit phasors (about log2(n) 2^-24 of the rms)


def _pcc2(fp, orc, x, W, N, lag=60, stack="none"):
    y = fp.allpairs(x, W, N, -lag, lag, kind="pcc2", stack=stack)
    yr = orc.allpairs("pcc2", x[:, : W * N], W, N, -lag, lag, stacked=stack != "none", f64=True)
    err = np.abs(y - yr).max()
    print(f"N={N} W={W}: max|gpu-fp64| {err:.2e}", flush=True)
    assert np.isfinite(y).all() and err <= TOL


# halves 8 x 8 x .., 3^8, 5^6, 7^5, 2^14, the largest with a plan and the next above it
@pytest.mark.parametrize("N", [8194 + 6, 8232, 13122, 31250, 33614, 32768, 38400, 38416, 38880])
@pytest.mark.parametrize("odd_stride", [0, 1])
def test_lengths(fp, orc, N, odd_stride):
    W = 2
    x, _ = synth.make_stations(3, W * N + odd_stride, 50, seed=N)
    _pcc2(fp, orc, x, W, N)


# Nz > 8192 with a window under 8192, and lengths of every column pass through Bluestein
# (grids 2^14 .. 2^17: columns of 32, 64, 128, 256 points)
@pytest.mark.parametrize("N", [8000, 5003, 9001, 20011, 40009])
def test_other_routes(fp, orc, N):
    lag = 400 if N == 8000 else 60
    x, _ = synth.make_stations(3, N, 50, seed=N)
    _pcc2(fp, orc, x, 1, N, lag=lag)


def test_special_windows(fp, orc):
    """A silent window correlates to zero, a constant one has phasors +-1, and the
    alternating one's analytic signal is itself."""
    N = 9000
    x = np.ones((4, N), dtype=np.float32)
    x[0] = 0
    x[1] = 3.0
    x[2] = -0.5
    x[3] = 2.0 * (-1.0) ** np.arange(N)
    y = fp.allpairs(x, 1, N, -4, 4, kind="pcc2", stack="none")[:, 0]
    yr = orc.allpairs("pcc2", x, 1, N, -4, 4, stacked=False, f64=True)[:, 0]
    assert not y[:3].any()
    assert np.abs(y - yr).max() <= 2e-6  # the regulariser's 1e-6 and the transforms


@pytest.mark.parametrize("N", [14000, 20000, 40000, 100000])
@pytest.mark.parametrize("kind", ["gncc", "cc1b"])
def test_real_kinds_through_each_column_length(fp, orc, kind, N):
    x, _ = synth.make_stations(3, N, 50, seed=N)
    y = fp.allpairs(x, 1, N, -200, 200, kind=kind, stack="none")
    yr = orc.allpairs(kind, x, 1, N, -200, 200, stacked=False, f64=True)
    err = np.abs(y - yr).max()
    print(f"{kind} N={N}: max|gpu-fp64| {err:.2e}", flush=True)
    assert err <= TOL
