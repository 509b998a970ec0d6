"""WPCC where the scales' column passes keep their columns in registers (zero-pad lengths
2^17 and 2^18, columns of 256 points), one and several windows, against the FP64 oracle."""
import numpy as np
import pytest

from fastpcc_amd import synth

pytestmark = pytest.mark.gpu
# FP32 transforms of 2^17 .. 2^18 points and AmpNorm phasors of every scale: 2e-7 of full
# scale at these lengths in the other WPCC tests, five times that here
TOL = 1e-6


@pytest.mark.parametrize("S,W,N,stack", [(2, 1, 66000, "none"), (3, 1, 100000, "plain"), (2, 2, 70000, "none"),
                                         (2, 1, 140000, "plain")])
def test_scales_in_registers(fp, orc, S, W, N, stack):
    x, _ = synth.make_stations(S, W * N, 50, seed=N % 997)
    kw = dict(pmin=4.0, pmax=16.0, V=2)
    y = fp.allpairs(x, W, N, -300, 300, kind="wpcc", stack=stack, **kw)
    yr = orc.allpairs("wpcc", x, W, N, -300, 300, stacked=stack != "none", f64=True, **kw)
    yr = yr[..., : y.shape[-1]]
    err = np.abs(y[..., : yr.shape[-1]] - yr).max()
    print(f"wpcc/{stack} S={S} W={W} N={N}: max|gpu-fp64| {err:.2e}", flush=True)
    assert err <= TOL


def test_silent_window(fp):
    """A silent record's scales have no phase: zero correlations, no NaN."""
    x, _ = synth.make_stations(3, 66000, 50, seed=1)
    x[1] = 0
    y = fp.allpairs(x, 1, 66000, -20, 20, kind="wpcc", stack="plain", pmin=4.0, pmax=16.0, V=2)
    assert np.isfinite(y).all() and not y[0].any() and not y[2].any() and y[1].any()
