"""How many tracks the fused fit leaves to the RTS program, on the CPU build of both."""
import dataclasses

import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

from test_fused_fit import fused_fit, turned
from test_host_fit import host_fit

W = configs.WORKLOAD_FIT_OPTIONS
PRECISIONS = [abi.KF_PRECISION_FP64, abi.KF_PRECISION_MIXED]


@pytest.mark.parametrize("precision", PRECISIONS)
def test_a_weak_prior_hands_nothing_back(built, precision):
    """Start errors of a radian: the filtered angles are tight from the second
    plane on, and facing +x no smoothed angle is near its bound.  The bars are
    the modes' own times the posterior's 1e4 loss of digits against that prior
    (1 rad and 100 mm against 0.3 mrad and 50 um, squared, in FP64), and the
    start's position and angles decide nothing discrete."""
    b = G.generate(1, n_tracks=400)
    b = dataclasses.replace(b, start_cov=b.start_cov * 1e6)
    opt = abi.default_options(precision=precision, **W)
    f, r = fused_fit(b, opt), host_fit(b, opt)
    assert not f["redo"].any()
    assert np.array_equal(f["status"], r["status"])
    if precision == abi.KF_PRECISION_FP64:
        sig = np.sqrt(np.abs(r["cov"][abi.DIAG_INDEX]))
        assert (np.abs(f["params"] - r["params"])
                <= 1e-7 * np.maximum(np.abs(r["params"]), sig)).all()


@pytest.mark.parametrize("precision", PRECISIONS)
def test_facing_the_wrap(built, precision):
    """Tracks around phi = pi: one state's distance from the wrap counts against
    that state's error and the chi2 still to come, not the largest error of the
    track against all of its chi2 (8.0 % then)."""
    b = turned(G.generate(1, n_tracks=2000), np.pi)
    f = fused_fit(b, abi.default_options(precision=precision, **W))
    assert 0.0 < (f["redo"] != 0).mean() < 0.06
