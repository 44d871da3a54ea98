"""The mixed fused program built for one field kind, as the kernels have it, against
the oracle (on the CPU)."""
import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

import oracle
from parity import compare_fit
from test_step_forms import fit_kind


@pytest.mark.parametrize("cfg,kind", [(1, 0), (1, 1), (3, 0), (3, 2), (5, 0), (5, 2)])
def test_mixed_build_of_one_field_kind(built, cfg, kind):
    """The mode's bars: 1e-5 of an error, 1e-3 of a covariance."""
    b = G.generate(cfg, n_tracks=300)
    opt = abi.default_options(precision=abi.KF_PRECISION_MIXED, **configs.WORKLOAD_FIT_OPTIONS)
    f = fit_kind(b, opt, kind)
    o, _, _, _ = oracle.fit(b, abi.default_options(**configs.WORKLOAD_FIT_OPTIONS))
    assert not f["redo"].any()
    assert np.array_equal(f["n_measured"], o.n_measured)
    assert np.array_equal(f["status"], o.status)
    pd, cd, _ = compare_fit(f, o)
    assert pd <= 1e-5 and cd <= 1e-3, (pd, cd)
