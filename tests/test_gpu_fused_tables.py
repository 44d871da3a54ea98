"""Plane tables at the edge of what the fused kernel keeps in LDS beside its sums
(224 planes in FP64, 112 in the mixed mode)."""
import dataclasses
from types import SimpleNamespace

import numpy as np
import pytest

from gpukalmanfitter_amd import configs
from gpukalmanfitter_amd import generate as G
from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions

from parity import compare_fit
from test_gpu_parity import _padded_planes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision,planes", [("fp64", 224), ("fp64", 225), ("mixed", 112),
                                              ("mixed", 113)])
@pytest.mark.parametrize("cfg", [1, 5])
def test_table_at_the_lds_limit(cfg, precision, planes):
    """The fit does not depend on planes no sequence uses: to rounding in FP64
    (1e-10 between two builds), within twice the mixed mode's bars (1e-5, 1e-3)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    b = G.generate(cfg, n_tracks=300)
    bp = dataclasses.replace(b, planes=_padded_planes(b.planes, planes - len(b.planes)))
    res = []
    for x in (b, bp):
        kf = KalmanFitter(x.planes, x.field)
        dev = DeviceBatch(x)
        kf.fit_batch(dev, KalmanFitterOptions(**dict(configs.WORKLOAD_FIT_OPTIONS,
                                                     precision=precision)))
        res.append(dev.results_numpy())
        kf.close()
    assert np.array_equal(res[0]["status"], res[1]["status"])
    pd, cd, _ = compare_fit(res[1], SimpleNamespace(**{k: res[0][k] for k in
                                                       ("status", "params", "cov", "chi2")}))
    if precision == "fp64":
        assert max(pd, cd) <= 1e-10, (pd, cd)
    else:
        assert pd <= 2e-5 and cd <= 2e-3, (pd, cd)
