"""Fits that sort by length of themselves (fused fits of ragged batches above one
wave per SIMD) against the fit in input order and the explicit sort."""
import numpy as np
import pytest

from gpukalmanfitter_amd import configs
from gpukalmanfitter_amd import generate as G
from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,n", [(3, 65535), (3, 65537), (3, 66561), (5, 67000)])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_ragged_batch_in_input_order_equals_the_sorted_one(cfg, n, precision):
    """One wave per SIMD is 65,536 tracks; 1,024 tracks are a block of the sort.
    Every schedule gives the same bits."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    b = G.generate(cfg, n_tracks=n)
    kf = KalmanFitter(b.planes, b.field)
    dev = DeviceBatch(b)
    opts = KalmanFitterOptions(**dict(configs.WORKLOAD_FIT_OPTIONS, precision=precision))
    kf.fit_batch_noalloc(dev, opts)  # always in input order
    want = dev.results_numpy()
    for sched in ({}, dict(sort_by_length=1)):
        kf.set_schedule(**sched)
        dev.clear_results()
        kf.fit_batch(dev, opts)
        got = dev.results_numpy()
        for k in got:
            assert np.array_equal(got[k], want[k]), (k, sched)
    kf.close()
