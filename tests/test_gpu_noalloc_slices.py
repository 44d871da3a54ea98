"""The fused fit in the fixed workspace, in more than one slice."""
import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

from test_fused_fit import turned


@pytest.mark.gpu
def test_gpu_noalloc_fused_slices(built):
    """1,300,000 FP64 tracks keep 281 MB of first states, the workspace holds 256 MB:
    two slices at least, with tracks of every kind in both (facing phi = pi, some
    without time variance); the bits of the fit in one piece, twice."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = turned(G.generate(1, n_tracks=1300000), np.pi)
    b.start_cov[20, ::1000] = 0.0
    opts = KalmanFitterOptions(**dict(configs.WORKLOAD_FIT_OPTIONS, max_rk_trials=20))
    kf = KalmanFitter(b.planes, b.field)
    dev = DeviceBatch(b)
    kf.fit_batch(dev, opts)
    want = dev.results_numpy()
    for _ in range(2):
        dev.clear_results()
        kf.fit_batch_noalloc(dev, opts)
        got = dev.results_numpy()
        for k in ("params", "cov", "chi2", "ndf", "n_measured", "status"):
            assert np.array_equal(got[k], want[k], equal_nan=True), k
    kf.close()
    assert ((want["status"] & abi.KF_STATUS_OK) != 0).mean() > 0.9
