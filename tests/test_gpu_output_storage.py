"""DeviceBatch.results_numpy reads the storage that the fit wrote."""
import numpy as np
import pytest

from gpukalmanfitter_amd import configs
from gpukalmanfitter_amd import generate as G


@pytest.mark.gpu
@pytest.mark.parametrize("how", ["tensor", "storage", "added", "shorter"])
def test_gpu_replaced_outputs_are_read(how):
    """A caller puts its own tensor, or its own storage under the old one, in the place
    of an output: the fit writes there, and that is what comes back."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = G.generate(1, n_tracks=100)
    kf = KalmanFitter(b.planes, b.field)
    opts = KalmanFitterOptions(**configs.WORKLOAD_FIT_OPTIONS)
    want = DeviceBatch(b)
    kf.fit_batch(want, opts)
    want = want.results_numpy()
    dev = DeviceBatch(b)
    own = torch.full((100,), -1.0, dtype=torch.float64, device=dev.device)
    if how == "tensor":
        dev.out["chi2"] = own
    elif how == "storage":
        dev.out["chi2"].data = own
    elif how == "added":
        dev.out["chi2"] = dev.out["chi2"].clone()
    else:
        dev.out["ndf"] = torch.zeros(128, dtype=torch.int32, device=dev.device)
    kf.fit_batch(dev, opts)
    got = dev.results_numpy()
    kf.close()
    for k in want:
        assert np.array_equal(got[k][..., :100], want[k]), k
