"""Track-state records at the edges of the copy kernel's blocks (64 tracks, one
state slot, half of the fields each)."""
import numpy as np
import pytest

from gpukalmanfitter_amd import configs
from gpukalmanfitter_amd import generate as G

pytestmark = pytest.mark.gpu

W = configs.WORKLOAD_FIT_OPTIONS


@pytest.mark.parametrize("n", [1, 63, 64, 65, 129])
@pytest.mark.parametrize("sort", [0, 1])
def test_records_of_a_batch_equal_those_of_its_tracks_in_a_larger_one(n, sort):
    """The records of the first n tracks are the same bits whatever the batch
    and the order it runs in; slots past a track's measured states are not
    written."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = G.generate(3, n_tracks=200)
    kf = KalmanFitter(b.planes, b.field)
    opts = KalmanFitterOptions(**W)
    whole = DeviceBatch(b, track_states=True)
    kf.fit_batch(whole, opts)
    ref = whole.results_numpy()
    kf.set_schedule(sort_by_length=sort)
    dev = DeviceBatch(b.subset(np.arange(n)), track_states=True, max_states=b.max_states)
    dev.out["track_states"].fill_(7.0)
    kf.fit_batch(dev, opts)
    got = dev.results_numpy()
    kf.close()
    nm = got["n_measured"]
    assert np.array_equal(nm, ref["n_measured"][:n])
    written = np.arange(b.max_states)[:, None] < nm[None, :]
    for f in range(got["track_states"].shape[1]):
        want = np.where(written, ref["track_states"][:, f, :n], 7.0)
        assert np.array_equal(got["track_states"][:, f], want), f
