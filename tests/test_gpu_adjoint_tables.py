"""The chi2 gradient with plane tables at and beyond what its kernels keep in LDS: the
sweep's limit (148 planes in a constant field, 47 in a grid), and the forward
pass's (256)."""
import dataclasses

import numpy as np
import pytest

from gpukalmanfitter_amd import configs
from gpukalmanfitter_amd import generate as G
from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions

from test_gpu_parity import _padded_planes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,planes", [(4, 148), (4, 149), (4, 257), (3, 47), (3, 48), (3, 257),
                                        (5, 47), (5, 48), (5, 257)])
def test_gradient_does_not_depend_on_unused_planes(cfg, planes):
    """Against the table without them (10, 30 and 40 planes, in LDS): the builds
    differ in how they contract, 1e-13 per gradient, so 1e-10 of the largest of
    each kind; unused planes have none."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    b = G.generate(cfg, n_tracks=700)
    n = len(b.planes)
    bp = dataclasses.replace(b, planes=_padded_planes(b.planes, planes - n))
    res = []
    for x in (b, bp):
        kf = KalmanFitter(x.planes, x.field)
        res.append(kf.chi2_gradient(DeviceBatch(x), KalmanFitterOptions(
            **configs.WORKLOAD_FIT_OPTIONS)))
        kf.close()
    (g, s, c, f, r), (gp, sp, cp, fp, rp) = res
    assert np.array_equal(f, fp) and (f == 0).any()
    assert abs(cp - c) <= 1e-12 * abs(c) and abs(sp - s) <= 1e-10 * abs(s)
    for got, want in ((gp, g), (rp, r)):  # shifts and centre, rotations and frame
        for kind in (slice(0, 3), slice(3, None)):
            dev = np.abs(got[:n, kind] - want[:, kind]).max()
            assert dev <= 1e-10 * np.abs(want[:, kind]).max(), dev
    assert not gp[n:].any() and not rp[n:].any()
