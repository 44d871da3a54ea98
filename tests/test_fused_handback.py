"""How many tracks the fused fit leaves to the RTS program, on the CPU build of both."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

import oracle
from test_adjoint_cpu import field_of
from test_fused_fit import fused_fit, fused_lib, turned
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


def near_wrap(b, opt):
    lib = fused_lib()
    P = C.c_void_p
    lib.kfh_near_wrap.argtypes = [P, C.c_int32, P, C.POINTER(abi.kf_tracks),
                                  C.POINTER(abi.kf_options), P]
    pick = np.zeros(b.n_tracks, dtype=np.int32)
    tr, fld = oracle.host_tracks(b), field_of(b, b.field.scale)
    assert lib.kfh_near_wrap(b.planes, len(b.planes), C.addressof(fld), C.byref(tr),
                             C.byref(opt), pick.ctypes.data) == 0
    return pick != 0


@pytest.mark.parametrize("cfg,most", [(1, 0.0), (3, 0.0), (5, 0.01)])
def test_tracks_near_the_wrap_are_known_at_the_start(built, cfg, most):
    """Of the tracks that the fused fit would leave in the end, next to none are
    fitted by both programs: the rest are picked from their start, with few
    others, and none where phi stays away from the wrap."""
    b = G.generate(cfg, n_tracks=1500)
    opt = abi.default_options(**dict(W, max_rk_trials=20))
    assert not near_wrap(b, opt).any()
    assert not near_wrap(turned(b, np.pi / 2), opt).any() or cfg == 5
    back = turned(b, np.pi)
    left, pick = fused_fit(back, opt)["redo"] != 0, near_wrap(back, opt)
    assert left.any()
    assert (left & ~pick).mean() <= most
    assert pick.mean() <= 0.25


def test_near_wrap_of_bad_input(built):
    """Tracks that the fit refuses, and values that are not finite, are read
    without going out of the plane table, and are not picked."""
    b = turned(G.generate(1, n_tracks=6), np.pi)
    b.seq_first[:] = [-1, 5, 2**31 - 1, 0, 0, 0]
    b.seq_count[:] = [10, 6, 10, 0, 10, 10]
    b.start_params[2, 4] = np.nan
    b.start_params[4, 5] = np.nan
    assert not near_wrap(b, abi.default_options(**W)).any()


@pytest.mark.parametrize("precision", PRECISIONS)
def test_a_singular_start_covariance_is_left_before_the_pass(built, precision):
    """Every third track without time variance: those are left with nothing of
    them fitted, the others are fitted as by the whole batch's program; tracks that
    the fit refuses keep their flag, and without smoothing nothing is left."""
    b = G.generate(1, n_tracks=60)
    b.start_cov[20, ::3] = 0.0
    b.seq_count[3] = 0
    opt = abi.default_options(precision=precision, **W)
    P = C.c_void_p
    lib = fused_lib()
    lib.kfh_fit_fused_early.argtypes = [P, C.c_int32, P, C.POINTER(abi.kf_tracks),
                                        C.POINTER(abi.kf_options)] + [P] * 6

    def early(o):
        n = b.n_tracks
        out = dict(params=np.zeros((6, n)), cov=np.zeros((21, n)), chi2=np.full(n, -1.0),
                   n_measured=np.full(n, -1, dtype=np.int32),
                   status=np.zeros(n, dtype=np.uint32), redo=np.zeros(n, dtype=np.int32))
        tr, fld = oracle.host_tracks(b), field_of(b, b.field.scale)
        assert lib.kfh_fit_fused_early(b.planes, len(b.planes), C.addressof(fld), C.byref(tr),
                                       C.byref(o), *[v.ctypes.data for v in out.values()]) == 0
        return out

    f, g = early(opt), fused_fit(b, opt)
    left = np.arange(60) % 3 == 0
    left[3] = False
    assert np.array_equal(f["redo"] != 0, left)
    assert (f["chi2"][left] == -1.0).all() and (f["n_measured"][left] == -1).all()
    for k in ("params", "cov", "chi2", "n_measured", "status"):
        assert np.array_equal(f[k][..., ~left], g[k][..., ~left]), k
    assert f["status"][3] == abi.KF_STATUS_BAD_INPUT
    assert not early(abi.default_options(precision=precision, **dict(W, smoothing=0)))["redo"].any()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg,n", [(1, 117), (1, 16385), (3, 40003), (1, 70001)])
def test_gpu_every_way_to_the_rts_program(cfg, n, precision):
    """Tracks around phi = pi, every fiftieth without time variance, so that tracks
    reach the RTS program in all three ways: picked from their start, over their
    own slot, and (beyond 32,768 tracks, or within a few MB) through the pool and
    the list.  The same bits in input order and sorted, replayed, in slices, and
    in the fixed workspace; the counts and flags of the fit with track states, and
    in FP64 its parameters: 1e-6 of an error, as a 2 pi jump of ~6,000 errors takes
    the rounding of 1e-10 there."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = turned(G.generate(cfg, n_tracks=n), np.pi)
    plain = np.arange(n) % 50 != 25
    b.start_cov[20, ~plain] = 0.0
    opts = KalmanFitterOptions(precision=precision, **dict(W, max_rk_trials=20))
    keys = ("params", "cov", "chi2", "ndf", "n_measured", "status")

    def fit(budget=0, call="fit_batch", calls=1, **sched):
        kf = KalmanFitter(b.planes, b.field)
        kf.set_memory_budget(budget)
        kf.set_schedule(**sched)
        dev = DeviceBatch(b)
        for _ in range(calls):
            dev.clear_results()
            getattr(kf, call)(dev, opts)
        res = dev.results_numpy()
        kf.close()
        return res

    want = fit()
    for how in (dict(calls=2), dict(sort_by_length=1), dict(graph=1, calls=3),
                dict(budget=4 << 20), dict(budget=4 << 20, graph=1, calls=3),
                dict(budget=4 << 20, sort_by_length=1), dict(call="fit_batch_noalloc", calls=2)):
        got = fit(**how)
        for k in keys:
            assert np.array_equal(got[k], want[k], equal_nan=True), (how, k)
    kf = KalmanFitter(b.planes, b.field)
    dev = DeviceBatch(b, track_states=True)
    kf.fit_batch(dev, opts)
    ref = dev.results_numpy()
    kf.close()
    for k in ("ndf", "n_measured"):
        assert np.array_equal(want[k], ref[k]), k
    if precision == "fp64":
        assert np.array_equal(want["status"][plain], ref["status"][plain])
        ok = plain & ((ref["status"] & abi.KF_STATUS_OK) != 0)
        sig = np.sqrt(np.abs(ref["cov"][abi.DIAG_INDEX]))[:, ok]
        p = ref["params"][:, ok]
        assert (np.abs(want["params"][:, ok] - p) <= 1e-6 * np.maximum(np.abs(p), sig)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cfg,n", [(1, 200), (1, 40000), (3, 5000)])
def test_gpu_handed_back_tracks_with_a_large_table(cfg, n, precision):
    """300 planes: the table is in global memory, and the RTS program the build for
    either field kind.  The flags and counts of the fit with the small table; in
    FP64 its parameters as in the test above, in the mixed mode those of tracks
    that no wrap is near (twice the mode's 1e-5 between two builds)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    from test_gpu_parity import _padded_planes
    b = turned(G.generate(cfg, n_tracks=n), np.pi)
    plain = np.arange(n) % 50 != 25
    b.start_cov[20, ~plain] = 0.0
    opts = KalmanFitterOptions(precision=precision, **dict(W, max_rk_trials=20))
    res = []
    for x in (b, dataclasses.replace(b, planes=_padded_planes(b.planes, 300 - len(b.planes)))):
        kf = KalmanFitter(x.planes, x.field)
        dev = DeviceBatch(x)
        kf.fit_batch(dev, opts)
        res.append(dev.results_numpy())
        kf.close()
    ref, got = res
    for k in ("ndf", "n_measured"):
        assert np.array_equal(got[k], ref[k]), k
    ok = plain & ((ref["status"] & abi.KF_STATUS_OK) != 0)
    if precision == "fp64":
        assert np.array_equal(got["status"][plain], ref["status"][plain])
    else:
        ok &= ~near_wrap(b, abi.default_options(**W))
        assert np.array_equal(got["status"][ok], ref["status"][ok])
    bar = 1e-6 if precision == "fp64" else 2e-5
    sig = np.sqrt(np.abs(ref["cov"][abi.DIAG_INDEX]))[:, ok]
    p = ref["params"][:, ok]
    assert (np.abs(got["params"][:, ok] - p) <= bar * np.maximum(np.abs(p), sig)).all()


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("lanes", [2, 4])
@pytest.mark.parametrize("n", [3001, 40000])
def test_gpu_handed_back_tracks_with_lane_groups(n, lanes, precision):
    """Several waves to 64 positions, in a small batch (slots of the positions) and
    through the pool and the list: repeated fits give the same bits, flags and
    counts are those of one lane per track, and so are in FP64 the parameters
    (1e-6 as above)."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = turned(G.generate(1, n_tracks=n), np.pi)
    plain = np.arange(n) % 50 != 25
    b.start_cov[20, ~plain] = 0.0
    opts = KalmanFitterOptions(precision=precision, **dict(W, max_rk_trials=20))
    kf = KalmanFitter(b.planes, b.field)
    dev = DeviceBatch(b)
    kf.fit_batch(dev, opts)
    want = dev.results_numpy()
    kf.set_schedule(lanes_per_track=lanes)
    got = []
    for _ in range(2):
        dev.clear_results()
        kf.fit_batch(dev, opts)
        got.append(dev.results_numpy())
    kf.close()
    for k in ("params", "cov", "chi2", "ndf", "n_measured", "status"):
        assert np.array_equal(got[0][k], got[1][k], equal_nan=True), k
    g = got[0]
    for k in ("ndf", "n_measured"):
        assert np.array_equal(g[k], want[k]), k
    if precision == "fp64":
        assert np.array_equal(g["status"][plain], want["status"][plain])
        ok = plain & ((want["status"] & abi.KF_STATUS_OK) != 0)
        sig = np.sqrt(np.abs(want["cov"][abi.DIAG_INDEX]))[:, ok]
        p = want["params"][:, ok]
        assert (np.abs(g["params"][:, ok] - p) <= 1e-6 * np.maximum(np.abs(p), sig)).all()
