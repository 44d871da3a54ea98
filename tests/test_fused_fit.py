"""The fused FP64 fit (fixed-point smoother) against the RTS program, on the CPU
(tests/host/libkffusedcheck.so) and on the GPU, over what decides which of the
two a track ends on: angles near the phi wrap, singular covariances, exact
hits, one to forty planes, holes."""
import ctypes as C
import dataclasses
import os

import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

import oracle
from parity import compare_fit
from test_adjoint_cpu import HOST, field_of
from test_host_fit import host_fit

W = configs.WORKLOAD_FIT_OPTIONS


def fused_lib():
    path = os.path.join(HOST, "libkffusedcheck.so")
    if not os.path.exists(path):
        import subprocess
        subprocess.run(["make", "-s", "-C", HOST], check=True)
    lib = C.CDLL(path)
    P = C.c_void_p
    lib.kfh_fit_fused.argtypes = [P, C.c_int32, P, C.POINTER(abi.kf_tracks),
                                  C.POINTER(abi.kf_options)] + [P] * 6
    return lib


def fused_fit(b, opt):
    n = b.n_tracks
    out = dict(params=np.zeros((6, n)), cov=np.zeros((21, n)), chi2=np.zeros(n),
               n_measured=np.zeros(n, dtype=np.int32), status=np.zeros(n, dtype=np.uint32),
               redo=np.zeros(n, dtype=np.int32))
    tr = oracle.host_tracks(b)
    fld = field_of(b, b.field.scale)
    assert fused_lib().kfh_fit_fused(b.planes, len(b.planes), C.addressof(fld), C.byref(tr),
                                     C.byref(opt),
                                     *[v.ctypes.data for v in out.values()]) == 0
    return out


def turned(b, angle):
    """The batch turned about the z axis."""
    c, s = np.cos(angle), np.sin(angle)
    R = np.array([[c, -s, 0.0], [s, c, 0.0], [0.0, 0.0, 1.0]])
    planes = (abi.kf_plane * len(b.planes))()
    C.memmove(planes, b.planes, C.sizeof(planes))
    for p in planes:
        p.center[:] = list(R @ np.array(p.center[:]))
        p.rot[:] = list((R @ np.array(p.rot[:]).reshape(3, 3)).ravel())
    params = b.start_params.copy()
    params[2] = (params[2] + angle + np.pi) % (2 * np.pi) - np.pi
    return dataclasses.replace(b, planes=planes, start_params=params, perigee=R @ b.perigee)


def variant(name, n, cfg=1):
    if name == "one plane":
        return G.generate(1, n_tracks=n, n_planes=1, min_planes=1, max_planes=1)
    if name == "two planes":
        return G.generate(1, n_tracks=n, n_planes=2, min_planes=2, max_planes=2)
    b = G.generate(cfg, n_tracks=n)
    if name == "phi wrap":
        return turned(b, np.pi)
    if name == "no time variance":
        cov = b.start_cov.copy()
        cov[20] = 0.0
        return dataclasses.replace(b, start_cov=cov)
    if name == "correlated start":
        cov = b.start_cov.copy()
        cov[1] = np.sqrt(cov[0] * cov[6])  # loc0 and loc1 fully correlated
        return dataclasses.replace(b, start_cov=cov)
    if name == "exact hits":
        hc = b.hit_cov.copy()
        hc[0] *= 1e-20
        hc[2] *= 1e-20
        return dataclasses.replace(b, hit_cov=hc)
    return b


# whether the tracks stay with the fixed-point smoother
CASES = [("one plane", 1, "all"), ("two planes", 1, "all"), ("plain", 1, "all"),
         ("plain", 3, "all"), ("plain", 5, "all"), ("phi wrap", 1, "some"),
         ("no time variance", 1, "none"), ("correlated start", 1, "none"),
         ("exact hits", 1, "none")]


@pytest.mark.parametrize("name,cfg,stay", CASES)
def test_fused_program_equals_rts_program(built, name, cfg, stay):
    """Tracks that stay give the RTS program's fit (bar: the 1e-9 of the FP64
    parity); the others are exactly those its discrete behaviour could touch."""
    b = variant(name, 400, cfg)
    opt = abi.default_options(**W)
    f, r = fused_fit(b, opt), host_fit(b, opt)
    kept = f["redo"] == 0
    assert {"all": kept.all(), "none": not kept.any(),
            "some": kept.any() and not kept.all()}[stay]
    assert np.array_equal(f["n_measured"], r["n_measured"])
    assert np.array_equal(f["chi2"], r["chi2"], equal_nan=True)
    if not kept.any():
        return
    assert np.array_equal(f["status"][kept], r["status"][kept])
    sig = np.sqrt(np.abs(r["cov"][abi.DIAG_INDEX]))[:, kept]
    p = r["params"][:, kept]
    assert (np.abs(f["params"][:, kept] - p) <= 1e-9 * np.maximum(np.abs(p), sig)).all()
    for (i, j), k in abi.SYM_INDEX.items():
        d = np.abs(f["cov"][k, kept] - r["cov"][k, kept])
        assert (d <= 1e-9 * sig[i] * sig[j]).all(), (i, j)
    if name == "phi wrap":  # no smoothed angle of a track that stays is near the wrap
        assert (np.abs(f["params"][2, kept]) < np.pi).all()


@pytest.mark.parametrize("name,cfg,stay", CASES)
def test_mixed_fused_program_equals_rts_program(built, name, cfg, stay):
    """The mixed mode's sums (RTS gains of the float covariances) against its RTS
    program.  The float operations are the same and the rest is double, so the two
    differ by 1e-13 and, where that turns the rounding of a float covariance entry
    (one entry in a million), by what 6e-8 of it becomes: a tenth of the mode's
    bars against the oracle."""
    b = variant(name, 400, cfg)
    opt = abi.default_options(precision=abi.KF_PRECISION_MIXED, **W)
    f, r = fused_fit(b, opt), host_fit(b, opt)
    kept = f["redo"] == 0
    assert {"all": kept.all(), "none": not kept.any(),
            "some": kept.any() and not kept.all()}[stay]
    if not kept.any():
        return
    assert np.array_equal(f["n_measured"][kept], r["n_measured"][kept])
    assert np.array_equal(f["status"][kept], r["status"][kept])
    sig = np.sqrt(np.abs(r["cov"][abi.DIAG_INDEX]))[:, kept]
    p = r["params"][:, kept]
    assert (np.abs(f["params"][:, kept] - p) <= 1e-6 * np.maximum(np.abs(p), sig)).all()
    for (i, j), k in abi.SYM_INDEX.items():
        d = np.abs(f["cov"][k, kept] - r["cov"][k, kept])
        assert (d <= 1e-4 * sig[i] * sig[j]).all(), (i, j)


@pytest.mark.gpu
@pytest.mark.parametrize("name,cfg,n", [("one plane", 1, 1), ("two planes", 1, 65),
                                        ("phi wrap", 1, 20000), ("no time variance", 1, 20000),
                                        ("correlated start", 1, 129)])
@pytest.mark.parametrize("sched", [dict(), dict(sort_by_length=1, persistent=1, graph=1),
                                   dict(lanes_per_track=2)])
def test_gpu_fused_fit_with_handed_back_tracks(name, cfg, n, sched):
    """The GPU fit, tracks handed back included (20,000 are more than the pool of
    store chunks holds: the rest goes through the list), against the fit with
    track states, which runs the RTS program for every track.  Twice, so the
    second call meets the counters the first one left.  Bar: 1e-10 between two
    builds of the same program; a phi wrap puts a 2 pi jump (~6,000 sigma)
    through the recursion, 1e-6 there; near-singular matrices amplify rounding
    without bound, so only what is discrete is compared."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = variant(name, n, cfg)
    kf = KalmanFitter(b.planes, b.field)
    opts = KalmanFitterOptions(**W)
    ref_dev = DeviceBatch(b, track_states=True)
    kf.fit_batch(ref_dev, opts)
    ref = ref_dev.results_numpy()
    kf.set_schedule(**sched)
    dev = DeviceBatch(b)
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
        assert np.array_equal(g[k], ref[k]), k
    if name in ("no time variance", "correlated start"):
        return
    assert np.array_equal(g["status"], ref["status"])

    class R:
        pass
    o = R()
    o.status, o.params, o.cov, o.chi2 = (ref[k] for k in ("status", "params", "cov", "chi2"))
    pd, cd, c2 = compare_fit(g, o)
    bar = 1e-6 if name == "phi wrap" else 1e-10
    assert max(pd, cd, c2) <= bar, (pd, cd, c2)


@pytest.mark.gpu
@pytest.mark.parametrize("name,cfg,n", [("one plane", 1, 1), ("two planes", 1, 65),
                                        ("phi wrap", 1, 20000), ("no time variance", 1, 20000)])
@pytest.mark.parametrize("sched", [dict(), dict(sort_by_length=1, persistent=1, graph=1),
                                   dict(lanes_per_track=4), dict(store_by_plane=1)])
def test_gpu_mixed_fused_fit_with_handed_back_tracks(name, cfg, n, sched):
    """The same in the mixed mode: repeated calls and every schedule give the same
    bits, and tracks that are not at the phi wrap are within twice the mode's
    bars (1e-5, 1e-3) of the fit with track states."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import DeviceBatch, KalmanFitter, KalmanFitterOptions
    b = variant(name, n, cfg)
    kf = KalmanFitter(b.planes, b.field)
    opts = KalmanFitterOptions(precision="mixed", **W)
    ref_dev = DeviceBatch(b, track_states=True)
    kf.fit_batch(ref_dev, opts)
    ref = ref_dev.results_numpy()
    dev = DeviceBatch(b)
    kf.fit_batch(dev, opts)
    got = [dev.results_numpy()]
    kf.set_schedule(**sched)
    for _ in range(2):
        dev.clear_results()
        kf.fit_batch(dev, opts)
        got.append(dev.results_numpy())
    kf.close()
    for k in ("ndf", "n_measured"):
        assert np.array_equal(got[0][k], ref[k]), k
    if sched.get("lanes_per_track", 1) == 1:
        for k in ("params", "cov", "chi2", "ndf", "n_measured", "status"):
            assert np.array_equal(got[0][k], got[1][k], equal_nan=True), k
    for k in ("params", "cov", "chi2", "ndf", "n_measured", "status"):
        assert np.array_equal(got[1][k], got[2][k], equal_nan=True), k
    if name in ("no time variance", "phi wrap"):
        return
    assert np.array_equal(got[1]["status"], ref["status"])

    class R:
        pass
    o = R()
    o.status, o.params, o.cov, o.chi2 = (ref[k] for k in ("status", "params", "cov", "chi2"))
    pd, cd, _ = compare_fit(got[1], o)
    assert pd <= 2e-5 and cd <= 2e-3, (pd, cd)
