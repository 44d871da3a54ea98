"""When a fit sorts its tracks by length, and what the autotuner tries (the library's
own rules, in the CPU build)."""
import ctypes as C

import pytest

from gpukalmanfitter_amd import abi
from gpukalmanfitter_amd import generate as G

from test_fused_fit import fused_lib

N_CU = 256


def sorts(sort, n=100000, fill=0.6, max_states=30, fused=True, lanes=1):
    lib = fused_lib()
    lib.kfh_sorts.argtypes = [C.POINTER(abi.kf_schedule), C.c_int32, C.c_int64, C.c_int64,
                              C.c_int32, C.c_int32]
    s = abi.kf_schedule(sort_by_length=sort, lanes_per_track=lanes)
    return bool(lib.kfh_sorts(C.byref(s), int(fused), n, int(fill * n * max(max_states, 1)),
                              max_states, N_CU))


def candidates(track_states):
    lib = fused_lib()
    lib.kfh_schedule_candidates.argtypes = [C.c_int32, C.c_void_p, C.c_int32]
    buf = (abi.kf_schedule * 64)()
    n = lib.kfh_schedule_candidates(int(track_states), C.addressof(buf), 64)
    return [buf[k].as_dict() for k in range(n)]


@pytest.mark.parametrize("fused", [True, False])
def test_an_explicit_choice_is_kept(built, fused):
    assert not sorts(0, fused=fused)
    assert sorts(1, fused=fused)
    assert sorts(1, n=100, fill=1.0, fused=fused)


def test_the_automatic_choice(built):
    auto = abi.KF_SORT_AUTO
    assert sorts(auto)
    assert not sorts(auto, fused=False)
    assert not sorts(auto, fill=0.95)           # equal lengths with few holes
    assert not sorts(auto, max_states=0)        # the longest track is not stated
    assert not sorts(auto, n=256 * N_CU)        # one wave per SIMD
    assert sorts(auto, n=256 * N_CU + 1)
    assert sorts(auto, n=128 * N_CU + 1, lanes=2)


def test_autotuner_candidates(built):
    """Each states whether it sorts; no two of them launch the same kernels in the
    same way."""
    for states, count in ((False, 6), (True, 32)):
        c = candidates(states)
        assert len(c) == count
        assert all(s["sort_by_length"] in (0, 1) and s["graph"] == 1 for s in c)
        assert len({tuple(s.items()) for s in c}) == count
        if not states:
            assert not any(s["persistent"] or s["store_by_plane"] for s in c)


@pytest.mark.gpu
def test_gpu_default_and_explicit_order(built):
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    from gpukalmanfitter_amd.fitter import KalmanFitter
    b = G.generate(1, n_tracks=64)
    kf = KalmanFitter(b.planes, b.field)
    assert kf.schedule()["sort_by_length"] == abi.KF_SORT_AUTO
    for sort in (0, 1):
        kf.set_schedule(sort_by_length=sort)
        assert kf.schedule()["sort_by_length"] == sort
    kf.close()
