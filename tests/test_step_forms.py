"""The RK step's two forms (polynomials of the direction in a constant field,
column-by-column transport in any field) and the angles by rotation, in the
fused program built for the CPU, against the oracle."""
import ctypes as C
import dataclasses

import numpy as np
import pytest

from gpukalmanfitter_amd import abi, configs
from gpukalmanfitter_amd import generate as G

import oracle
from parity import compare_fit
from test_adjoint_cpu import field_of
from test_fused_fit import fused_lib, turned

W = configs.WORKLOAD_FIT_OPTIONS
T = configs.TESLA


def fit_kind(b, opt, kind):
    n = b.n_tracks
    out = dict(params=np.zeros((6, n)), cov=np.zeros((21, n)), chi2=np.zeros(n),
               n_measured=np.zeros(n, dtype=np.int32), status=np.zeros(n, dtype=np.uint32),
               redo=np.zeros(n, dtype=np.int32))
    lib = fused_lib()
    P = C.c_void_p
    lib.kfh_fit_fused_kind.argtypes = [P, C.c_int32, P, C.POINTER(abi.kf_tracks),
                                       C.POINTER(abi.kf_options), C.c_int32] + [P] * 6
    tr, fld = oracle.host_tracks(b), field_of(b, b.field.scale)
    assert lib.kfh_fit_fused_kind(b.planes, len(b.planes), C.addressof(fld), C.byref(tr),
                                  C.byref(opt), kind, *[v.ctypes.data for v in out.values()]) == 0
    return out


@pytest.mark.parametrize("kind", [0, 1])
@pytest.mark.parametrize("field,scale,tol", [
    ((0.0, 0.0, 0.0), 1.0, 1e-4),           # no curvature: every stage is zero
    ((0.0, 0.0, 2.0 * T), 1.0, 1e-4),
    ((0.0, 0.0, 2.0 * T), 1.01, 1e-4),
    ((0.2 * T, -0.3 * T, 2.0 * T), 1.0, 1e-4),
    ((0.0, 0.0, 2.0 * T), 1.0, 1e-9),       # many rejected trials per step
])
@pytest.mark.parametrize("angle", [0.0, 2.0])
def test_constant_field_fit_matches_oracle(built, kind, field, scale, tol, angle):
    """Bar: the 1e-9 of the FP64 parity."""
    b = G.generate(1, n_tracks=300)
    b = turned(dataclasses.replace(b, field=dataclasses.replace(b.field, b=field, scale=scale)),
               angle)
    opt = abi.default_options(**W)
    opt.tolerance = tol
    f = fit_kind(b, opt, kind)
    o, _, _, _ = oracle.fit(b, opt)
    keep = f["redo"] == 0
    assert keep.sum() > 250
    assert np.array_equal(f["status"][keep], o.status[keep])
    fin = keep & ((o.status & abi.KF_STATUS_FINISHED) != 0)
    pd, cd, c2 = compare_fit(f, o, mask=fin)
    assert max(pd, cd, c2) <= 1e-9, (pd, cd, c2)


@pytest.mark.parametrize("p", [0.02, 0.1, 0.5])
def test_low_momentum_rotations_match_oracle(built, p):
    """Momenta at which the direction turns by more than 1/16 between planes (the
    library's arc tangents) and by less (the series).  Bar: 1e-9."""
    b = G.generate(1, n_tracks=200, p_min=p, p_max=1.5 * p, pitch=6.0, first_x=6.0)
    opt = abi.default_options(**W)
    f = fit_kind(b, opt, 1)
    o, _, _, _ = oracle.fit(b, opt)
    keep = (f["redo"] == 0)
    assert np.array_equal(f["status"][keep], o.status[keep])
    fin = keep & ((o.status & abi.KF_STATUS_OK) != 0)
    print(p, keep.sum(), fin.sum())
    if fin.any():
        pd, cd, c2 = compare_fit(f, o, mask=fin)
        assert max(pd, cd, c2) <= 1e-9, (pd, cd, c2)


@pytest.mark.parametrize("n,half", [((2, 2, 2), 2000.0), ((3, 2, 5), 150.0), ((40, 40, 40), 290.0)])
def test_grid_lookups_match_oracle(built, n, half):
    """The grid build, which keeps the cell of its last lookup: one cell for the
    whole detector, boxes that end inside it (lookups clamped to the edge), and
    cells smaller than a step.  Bar: 1e-9."""
    b = G.generate(1, n_tracks=300)
    rng = np.random.default_rng(3)
    v = np.zeros(n + (3,), dtype=np.float32)
    v[..., 2] = 2.0 * T
    v += (0.2 * T * rng.standard_normal(v.shape)).astype(np.float32)
    fld = G.FieldSpec(kind="grid", values=v, lo=(-half,) * 3, hi=(half,) * 3, scale=1.01)
    b = dataclasses.replace(b, field=fld)
    opt = abi.default_options(**W)
    f = fit_kind(b, opt, 2)
    o, _, _, _ = oracle.fit(b, opt)
    keep = f["redo"] == 0
    assert keep.sum() > 250
    assert np.array_equal(f["status"][keep], o.status[keep])
    fin = keep & ((o.status & abi.KF_STATUS_OK) != 0)
    assert fin.sum() > 250
    pd, cd, c2 = compare_fit(f, o, mask=fin)
    assert max(pd, cd, c2) <= 1e-9, (pd, cd, c2)
