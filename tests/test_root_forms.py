"""The square root and reciprocal square root by Newton iterations on an estimate (the
device's, run here on estimates of several accuracies)."""
import ctypes as C

import numpy as np
import pytest

from test_fused_fit import fused_lib


@pytest.mark.parametrize("estimate", [1e-5, 6e-8, 1e-8, 1e-9])
def test_roots_do_not_lean(built, estimate):
    """Against 80-bit roots: the root to half an ulp, its reciprocal to the half ulp of
    the root and one of its own, and neither to one side.  A mean of 400,000 errors
    below 1.5 ulp and spread over at least one has a standard error below 0.0012;
    five of them."""
    rng = np.random.default_rng(3)
    n = 400000
    x = rng.uniform(0.25, 1.0, n)
    y = (1.0 / np.sqrt(x)) * (1.0 + rng.uniform(-estimate, estimate, n))
    s, inv = np.empty(n), np.empty(n)
    lib = fused_lib()
    lib.kfh_roots.argtypes = [C.c_int64] + [C.c_void_p] * 4
    lib.kfh_roots(n, *[v.ctypes.data for v in (x, y, s, inv)])
    root = np.sqrt(x.astype(np.longdouble))
    for got, want, most in ((s, root, 0.501), (inv, 1 / root, 1.501)):
        err = ((got - want) / np.spacing(got)).astype(np.float64)
        assert np.abs(err).max() <= most
        assert abs(err.mean()) <= 0.006, err.mean()
