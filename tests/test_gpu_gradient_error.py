"""The rounding error of the chi2 gradient, a sum over tracks of terms that cancel."""
import os
import sys

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.gpu
@pytest.mark.parametrize("seed", [0, 1])
def test_gpu_gradient_error_against_autograd(seed):
    """262,144 tracks, the derivatives to the planes' centres and frames against the same
    fit in plain torch FP64 by autograd: 2.4e-13 of their length with correctly
    rounded roots and quotients (the reference's own rounding in it), and no more
    with the kernels' Newton forms."""
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    if ROOT not in sys.path:
        sys.path.insert(0, ROOT)
    from perf import cases
    case = dict(call="gradient", detector=4, tracks=262144, precision="fp64")
    got = cases.run(cases.prepare(case, seed))
    want = cases.exact(case, seed)
    raw, ref = (np.asarray(x["raw"].cpu() if torch.is_tensor(x["raw"]) else x["raw"])
                for x in (got, want))
    err = np.sqrt(((raw - ref) ** 2).sum() / (ref ** 2).sum())
    print(f"gradient error {err:.3e}")
    assert err <= 2.4e-13, err
