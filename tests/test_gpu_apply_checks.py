"""One application of the preconditioner on device arrays: a residual with a
single non-finite entry, wherever it sits, is refused and leaves the output as
it was, the next application is what it would have been, and the output may be
the residual's own array."""
import numpy as np
import pytest

import cfdx_dev_amd as cx
from hipmem import DeviceArray
from systems import box_mesh, pressure_system

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims", [(4, 3, 2), (12, 11, 9)])  # one level; several
def test_refused_residual_leaves_no_trace(oracle, precision, dims):
    s = pressure_system(oracle, box_mesh(*dims, jitter=0.15, seed=6), sigma=1.2, seed=6)
    n = s["n"]
    h = cx.NativeAMGPreconditioner(method="sa", precision=precision, require_smoother_certificate=False)
    assert h.setup(n, s["rowp"], s["cols"], s["vals"]), h.last_error()
    r = np.random.default_rng(4).normal(size=n)
    good = h.apply(r)
    for at, bad in ((0, np.nan), (n // 2, -np.inf), (n - 1, np.inf)):
        x = r.copy()
        x[at] = bad
        dx, dz = DeviceArray(x), DeviceArray(np.full(n, 7.0))
        assert not h.apply_device(dx.ptr, dz.ptr)
        assert "non-finite residual" in h.last_error()
        assert np.array_equal(dz.download(), np.full(n, 7.0))
        dx.upload(r)
        assert h.apply_device(dx.ptr, dz.ptr), h.last_error()
        assert np.array_equal(dz.download(), good)
    dx = DeviceArray(r)
    assert h.apply_device(dx.ptr, dx.ptr), h.last_error()
    assert np.array_equal(dx.download(), good)
