"""The coarse end of the FP64 V-cycle, run by one workgroup from the first
level that fits it (cfdx_dev_amd/csrc/coarse_tail.hpp), against the oracle bit
for bit, where it can go wrong:
* the whole hierarchy in one launch, and only its end;
* rows of more than 64 entries in groups (classical C/F on the 2-D Poisson
  square) and alone in their group (arrow rows of the filtered channel
  hierarchy, longer than one staged chunk);
* a coarsest level without dense factors (24 sweeps), policies of 2 and 6
  sweeps, Chebyshev smoothing with a recurrence;
* after a numeric refresh (packed values, damping and coefficients renewed).
A hierarchy with the constant null space, whose mean removals are launches
between the sweeps, keeps the launches.
"""
import numpy as np
import pytest

import cfdx_dev_amd as cx
from systems import box_mesh, channel_system, neumann_system, pressure_system
from test_poisson_mms import mms_system

pytestmark = pytest.mark.gpu

FILTER = dict(prolongator_filter=0.2, filter_keeps_aggregate=True)
CASES = {
    "whole_box": ("sa", "balanced", {}, lambda o: pressure_system(o, box_mesh(8, 7, 6, seed=5), seed=5)),
    "end_of_box": ("sa", "low", {}, lambda o: pressure_system(o, box_mesh(24, 23, 22, seed=5), seed=5)),
    "grouped_rows": ("boomer", "balanced", {}, lambda o: mms_system(o, 128)),
    "grouped_rows_small": ("boomer", "balanced", {}, lambda o: mms_system(o, 50)),
    "arrow_rows": ("sa", "balanced", FILTER, lambda o: channel_system(o, (80, 32, 30), 3, 1)),
    "chebyshev": ("sa", "balanced", dict(FILTER, smoother="chebyshev"),
                  lambda o: channel_system(o, (40, 16, 14), 3, 2)),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_coarse_end_bit_identical(oracle, name):
    method, policy, opt, make = CASES[name]
    s = make(oracle)
    ao = oracle.amg(method, policy=policy, **opt)
    assert ao.setup(s["n"], s["rowp"], s["cols"], s["vals"])
    ap = cx.NativeAMGPreconditioner(method=method, policy=policy, **opt)
    assert ap.setup(s["n"], s["rowp"], s["cols"], s["vals"]), ap.last_error()
    # the coarse end runs: of every level, or from one below the first on
    assert ap.num_levels() > 2
    assert ap.coarse_end() == 0 if name == "whole_box" else 0 < ap.coarse_end() < ap.num_levels() - 1
    rng = np.random.default_rng(11)
    for refresh in (False, True):
        if refresh:
            # A few percent; entries of the boxes' Galerkin products that
            # cancel exactly stay pruned only under a uniform scaling.
            d = np.full(s["n"], 2.0) if "box" in name else np.exp(0.05 * rng.normal(size=s["n"]))
            rows = np.repeat(np.arange(s["n"]), np.diff(s["rowp"].astype(np.int64)))
            vals = s["vals"] * d[rows] * d[s["cols"]]
            assert ao.update_values(vals) and ap.update_values(vals), ap.last_error()
        for _ in range(2):
            r = rng.normal(size=s["n"])
            assert np.array_equal(ao.apply(r), ap.apply(r))


@pytest.mark.parametrize("method,dims", [("sa", (8, 7, 6)), ("sa", (20, 18, 16)), ("boomer", (14, 12, 11))])
def test_null_space_keeps_the_launches(oracle, method, dims):
    s = neumann_system(oracle, box_mesh(*dims, jitter=0.15, seed=6), seed=6)
    h = cx.NativeAMGPreconditioner(method=method, constant_null_space=True)
    assert h.setup(s["n"], s["rowp"], s["cols"], s["vals"]), h.last_error()
    assert h.num_levels() > 2 and h.coarse_end() == h.num_levels()
