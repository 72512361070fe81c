"""The predictor straight from HBM on grids whose interior rows have a launch of
their own (k_momentum_rows, from 1.5 M cells on): with the fast divisions (variant
4), and with the division instruction, which the default takes when a spacing lies
outside [2^-64, 2^64] (the same grid 1e25 times smaller).  Last tiles of one and of
63 columns, sides that are no multiple of the four rows of a workgroup.  The same
arithmetic in the same order, so every fluid cell must have the oracle's bits, and
the others stay as they were."""
import os

import numpy as np
import pytest
from test_gpu_momentum_rows import OUT, _fields

pytestmark = pytest.mark.gpu

GRIDS = [(18, (68, 151, 149)), (12, (129, 110, 107)), (12, (131, 109, 106)), (12, (130, 108, 107))]


def _dp(a):
    import ctypes
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_double))


@pytest.mark.parametrize("per,n", GRIDS)
def test_rows_match_the_oracle(tmp_path, per, n):
    from ib3d_amd import cases
    from ib3d_amd.native import Solver
    import pyoracle
    assert np.prod(n) >= 1500000
    cfg = cases.CaseConfig("large", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / per, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s, o = Solver.from_case(str(tmp_path)), pyoracle.Oracle.from_case(str(tmp_path))
    try:
        rng = np.random.default_rng(sum(n))
        grid = [cases.read_grid(os.path.join(str(tmp_path), f"grid{a}.dat"), k + 1) for a, k in zip("xyz", n)]
        for scale, variant, odd in ((1.0, 4, False), (1.0, 4, True), (1e-25, 0, False), (1e-25, 4, True)):
            if scale != 1.0:
                g = [np.ascontiguousarray(scale * a) for a in grid]
                assert s.L.ib3d_set_grid(*map(_dp, g)) == 0
                assert s.L.ib3d_coefficientMatrix() == 0 and s.L.ib3d_non_uni_coeff() == 0
                o._ok(o.L.orc_set_grid(o.h, *map(_dp, g)))
                o._ok(o.L.orc_coefficient_matrix(o.h))
                o._ok(o.L.orc_non_uni_coeff(o.h))
            for f, a in _fields(n, rng, odd).items():
                s.upload(f, a)
                o.field(f)[...] = a
            for f in OUT:
                s.upload(f, np.full((n[0] + 2) * (n[1] + 2) * (n[2] + 2), 7.0))
            o.call("ns_momentum")
            print(f"[gpu] direct momentum {n} scale={scale} variant {variant} odd={odd}", flush=True)
            s.set_momentum_tiles(variant)
            s.nsMomentum()
            cells = s.download("cell").reshape([k + 2 for k in n], order="F")
            inner = np.zeros(cells.shape, bool)
            inner[1:-1, 1:-1, 1:-1] = True
            fluid = (inner & (cells == 0)).reshape(-1, order="F")
            for f in OUT:
                got = s.download(f)
                x, y = got[fluid], o.array(f)[fluid]
                # (the sign of a NaN that an operation makes is the machine's)
                np.testing.assert_array_equal(np.isnan(x), np.isnan(y), err_msg=f)
                x, y = x[~np.isnan(x)], y[~np.isnan(y)]
                np.testing.assert_array_equal(x.view(np.int64), y.view(np.int64), err_msg=f)
                np.testing.assert_array_equal(got[~fluid], 7.0, err_msg=f)
    finally:
        s.set_momentum_tiles(0)
        s.close()
