"""The predictor's two kernels for large grids: rows without a branch by the
tiles, the rows they list (walls, bodies, velocities or pressure differences
outside the range of the untested quotients) by the general one.  Grids around
the tile's 64 columns and 8 rows and with a few planes; fields with runs of equal
values, zeros of both signs and, in places, values outside the range.  The same
arithmetic in the same order, so every value must have the oracle's bits, also
on further calls, whose row counts start from the other counter."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
OUT = ("ut", "vt", "wt", "resi_u", "resi_v", "resi_w")

# cells per unit length of the uniform box, and the interior grid
GRIDS = [(4, (66, 23, 17)), (4, (67, 24, 18)), (4, (68, 25, 19)), (8, (130, 33, 30)), (8, (131, 34, 31)),
         (4, (33, 16, 38)), (10, (49, 66, 98)),
         (10, (69, 98, 98))]   # the last tile has 2 columns, a workgroup 6 planes


def _fields(n, rng, odd):
    shape = tuple(k + 2 for k in n)
    out = {}
    for f in ("u", "v", "w", "p"):
        a = rng.standard_normal(shape)
        a[:, : shape[1] // 3] = 1.0                      # differences of exactly zero
        a[shape[0] // 2:, shape[1] // 3: shape[1] // 2] = -0.0
        a[: shape[0] // 2, shape[1] // 3: shape[1] // 2] *= rng.choice([0.0, -0.0, 1.0, -1.0, 1e-30], a[: shape[0] // 2, shape[1] // 3: shape[1] // 2].shape)
        if odd:
            at = tuple(rng.integers(0, k, 12) for k in shape)
            a[at] = rng.choice([1e-250, 5e-324, 1e-201, -1e250, 1e150], 12)
        out[f] = np.asfortranarray(a)
    return out


@pytest.mark.parametrize("per,n", GRIDS)
def test_rows_match_the_oracle(tmp_path, per, n):
    from ib3d_amd import cases
    from ib3d_amd.native import Solver
    import pyoracle
    cfg = cases.CaseConfig("rows", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / per, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s, o = Solver.from_case(str(tmp_path)), pyoracle.Oracle.from_case(str(tmp_path))
    try:
        rng = np.random.default_rng(sum(n))
        for odd in (False, True, False):
            for f, a in _fields(n, rng, odd).items():
                s.upload(f, a)
                o.field(f)[...] = a
            o.call("ns_momentum")
            for variant in (1, 1, 4, 0):
                for f in OUT:
                    s.upload(f, np.full(a.size, 7.0))
                o_before = {f: o.array(f).copy() for f in OUT}
                print(f"[gpu] momentum rows {n} odd={odd} variant {variant}", flush=True)
                s.set_momentum_tiles(variant)
                s.nsMomentum()
                cells = s.download("cell").reshape([k + 2 for k in n], order="F")
                inner = np.zeros(cells.shape, bool)
                inner[1:-1, 1:-1, 1:-1] = True
                fluid = (inner & (cells == 0)).reshape(-1, order="F")
                assert fluid.any()
                for f in OUT:
                    got = s.download(f)
                    x, y = got[fluid], o_before[f][fluid]
                    # (the sign of a NaN that an operation makes is the machine's)
                    np.testing.assert_array_equal(np.isnan(x), np.isnan(y), err_msg=f)
                    x, y = x[~np.isnan(x)], y[~np.isnan(y)]
                    np.testing.assert_array_equal(x.view(np.int64), y.view(np.int64), err_msg=f)
                    np.testing.assert_array_equal(got[~fluid], 7.0, err_msg=f)
    finally:
        s.set_momentum_tiles(0)
        s.close()
