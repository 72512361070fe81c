"""Two sweeps per launch (k_sor_block, k_sor_march) against the oracle's plain
loops.

FP64: the same operations per cell in the same order, so the iteration count
and every value of pc must be bit-identical, under the reference rule (whose
last launch may hold one sweep too many) and in the L2 mode.  FP32 (the defect
equation): n sweeps from zero differ from n FP64 sweeps by rounding only.  The
grids lie around the block shapes' and the march's tiles' edges and on both sides
of the size rules."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells per unit length of the uniform box, and the interior grid
GRIDS = [(4, (32, 24, 24)), (4, (33, 25, 23)), (4, (31, 17, 18)), (6, (42, 40, 39)), (6, (66, 50, 46)),
         (8, (65, 63, 64)), (8, (73, 66, 57)), (10, (98, 64, 49)), (12, (121, 113, 112)), (14, (122, 128, 97)),
         (10, (190, 90, 91)), (12, (119, 93, 73))]


def _pair(tmp_path, per, n, scale=1.0, seed=3):
    """GPU solver and oracle of one sphere case with the same random ut, vt,
    wt (and so the same right-hand side)."""
    from ib3d_amd import cases
    from ib3d_amd.native import Solver
    import pyoracle
    cfg = cases.CaseConfig("block", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / per, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s, o = Solver.from_case(str(tmp_path)), pyoracle.Oracle.from_case(str(tmp_path))
    rng = np.random.default_rng(seed)
    shape = tuple(k + 2 for k in n)
    for f in ("ut", "vt", "wt"):
        a = np.asfortranarray(scale * rng.standard_normal(shape))
        s.upload(f, a)
        o.field(f)[...] = a
    return s, o


def _same(a, b):
    return np.array_equal(a.view(np.int64), b.view(np.int64))


@pytest.mark.parametrize("per,n", GRIDS)
def test_reference_rule_matches_the_oracle(tmp_path, per, n):
    s, o = _pair(tmp_path, per, n)
    try:
        assert s.computeDiv() == o.compute_div()
        counts = set()
        # each solve goes on from the last one's pc
        for eps in (2.0, 0.8, 0.5, 0.3):
            print(f"[gpu] blocks {n} eps={eps}", flush=True)
            it, d2 = s.REDBLACKSOR(eps)
            ito, d2o = o.redblack_sor(eps)
            assert (it, d2) == (ito, d2o)
            counts.add(it % 2)
            assert _same(s.download("pc"), o.array("pc"))
        print(f"[gpu] blocks {n}: identical, parities of the counts {counts}", flush=True)
    finally:
        s.close()


@pytest.mark.parametrize("scale", [1e-270, 1e-305, 1e120, 0.0])
def test_extreme_values_match_the_oracle(tmp_path, scale):
    """Numerators outside the range of the blocks' own division (and zeros)."""
    s, o = _pair(tmp_path, 4, (33, 25, 23), scale)
    try:
        s.computeDiv()
        o.compute_div()
        for eps in (scale, 0.3 * scale) if scale else (1e-5,):
            it, d2 = s.REDBLACKSOR(eps)
            ito, d2o = o.redblack_sor(eps)
            assert (it, d2) == (ito, d2o)
            assert _same(s.download("pc"), o.array("pc"))
    finally:
        s.close()


@pytest.mark.parametrize("check", [2, 3, 4, 7, 10])
@pytest.mark.parametrize("per,n", [GRIDS[1], GRIDS[4], GRIDS[6], GRIDS[8], GRIDS[11]])
def test_sweep_counts_match_the_oracle(tmp_path, per, n, check):
    """`check` sweeps of the L2 modes: FP64 bitwise, FP32 to rounding."""
    from ib3d_amd.native import IB3DError
    s, o = _pair(tmp_path, per, n)
    try:
        s.computeDiv()
        o.compute_div()
        for mode in (1, 2):
            print(f"[gpu] blocks {n} mode {mode} check {check}", flush=True)
            s.set_poisson_mode(mode, omega=1.9, tol=1e-30, check=check, max_sweeps=check)
            with pytest.raises(IB3DError, match="sweep cap"):
                s.poissonSolver()
            if mode == 1:
                o.array("pc")[:] = 0.0
                o.sor_l2(1.9, 1e-30, check, check)
                ref = o.array("pc").copy()
                assert _same(s.download("pc"), ref)
            else:
                # a sweep is about 20 roundings of 2^-24 per value, of which the
                # relaxation (omega 1.9) carries less than twice on: check sweeps
                # stay below 20 x 2 x check x 2^-24 < 2e-5 x the largest value
                err = np.max(np.abs(s.download("pc") - ref)) / np.max(np.abs(ref))
                assert err < 2e-5, err
    finally:
        s.close()
