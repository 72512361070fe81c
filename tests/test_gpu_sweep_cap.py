"""The reference rule stopped by the sweep cap: the solve fails, and pc holds the
sweep at which it gave up.  The cap is looked at after batches of 32, 64, 128 and
then 256 sweeps, so that sweep is the first of their sums above max_sweeps.  The
oracle does that many sweeps from the same pc; every value must have its bits,
and so must those of a solve that goes on from there."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# cells per unit length of the uniform box, and the interior grid: the three
# block shapes and both tiles of the march
GRIDS = [(4, (33, 25, 23)), (8, (65, 63, 64)), (10, (98, 64, 49)), (12, (121, 113, 112)), (10, (190, 90, 91))]


def _sweeps_at_cap(max_sweeps):
    done, batch = 0, 32
    while done <= max_sweeps:
        done, batch = done + batch, min(2 * batch, 256)
    return done


@pytest.mark.parametrize("max_sweeps", [1, 32, 100])
@pytest.mark.parametrize("per,n", GRIDS)
def test_pc_holds_the_last_sweep(tmp_path, per, n, max_sweeps):
    from ib3d_amd import cases
    from ib3d_amd.native import IB3DError, Solver
    import pyoracle
    cfg = cases.CaseConfig("cap", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / per, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s, o = Solver.from_case(str(tmp_path)), pyoracle.Oracle.from_case(str(tmp_path))
    try:
        rng = np.random.default_rng(5)
        for f in ("ut", "vt", "wt"):
            a = np.asfortranarray(rng.standard_normal(tuple(k + 2 for k in n)))
            s.upload(f, a)
            o.field(f)[...] = a
        s.computeDiv()
        o.compute_div()
        s.set_poisson_mode(0, max_sweeps=max_sweeps)
        print(f"[gpu] sweep cap {n} max_sweeps={max_sweeps}", flush=True)
        # (twice: the second solve starts where the first gave up, and queues
        # its batches by the same rule)
        for _ in range(2):
            with pytest.raises(IB3DError, match="sweep cap"):
                s.REDBLACKSOR(1e-30)
            cap = _sweeps_at_cap(max_sweeps)
            o.sor_l2(1.99, 1e-300, cap, cap)
            assert np.array_equal(s.download("pc").view(np.int64), o.array("pc").view(np.int64))
        s.set_poisson_mode(0)
        o.array("pco")[:] = o.array("pc")   # (which the oracle's loop starts from, and sor_l2 leaves behind)
        eps = 0.5 * np.max(np.abs(o.array("pc")))
        assert s.REDBLACKSOR(eps) == o.redblack_sor(eps)
        assert np.array_equal(s.download("pc").view(np.int64), o.array("pc").view(np.int64))
    finally:
        s.close()
