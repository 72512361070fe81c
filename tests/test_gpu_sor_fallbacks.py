"""The parts of the two-sweep launches that ordinary data does not reach.

Quotients out of the range of the launches' own division (numerators below 2^-900
or above 2^900): the march does the whole chunk again with divisions, the blocks
divide in place; with velocities of 1 in the lower half of the planes and 1e-280 in
the upper one, some chunks do and others do not.  Every value and the iteration
count must be the oracle's, bit for bit.

FP32 increments over several outer iterations: each adds the increment of the one
before to the FP64 unknown.  `check` sweeps of the defect equation from zero are
`check` sweeps of the equation itself, so k outer iterations are k * check FP64
sweeps, to rounding.  A sweep is about 20 roundings of 2^-24 per value of the
increment, of which the relaxation (omega 1.9) carries less than twice on within
the iteration and less than twice through the later ones: together less than
20 x 2 x 2 x check x 2^-24 of the sum of the increments' largest values."""
import numpy as np
import pytest
from test_gpu_sor_blocks import _pair, _same

pytestmark = pytest.mark.gpu

# cells per unit length of the uniform box, and the interior grid: blocks of
# 8 x 8 x 8 and 24 x 16 x 8 cells, march tiles of 36 x 28 and 32 x 32
GRIDS = [(8, (65, 63, 64)), (10, (98, 64, 49)), (12, (121, 113, 112)), (10, (190, 90, 91))]


@pytest.mark.parametrize("scale", [1e-274, 1e-305, 1e268, "mixed"])
@pytest.mark.parametrize("per,n", GRIDS)
def test_extreme_values_match_the_oracle(tmp_path, per, n, scale):
    from ib3d_amd.native import IB3DError
    size = 1.0 if scale == "mixed" else scale
    s, o = _pair(tmp_path, per, n, size)
    try:
        if scale == "mixed":
            for f in ("ut", "vt", "wt"):
                a = np.array(o.field(f))
                a[:, :, n[2] // 2:] *= 1e-280
                o.field(f)[...] = a
                s.upload(f, np.asfortranarray(a))
        s.computeDiv()
        o.compute_div()
        for eps in (2.0 * size, size, 0.6 * size):
            print(f"[gpu] extremes {n} scale={scale} eps={eps}", flush=True)
            it, d2 = s.REDBLACKSOR(eps)
            assert (it, d2) == o.redblack_sor(eps)
            assert _same(s.download("pc"), o.array("pc"))
        if scale == "mixed":   # without the tracking of the stopping rule
            s.set_poisson_mode(1, omega=1.9, tol=1e-30, check=4, max_sweeps=4)
            with pytest.raises(IB3DError, match="sweep cap"):
                s.poissonSolver()
            o.array("pc")[:] = 0.0
            o.sor_l2(1.9, 1e-30, 4, 4)
            assert _same(s.download("pc"), o.array("pc"))
    finally:
        s.close()


@pytest.mark.parametrize("check", [2, 4, 6, 8])
@pytest.mark.parametrize("per,n", [(4, (33, 25, 23)), (8, (65, 63, 64)), (12, (121, 113, 112)), (10, (190, 90, 91))])
def test_increments_of_several_outer_iterations(tmp_path, per, n, check):
    from ib3d_amd.native import IB3DError
    s, o = _pair(tmp_path, per, n)
    try:
        s.computeDiv()
        o.compute_div()
        o.array("pc")[:] = 0.0
        total, before = 0.0, o.array("pc").copy()
        for outer in (1, 2, 3):
            print(f"[gpu] increments {n} check={check} outer={outer}", flush=True)
            o.sor_l2(1.9, 1e-30, check, check)
            now = o.array("pc").copy()
            total += np.max(np.abs(now - before))
            before = now
            s.set_poisson_mode(2, omega=1.9, tol=1e-30, check=check, max_sweeps=outer * check)
            with pytest.raises(IB3DError, match="sweep cap"):
                s.poissonSolver()
            err = np.max(np.abs(s.download("pc") - now))
            assert err < 80.0 * check * 2.0 ** -24 * total, (err, total)
    finally:
        s.close()
