"""The multigrid levels cycled inside one workgroup where a level has more pairs of
cells than its threads keep in registers (over 2048) and still fits its 64 KB:
36x32x32 with the level 18x16x16 between the finest and 9x8x8, the same with
18x16x16 as the coarsest, and 64x24x24 with 32x12x12 as the coarsest.  Against the
direct solution of the coarsest level, as test_gpu_multigrid_in_kernel has it: with
a relaxation factor of 1e-12 above that level and one Krylov step, pc is a multiple
of P A^-1 R b.

Tolerance: FP32 throughout.  Rounding in the coarsest sweeps is amplified by the
operator's condition number, at most about 4 / (pi / 64)^2 = 1.7e3 for a row of 32
cells with a fixed value at one end: 1.7e3 * 2^-24 = 1e-4, and a few such roundings
per sweep; 1e-3 of the norm of pc.  The coarsest sweeps (relaxation 1.8: an error
falls to about 1 - (pi / 64)^2 * 9 = 0.978 per sweep) leave 1e-9 after 1000."""
import numpy as np
import pytest
from test_gpu_multigrid_in_kernel import _rows
from test_gpu_multigrid_prolongation import _axis

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per,n,levels", [(4, (36, 32, 32), 3), (4, (36, 32, 32), 2), (5, (64, 24, 24), 2)])
def test_correction_is_the_coarse_solution(tmp_path, per, n, levels):
    from ib3d_amd import cases, presets
    from ib3d_amd.native import IB3DError, Solver
    cfg = cases.CaseConfig("inkernel", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / per, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s = Solver.from_case(str(tmp_path))
    try:
        s.set_poisson_mode(4, omega=1.5, tol=1e-6, check=1, warm=False, max_sweeps=1)   # one cycle
        s.set_krylov(1)
        s.set_multigrid(1, 0, 1e-12, 1000, 1.8, levels)
        rng = np.random.default_rng(sum(n))
        vel = {}
        for f in ("ut", "vt", "wt"):
            vel[f] = rng.standard_normal(tuple(m + 2 for m in n))
            s.upload(f, vel[f])
        print(f"[gpu] large in-kernel levels {n}, {levels} levels", flush=True)
        with pytest.raises(IB3DError, match="sweep cap"):
            s.poissonSolver()
        got = s.field("pc")[1:-1, 1:-1, 1:-1]
        solved = [s.field("cell")[1:-1, 1:-1, 1:-1] == 0]
        faces = [s.download(a)[1: m + 2] for a, m in zip(("x1", "y1", "z1"), n)]
        d = [np.diff(f) for f in faces]
        core = np.s_[1:-1, 1:-1, 1:-1]
        b = ((vel["ut"][core] - vel["ut"][:-2, 1:-1, 1:-1]) / d[0][:, None, None]
             + (vel["vt"][core] - vel["vt"][1:-1, :-2, 1:-1]) / d[1][None, :, None]
             + (vel["wt"][core] - vel["wt"][1:-1, 1:-1, :-2]) / d[2][None, None, :])
        for _ in range(levels - 1):   # averages over the cells solved for
            c = [m // 2 for m in b.shape]
            kids = solved[-1].reshape(c[0], 2, c[1], 2, c[2], 2)
            count = kids.sum(axis=(1, 3, 5))
            b = np.where(kids, b.reshape(c[0], 2, c[1], 2, c[2], 2), 0.0).sum(axis=(1, 3, 5)) / np.maximum(count, 1)
            solved.append(count > 0)
        rows = [_rows(faces[a][:: 2 ** (levels - 1)], a == 0) for a in range(3)]
        shape, idx = b.shape, np.indices(b.shape)
        mat = np.zeros(shape + shape)
        for a in range(3):
            west, mid, east = (rows[a][:, k][idx[a]] for k in range(3))
            mat[idx[0], idx[1], idx[2], idx[0], idx[1], idx[2]] += mid
            for step, coef in ((-1, west), (1, east)):
                to = [i.copy() for i in idx]
                to[a] = to[a] + step
                ok = (to[a] >= 0) & (to[a] < shape[a])
                mat[tuple(i[ok] for i in idx) + tuple(i[ok] for i in to)] += coef[ok]
        on = solved[-1].reshape(-1)
        x = np.zeros(b.size)
        x[on] = np.linalg.solve(mat.reshape(b.size, b.size)[np.ix_(on, on)], b.reshape(-1)[on])
        want = x.reshape(shape)
        for lv in range(levels - 2, -1, -1):
            mats = [_axis(faces[a][:: 2 ** lv], faces[a][:: 2 ** (lv + 1)], a == 0) for a in range(3)]
            for a in range(3):
                want = np.moveaxis(np.tensordot(mats[a], want, axes=(1, a)), 0, a)
            want = np.where(solved[lv], want, 0.0)
        got, want = got[solved[0]], want[solved[0]]
        scale = got @ want / (want @ want)
        assert scale != 0.0
        err = np.linalg.norm(got - scale * want) / np.linalg.norm(got)
        print(f"[gpu] error {err:.1e}", flush=True)
        assert err < 1e-3
    finally:
        presets.apply(s, "mixed")
        s.close()
