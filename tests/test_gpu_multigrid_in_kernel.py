"""The multigrid levels cycled inside one workgroup, against a direct solution.
With a relaxation factor of 1e-12 above the coarsest level, enough sweeps on it,
and one Krylov step, the correction pc is a multiple of P A^-1 R b: the right-hand
side averaged down over the cells solved for, solved on the coarsest level,
interpolated up.  The grids make the levels' cells fit one wave with and without a
remainder, need the whole workgroup once or twice per thread, and have an odd or a
two-cell row on the coarsest level.

Tolerance: FP32 throughout.  Rounding in the coarsest sweeps is amplified by the
operator's condition number, at most about 1e3 on these levels: 1e3 * 2^-24 =
6e-5, and a few such roundings per sweep; 1e-3 of the norm of pc."""
import numpy as np
import pytest

from test_gpu_multigrid_prolongation import _axis

pytestmark = pytest.mark.gpu


def _rows(faces, x_axis):
    """Laplacian rows (west, centre, east) of an axis with the given faces."""
    n = faces.size - 1
    f = np.concatenate([[2 * faces[0] - faces[1]], faces, [2 * faces[-1] - faces[-2]]])
    c = 0.5 * (f[:-1] + f[1:])          # centres of padded cells 0..n+1
    r1, r2 = c[1:-1] - c[:-2], c[2:] - c[1:-1]
    a = np.stack([2 / (r1 * (r1 + r2)), -2 / (r1 * r2), 2 / (r2 * (r1 + r2))], axis=1)
    a[0, 1] += a[0, 0]
    a[0, 0] = 0
    a[n - 1, 1] += -a[n - 1, 2] if x_axis else a[n - 1, 2]
    a[n - 1, 2] = 0
    return a


@pytest.mark.parametrize("per,n,levels", [(2, (20, 12, 12), 2), (4, (32, 24, 24), 2), (4, (36, 20, 16), 3),
                                          (2, (8, 12, 12), 3), (2, (32, 16, 16), 3)])
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
        s.set_multigrid(1, 0, 1e-12, 1000, 1.5, levels)
        rng = np.random.default_rng(sum(n))
        vel = {}
        for f in ("ut", "vt", "wt"):
            vel[f] = rng.standard_normal(tuple(m + 2 for m in n))
            s.upload(f, vel[f])
        print(f"[gpu] in-kernel levels {n}, {levels} levels", flush=True)
        with pytest.raises(IB3DError, match="sweep cap"):
            s.poissonSolver()
        pc = s.field("pc")[1:-1, 1:-1, 1:-1]
        solved = s.field("cell")[1:-1, 1:-1, 1:-1] == 0
        fluid = solved
        faces = [s.download(a)[1: m + 2] for a, m in zip(("x1", "y1", "z1"), n)]
        d = [np.diff(f) for f in faces]
        core = np.s_[1:-1, 1:-1, 1:-1]
        b = ((vel["ut"][core] - vel["ut"][:-2, 1:-1, 1:-1]) / d[0][:, None, None]
             + (vel["vt"][core] - vel["vt"][1:-1, :-2, 1:-1]) / d[1][None, :, None]
             + (vel["wt"][core] - vel["wt"][1:-1, 1:-1, :-2]) / d[2][None, None, :])
        up = None
        for lv in range(levels - 1):
            mats = [_axis(faces[a][:: 2 ** lv], faces[a][:: 2 ** (lv + 1)], a == 0) for a in range(3)]
            q = np.einsum("ia,jb,kc->ijkabc", *mats).reshape(solved.size, -1)
            q[~solved.reshape(-1)] = 0.0
            up = q if up is None else up @ q
            c = [m // 2 for m in solved.shape]
            kids = solved.reshape(c[0], 2, c[1], 2, c[2], 2)
            count = kids.sum(axis=(1, 3, 5))
            b = np.where(kids, b.reshape(c[0], 2, c[1], 2, c[2], 2), 0.0).sum(axis=(1, 3, 5)) / np.maximum(count, 1)
            solved = count > 0
        rows = [_rows(faces[a][:: 2 ** (levels - 1)], a == 0) for a in range(3)]
        shape = solved.shape
        mat = np.zeros(shape + shape)
        idx = np.indices(shape)
        for a in range(3):
            west, mid, east = (rows[a][:, k][idx[a]] for k in range(3))
            mat[idx[0], idx[1], idx[2], idx[0], idx[1], idx[2]] += mid
            for step, coef in ((-1, west), (1, east)):
                to = [i.copy() for i in idx]
                to[a] = to[a] + step
                ok = (to[a] >= 0) & (to[a] < shape[a])
                mat[tuple(i[ok] for i in idx) + tuple(i[ok] for i in to)] += coef[ok]
        mat = mat.reshape(solved.size, solved.size)
        on = solved.reshape(-1)
        x = np.zeros(solved.size)
        x[on] = np.linalg.solve(mat[np.ix_(on, on)], b.reshape(-1)[on])
        want = (up @ x)[fluid.reshape(-1)]
        got = pc.reshape(-1)[fluid.reshape(-1)]
        scale = got @ want / (want @ want)
        assert scale != 0.0
        assert np.linalg.norm(got - scale * want) < 1e-3 * np.linalg.norm(got)
    finally:
        presets.apply(s, "mixed")
        s.close()
