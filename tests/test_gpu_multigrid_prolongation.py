"""The prolongation of the multigrid levels cycled by launches, by its range: with
a relaxation factor of 1e-12 above the coarsest level and one Krylov step, the
correction pc is a multiple of the interpolant P x of the coarsest level's
solution, on the cells each level solves for.  P is formed here from the grid lines (linear between
coarse centres, constant beyond the last, antisymmetric at the outlet), and pc
must lie in its range.

Tolerance: an interpolant is a sum of eight products per level, each of a few FP32
roundings: at most 8 * 2^-24 = 4.8e-7 of sum |w x| per level, which is a few times
|sum w x|; 4e-6 of the norm of pc.  A wrong weight or neighbour anywhere is off by
1e-3 or more."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _axis(fine, coarse, outlet):
    """Interpolation matrix from coarse to fine cell centres (faces given)."""
    def centres(f):
        c = np.empty(f.size + 1)
        c[1:-1] = 0.5 * (f[:-1] + f[1:])
        c[0] = f[0] - 0.5 * (f[1] - f[0])
        c[-1] = f[-1] + 0.5 * (f[-1] - f[-2])
        return c
    xf, xc = centres(fine), centres(coarse)
    nf, nc = fine.size - 1, coarse.size - 1
    m = np.zeros((nf, nc))
    for i in range(1, nf + 1):
        own = (i + 1) // 2
        other = own - 1 if xf[i] < xc[own] else own + 1
        w = (xf[i] - xc[other]) / (xc[own] - xc[other])
        m[i - 1, own - 1] += w
        if 1 <= other <= nc:
            m[i - 1, other - 1] += 1.0 - w
        else:
            m[i - 1, own - 1] += -(1.0 - w) if other > nc and outlet else 1.0 - w
    return m


@pytest.mark.parametrize("n,levels", [((26, 16, 18), 2), ((28, 18, 16), 2), ((34, 20, 22), 2), ((32, 16, 20), 3),
                                      ((36, 20, 16), 3)])
def test_correction_lies_in_the_range_of_the_interpolation(tmp_path, n, levels):
    from ib3d_amd import cases
    from ib3d_amd.native import IB3DError, Solver
    cfg = cases.CaseConfig("prolong", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / 4, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s = Solver.from_case(str(tmp_path))
    try:
        s.set_poisson_mode(4, omega=1.5, tol=1e-6, check=1, warm=False, max_sweeps=1)   # one cycle
        s.set_krylov(1)
        s.set_multigrid(1, 0, 1e-12, 6, 1.2, levels)
        rng = np.random.default_rng(sum(n))
        for f in ("ut", "vt", "wt"):
            s.upload(f, rng.standard_normal(s.download(f).size))
        print(f"[gpu] prolongation {n}, {levels} levels", flush=True)
        with pytest.raises(IB3DError, match="sweep cap"):
            s.poissonSolver()
        pc = s.field("pc")[1:-1, 1:-1, 1:-1]
        fluid = s.field("cell")[1:-1, 1:-1, 1:-1] == 0
        faces = [s.download(a)[1: m + 2] for a, m in zip(("x1", "y1", "z1"), n)]
        p, solved = None, fluid   # a coarse cell is solved for if one of its eight is
        for lv in range(levels - 1):
            mats = [_axis(faces[a][:: 2 ** lv], faces[a][:: 2 ** (lv + 1)], a == 0) for a in range(3)]
            q = np.einsum("ia,jb,kc->ijkabc", *mats).reshape(solved.size, -1)
            q[~solved.reshape(-1)] = 0.0
            p = q if p is None else p @ q
            c = [m // 2 for m in solved.shape]
            solved = solved.reshape(c[0], 2, c[1], 2, c[2], 2).any(axis=(1, 3, 5))
        p = p[fluid.reshape(-1)]
        v = pc.reshape(-1)[fluid.reshape(-1)]
        assert np.linalg.norm(v) > 0.0
        x = np.linalg.lstsq(p, v, rcond=None)[0]
        assert np.linalg.norm(p @ x - v) < 4e-6 * np.linalg.norm(v)
    finally:
        from ib3d_amd import presets
        presets.apply(s, "mixed")
        s.close()
