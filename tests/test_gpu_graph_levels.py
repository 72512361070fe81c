"""The captured Krylov cycle goes with the multigrid levels it was captured with:
changing the number of levels frees and reallocates every level's buffers, also
where the hierarchy stays the same (an explicit count equal to the one found), and
the next solve captures again.  The same launches in the same order, so every field
has the bits of the run without graphs."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEVELS = (0, 5, 5, 0, 3, 5, 0)   # 48x32x32 halves four times: 0 (no limit) and 5 are the same hierarchy


def _run(case, graphs):
    from ib3d_amd.native import Solver
    s = Solver.from_case(case)
    try:
        s.set_poisson_mode(4, tol=1e-6, warm=True)
        s.set_krylov(6)
        s.set_graphs(graphs)
        out = []
        for q, levels in enumerate(LEVELS):
            s.set_multigrid(4, 4, 1.55, 4, 1.5, levels)
            print(f"[gpu] graphs={graphs} step {q + 1}: max_levels {levels}", flush=True)
            s.step()
            out.append([s.download(f).copy() for f in ("u", "v", "w", "p")])
    finally:
        s.close()
    return out


def test_levels_change_between_replays(case_dir):
    case = case_dir("small")
    eager, graph = _run(case, False), _run(case, True)
    for q, (a, b) in enumerate(zip(eager, graph)):
        for name, x, y in zip("uvwp", a, b):
            assert np.array_equal(x.view(np.int64), y.view(np.int64)), f"{name} differs after step {q + 1}"
