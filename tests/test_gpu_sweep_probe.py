"""The sweep probe (ib3d_bench_sor) in every form, on a grid of blocks and on one
of the march: it returns a time, refuses other precisions, and the solves after it
are, bit for bit, those of a run without it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(case, mode, probe):
    from ib3d_amd import presets
    from ib3d_amd.native import IB3DError, Solver
    s = Solver.from_case(case)
    try:
        presets.apply(s, mode)
        s.step()
        if probe:
            pc = s.download("pc")
            for precision in (32, 33, 34, 64, 65):
                for sweeps in (1, 6, 7):
                    assert s.bench_sor(precision, sweeps, 1.5) > 0.0
            with pytest.raises(IB3DError, match="precision"):
                s.bench_sor(35, 4, 1.5)
            s.upload("pc", pc)
        s.step()
        return [s.download(f) for f in ("u", "v", "w", "p", "pc")]
    finally:
        s.close()


@pytest.mark.parametrize("mode", ["mixed", "fp64"])
@pytest.mark.parametrize("name", ["cfg1", "cfg2"])
def test_probe_leaves_the_solver_alone(case_dir, name, mode):
    print(f"[gpu] sweep probe {name} {mode}", flush=True)
    case = case_dir(name)
    for a, b in zip(_run(case, mode, False), _run(case, mode, True)):
        assert np.array_equal(a.view(np.int64), b.view(np.int64))
