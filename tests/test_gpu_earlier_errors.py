"""A HIP call of the user's program that failed earlier leaves its error behind.  A
field that comes back or goes over in pieces reports its own outcome, like a small
one; the predictor, which reports the error as every kernel launch does, starts its
next call with clean row counts.  The error is an impossible device number."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _leave_an_error(s):
    assert s.L.hipSetDevice(9999) != 0


@pytest.mark.parametrize("n", [(46, 40, 40), (126, 126, 126), (190, 150, 149)])
def test_transfers_report_their_own_outcome(n):
    from ib3d_amd.native import Solver
    s = Solver(*n)
    try:
        src = np.random.default_rng(1).standard_normal(int(np.prod([k + 2 for k in n])))
        print(f"[gpu] transfers of {src.nbytes} bytes after an error", flush=True)
        s.L.ib3d_sync()
        _leave_an_error(s)
        s.upload("u", src)
        back = s.download("u")
        s.L.hipGetLastError()
        assert back.tobytes() == src.tobytes()
    finally:
        s.close()


def test_predictor_after_a_reported_error(tmp_path):
    from test_gpu_momentum_rows import OUT, _fields

    from ib3d_amd import cases
    from ib3d_amd.native import IB3DError, Solver
    n = (130, 33, 30)
    cfg = cases.CaseConfig("rows", n, (-5.0, -5.0, -5.0), (15.0, 5.0, 5.0), (-1.0, -1.0, -1.0), (2.0, 1.0, 1.0),
                           1.0 / 8, 2, 0.01, shift=(0.0071, -0.0113, 0.0059))
    cases.write_case(cfg, str(tmp_path))
    s = Solver.from_case(str(tmp_path))
    try:
        for f, a in _fields(n, np.random.default_rng(4), True).items():
            s.upload(f, a)

        def predict(variant):
            for f in OUT:
                s.upload(f, np.full(int(np.prod([k + 2 for k in n])), 7.0))
            s.set_momentum_tiles(variant)
            s.nsMomentum()
            return [s.download(f) for f in OUT]
        want = predict(4)
        for _ in range(3):
            print("[gpu] predictor after an error", flush=True)
            for _ in range(2):
                for a, b in zip(want, predict(1)):
                    assert a.tobytes() == b.tobytes()
            _leave_an_error(s)
            with pytest.raises(IB3DError, match="invalid device"):
                s.nsMomentum()
    finally:
        s.set_momentum_tiles(0)
        s.close()
