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
