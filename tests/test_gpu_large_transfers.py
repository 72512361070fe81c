"""Fields large enough for the staged transfers (downloads from 2 MB, uploads
from 32 MB): sizes that end inside a piece, on a piece and after more pieces
than the ring holds, offsets that are 8 but not 16 bytes from an aligned
address, and repeated calls over the same ring.  What comes back is compared
byte for byte."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# bytes of a field around: 2 MB, whole 1 MB pieces (62*62*32 + 2 halves), the
# ring of 16 MB, the upload's 32 MB and a ragged one past it
GRIDS = [(62, 62, 60), (62, 62, 62), (126, 126, 126), (158, 126, 126), (190, 150, 149), (163, 161, 157)]


@pytest.mark.parametrize("n", GRIDS)
def test_fields_come_back_as_they_went(n):
    from ib3d_amd.native import Solver
    s = Solver(*n)
    try:
        count = int(np.prod([m + 2 for m in n]))
        print(f"[gpu] transfers of {count * 8} bytes", flush=True)
        rng = np.random.default_rng(count)
        src = {a: rng.standard_normal(count) for a in ("u", "v")}
        for a in src:
            s.upload(a, src[a])
        for _ in range(2):
            for a in src:
                assert s.download(a).tobytes() == src[a].tobytes()
        wide = np.zeros(count + 1)
        wide[1:] = src["u"]
        s.upload("v", wide[1:])     # host memory off by 8 bytes
        assert s.download("v").tobytes() == src["u"].tobytes()
    finally:
        s.close()


def test_pinned_and_tag_arrays():
    import ctypes

    from ib3d_amd.native import Solver
    n = (126, 126, 126)
    s = Solver(*n)
    try:
        count = 128 ** 3
        src = np.random.default_rng(3).standard_normal(count)
        s.upload("u", src)
        pinned = ctypes.c_void_p()   # (the runtime that the library loaded)
        assert s.L.hipHostMalloc(ctypes.byref(pinned), ctypes.c_size_t(count * 8), ctypes.c_uint(0)) == 0
        assert s.L.ib3d_download(b"u", pinned, ctypes.c_int64(count * 8)) == 0
        assert ctypes.string_at(pinned, count * 8) == src.tobytes()
        assert s.L.hipHostFree(pinned) == 0
        tags = (np.arange(count) % 3).astype(np.int64)
        s.upload("cell", tags)
        np.testing.assert_array_equal(s.download("cell"), tags)
    finally:
        s.close()
