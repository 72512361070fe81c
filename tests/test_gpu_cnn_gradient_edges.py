"""The weight-gradient kernel where its chunks of 32 voxels, its columns of
rows and its split over workgroups end: single voxels, rows one short of and one
past a chunk, columns that a workgroup starts or leaves in the middle, and a
volume whose last workgroups have no chunk left.  Against the FP64 oracle that
rounds what the GPU stores in BF16.

Tolerance: both sides round the same quantities, so they differ by FP32 sums and
by stored values that fall on the other side of a BF16 rounding (2^-8 of the
value).  A gradient passes through at most three stored layers, so even if every
value fell the other way an entry would move by 3 * 2^-8 = 1.2e-2 of its terms;
few do, so 1e-2 of a layer's largest entry bounds it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def net():
    from ib3d_amd.native import Net, Solver
    s = Solver(8, 8, 8)
    n = Net(seed=5)
    yield n
    n.release()
    s.close()


# (volumes, z, y, x)
SHAPES = [(1, 1, 1, 1), (1, 2, 1, 31), (2, 3, 2, 32), (1, 1, 3, 33), (3, 5, 4, 64), (1, 2, 67, 65), (1, 9, 233, 97)]


@pytest.mark.parametrize("shape", SHAPES)
def test_gradient_at_the_edges(net, shape):
    import cnn_oracle as co
    print(f"[gpu] cnn gradient {shape}", flush=True)
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal(shape + (3,)).astype(np.float32)
    dy = rng.standard_normal(shape).astype(np.float32)
    g = net.gradient(x, dy).astype(np.float64)
    again = net.gradient(x, dy)
    np.testing.assert_array_equal(g, again)
    ref = co.gradient(net.params(), x, dy, bf16=True)
    for layer in range(4):
        for part in co.SLICES[layer]:
            err = np.max(np.abs(g[part] - ref[part])) / max(np.max(np.abs(ref[part])), 1e-30)
            assert err < 1e-2, (layer, err)
