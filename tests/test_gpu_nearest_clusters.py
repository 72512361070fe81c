"""The clustered nearest-element search against the oracle's scan of all
elements: tags and nearest elements must be equal, including the choice of the
first among equally near elements.  Meshes around the cluster size (64), in a
random order, with every triangle twice, and a flat one whose centroids are
equidistant from many cells; after the set-up and after moves of the body."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mesh(kind):
    from ib3d_amd import cases
    rng = np.random.default_rng(11)
    v, f = cases.icosphere(3)
    if kind == "shuffled":
        f = f[rng.permutation(len(f))]
    elif kind == "twice":
        f = np.concatenate([f, f[::-1]])[rng.permutation(2 * len(f))]
    elif kind == "flat":   # a plate of equal triangles on the grid's own spacing
        g = np.arange(-4, 5) * 0.125
        v = np.array([(x, y, 0.0) for x in g for y in g])
        f = np.array([t for a in range(8) for b in range(8)
                      for t in ((9 * a + b, 9 * a + b + 9, 9 * a + b + 10), (9 * a + b, 9 * a + b + 10, 9 * a + b + 1))])
    else:
        f = f[rng.permutation(len(f))[:int(kind)]]
    return v, np.asarray(f, dtype=np.int64)


@pytest.mark.parametrize("kind", ["1", "63", "64", "65", "shuffled", "twice", "flat"])
def test_tags_and_nearest_elements_match_the_oracle(tmp_path, kind):
    from ib3d_amd import cases
    from ib3d_amd.native import Solver
    import pyoracle
    cfg = cases.CaseConfig("clusters", (33, 26, 27), (-3.0, -2.5, -2.5), (5.0, 2.5, 2.5), (-0.75, -0.75, -0.75),
                           (1.25, 0.75, 0.75), 0.125, 2, 0.01, shift=(0.0, 0.0, 0.0))
    cases.write_case(cfg, str(tmp_path))
    v, f = _mesh(kind)
    cases.write_gmsh(os.path.join(str(tmp_path), "geometries", "sphere.msh"), v, f, cfg.n_points)
    s, o = Solver.from_case(str(tmp_path)), pyoracle.Oracle.from_case(str(tmp_path))
    try:
        np.testing.assert_array_equal(s.download("cell"), o.array("cell"))
        np.testing.assert_array_equal(s.download("minElemcell"), o.array("minElemcell"))
        for q in range(1, 4):
            print(f"[gpu] clusters {kind} move {q}", flush=True)
            d = (0.03 * q, -0.02 * q, 0.01 * q)
            s.move_body(d)
            o.move_body(d)
            np.testing.assert_array_equal(s.download("cell"), o.array("cell"))
            np.testing.assert_array_equal(s.download("minElemcell"), o.array("minElemcell"))
            np.testing.assert_array_equal(s.download("interceptedIndexPtr"), o.array("interceptedIndexPtr"))
    finally:
        s.close()
