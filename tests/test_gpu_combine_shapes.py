"""The combine at the sizes where its table and cell passes have their edges, against the oracle.

Heights below, at and past a lane's eight voxels and a 64-bit occupancy word, column counts that
leave the last wavefront and block partly empty or are the last that take the one-kernel cell pass
(256 x 256) and the first that do not, rings of one slot to past a group of loads, and
an ego that moves by several voxels in x, y and z between scans, back and forth and far enough
for slots to leave the map altogether.
"""
import numpy as np
import pytest

import gvom_synth as synth
from oracle.gvom_oracle import OracleGvom
from parity import assert_equal, compare_combined, compare_maps

pytestmark = pytest.mark.gpu

# voxels moved per scan (x, y, z)
MOVES = [(0, 0, 0), (1, 0, 0), (-3, 2, 1), (0, 0, -1), (5, -7, 3), (0, 0, 0), (-2, 1, -6), (40, 3, 0)]


@pytest.mark.parametrize("xy,z,buffer", [
    (4, 4, 1), (5, 7, 2), (16, 8, 4), (37, 9, 5), (30, 16, 8), (33, 60, 3), (24, 63, 4), (20, 64, 9), (21, 65, 2),
    (17, 100, 3), (9, 128, 4), (12, 250, 1), (11, 256, 30), (130, 30, 3), (256, 5, 2), (257, 6, 2),
])
def test_combine_shapes(xy, z, buffer):
    import gvom
    args = synth.gvom_args(0.4, 0.2, xy, z, buffer)
    rng = np.random.default_rng(xy * 1000 + z)
    g, o = gvom.Gvom(*args), OracleGvom(*args)
    ego = np.array([0.1, -0.1, 0.3])
    for k, mv in enumerate(MOVES):
        ego = ego + np.array(mv) * np.array([0.4, 0.4, 0.2])
        n = 60 * xy
        half = np.array([0.2 * xy, 0.2 * xy, 0.1 * z]) * 1.1
        pts = (ego + rng.uniform(-1, 1, (n, 3)) * half).astype(np.float32)
        pts[: n // 3] = np.round(pts[: n // 3] / 0.4) * 0.4 + 0.13     # several points per voxel
        g.Process_pointcloud(pts, ego, None)
        o.Process_pointcloud(pts, ego, None)
        if k == 2:
            continue                                                    # two scans, one combine
        a, b = g.combine_maps(), o.combine_maps()
        label = f"{xy}x{xy}x{z} buffer {buffer} frame {k}"
        compare_combined(g.combined_state(), o.combined, label)
        compare_maps(g.maps_state(), o.combined, label)
        for name, j in (("positive", 1), ("negative", 2), ("visibility", 4)):
            assert_equal(f"{label} {name}", a[j], b[j])
