"""Debug clouds, the node's records and occupancy grids through the pinned staging and past its
limit, on odd and smallest map sides: equal to the exported state, bit for bit.
"""
import numpy as np
import pytest

import gvom_synth as synth
from oracle import ros_ref

pytestmark = pytest.mark.gpu

def _map(xy, z):
    import gvom
    base = synth.workload(2).map_args
    return gvom.Gvom(*base[:2], xy, z, 2, *base[5:])


def _points(n, reach, seed):
    rng = np.random.default_rng(seed)
    return np.stack([rng.uniform(-reach, reach, n), rng.uniform(-reach, reach, n), rng.normal(-1, 0.3, n)],
                    1).astype(np.float32)


# 774: the last side whose height map stays below the staging's limit, 775 the first above it
@pytest.mark.parametrize("xy,z", [(4, 4), (63, 5), (151, 70), (774, 4), (775, 4)])
def test_exports_equal_the_state(xy, z):
    import gvom_native as nat
    from gvom_node import HEIGHT_RECORD
    g = _map(xy, z)
    res, zres = g.xy_resolution, g.z_resolution
    for k in range(2):
        g.Process_pointcloud(_points(4000, 0.5 * xy * res, k), (0.3 * k, -0.2, 0.1), None)
        g.combine_maps()
    m, c = g.maps_state(), g.combined_state()
    o = c["origin"]
    y, x = (v.reshape(-1).astype(np.float64) for v in np.mgrid[0:xy, 0:xy])
    flat = {k: v.flatten("F") for k, v in m.items()}
    f32 = np.float32
    fx, fy = f32((x + o[0]) * res), f32((y + o[1]) * res)
    exp = np.stack([fx, fy, f32(flat["height"] - zres), f32(flat["rough"]), f32(flat["slope_x"]),
                    f32(flat["slope_y"]), f32(np.sqrt(flat["slope_x"] ** 2 + flat["slope_y"] ** 2))], 1)
    np.testing.assert_array_equal(g.make_debug_height_map(), exp)
    rec = g.height_map_records(HEIGHT_RECORD)
    np.testing.assert_array_equal(np.stack([rec[n] for n in HEIGHT_RECORD.names[:7]], 1), exp)
    np.testing.assert_array_equal(rec["obstacles"], flat["pos"])
    np.testing.assert_array_equal(g.make_debug_inferred_height_map(), np.stack([fx, fy, f32(flat["delta"] - zres)], 1))
    idx = c["index_map"]
    v = np.flatnonzero(idx >= 0)
    v = v[np.argsort(idx[v])]
    vx, vy, vz = v % xy, (v // xy) % xy, v // (xy * xy)
    ev = c["eigen"]
    vox = np.stack([f32((vx + o[0]) * res), f32((vy + o[1]) * res), f32((vz + o[2]) * zres),
                    f32(c["hit"] / c["total"].astype(np.float64)), f32(c["hit"]), ev[:, 0] - ev[:, 1],
                    ev[:, 1] - ev[:, 2], ev[:, 2]], 1)
    np.testing.assert_array_equal(g.make_debug_voxel_map(), vox)
    got = g.occupancy_grids()
    want = ros_ref.occupancy_payloads(m["pos"], m["neg"], m["rough"], m["vis"], 50, -10, 0)
    for name in nat.GRID_NAMES:
        np.testing.assert_array_equal(got[name], want[name], err_msg=name)
