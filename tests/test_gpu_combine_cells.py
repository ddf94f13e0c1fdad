"""The combine's one-kernel cell pass where its division of the work has its edges.

Ids are dealt out evenly over the threads and looked up through prefix sums of column groups, so
the cases are: more cells than the grid has threads, whole columns (every height of one column
occupied) beside empty ones, groups of 8 columns (the tallest maps) to 64 (the lowest), numbers of
groups at and around powers of four, the last of a wavefront each and the greatest one, a single cell in the first and in the last
column, and no cell at all.  Against the oracle.

The last test pins what the even division is for: the pass must not take longer when the same number
of cells fills whole columns (a wall) than when the cells are spread over the map.
"""
import numpy as np
import pytest

import gvom_synth as synth
from oracle.gvom_oracle import OracleGvom
from parity import compare_combined, compare_maps

pytestmark = pytest.mark.gpu

RES = np.array([0.4, 0.4, 0.2])


def _voxel_points(ego, xy, z, vox):
    """The centres of map voxels (rows of x, y, z indices) around the ego."""
    origin = np.floor(ego / RES - np.array([xy, xy, z]) / 2.0)
    return ((origin + vox + 0.5) * RES).astype(np.float32)


def _frames(xy, z, vox, frames=2, buffer=2, ego=(0.1, -0.1, 0.3)):
    import gvom
    args = synth.gvom_args(0.4, 0.2, xy, z, buffer)
    g, o = gvom.Gvom(*args), OracleGvom(*args)
    ego = np.array(ego)
    for k in range(frames):
        pts = _voxel_points(ego, xy, z, vox)
        g.Process_pointcloud(pts, ego, None)
        o.Process_pointcloud(pts, ego, None)
        g.combine_maps()
        o.combine_maps()
        label = f"{xy}x{xy}x{z} frame {k}"
        compare_combined(g.combined_state(), o.combined, label)
        compare_maps(g.maps_state(), o.combined, label)
    return len(o.combined.hit)


def _random(rng, xy, z, n):
    return np.stack([rng.integers(0, xy, n), rng.integers(0, xy, n), rng.integers(0, z, n)], 1)


def test_more_cells_than_threads():
    n = _frames(128, 64, _random(np.random.default_rng(1), 128, 64, 300_000))
    assert n > 131_072, n     # the grid's threads: a second round


@pytest.mark.parametrize("xy,z", [(64, 256), (40, 65), (48, 64), (96, 8), (64, 4), (33, 100)])
def test_whole_columns(xy, z):
    """A few full columns (consecutive ones and single ones) among empty ones."""
    cols = [(0, 0), (xy - 1, xy - 1), (xy // 2, 3)] + [(5, y) for y in range(7, min(xy, 27))]
    vox = np.array([(x, y, k) for x, y in cols for k in range(z)])
    _frames(xy, z, vox)


# groups of 4 * (64 // lanes) columns, or 64 // lanes where that is a multiple of 4 and gives at most 2048
@pytest.mark.parametrize("xy,z,groups", [(4, 8, 1), (5, 64, 4), (6, 64, 5), (11, 60, 16), (23, 16, 17), (32, 32, 64),
                                         (46, 16, 67), (33, 72, 39), (128, 64, 2048), (129, 64, 521),
                                         (256, 256, 8192)])
def test_group_counts(xy, z, groups):
    cols = 64 // -(-z // 8)
    if cols % 4 or -(-xy * xy // cols) > 2048:
        cols *= 4
    assert -(-xy * xy // cols) == groups
    _frames(xy, z, _random(np.random.default_rng(xy), xy, z, 40 * xy), frames=1 if z == 256 else 2)


@pytest.mark.parametrize("column", [0, 1])
def test_single_cell(column):
    at = 0 if column == 0 else 36
    assert _frames(37, 20, np.array([[at, at, 19]])) == 1


def test_no_cell():
    assert _frames(37, 20, np.array([[500, 500, 500]])) == 0


def test_time_does_not_follow_the_densest_columns():
    """16,384 cells spread over 256 x 256 columns, and as 256 neighbouring full columns: the cell
    pass (stage 5: ids, records, heights) may take at most twice as long on the wall.  With the
    columns divided over the blocks it took seven times as long (91 against 13 us)."""
    import gvom
    import gvom_native as nat
    import ctypes
    xy, z, n = 256, 64, 16_384
    rng = np.random.default_rng(5)
    spread = _random(rng, xy, z, 4 * n)
    spread = np.unique(spread[np.abs((spread - np.array([xy, xy, z]) / 2) * RES).max(axis=1) > 2.0], axis=0)
    spread = spread[rng.permutation(len(spread))[:n]]
    wall = np.array([(40, y, k) for y in range(256) for k in range(64)])
    assert len(spread) == len(wall) == n
    ego = np.array([0.1, -0.1, 0.3])
    times = {}
    for name, vox in (("spread", spread), ("wall", wall)):
        g = gvom.Gvom(*synth.gvom_args(0.4, 0.2, xy, z, 2))
        pts = _voxel_points(ego, xy, z, vox)
        for k in range(3):
            g.Process_pointcloud(pts, ego, None)
            g.combine_maps()
        assert len(g.combined_state()["hit"]) == n
        best = 1e9
        for k in range(12):
            nat.check(g._lib.gvom_set_timing(g._h, 1), g._h)
            g.Process_pointcloud(pts, ego, None)
            g.combine_maps()
            ms = (ctypes.c_float * 9)()
            nat.check(g._lib.gvom_stage_times(g._h, ms, 9), g._h)
            best = min(best, ms[5])
        times[name] = best * 1000
        del g
    print(f"cell pass, 16,384 cells: spread {times['spread']:.1f} us, wall {times['wall']:.1f} us", flush=True)
    assert times["wall"] < 2.0 * times["spread"], times
