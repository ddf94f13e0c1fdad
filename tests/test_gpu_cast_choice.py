"""Which ray cast a scan takes (runs on an MI355X): the casts leave the same counts, so tests that
compare counts cannot tell.  Both sides of the azimuth order's line (12e6 points x xy_size), every
setting, and each way a scan comes in: alone, in a batch, replayed, allocation-free, recorded."""
import ctypes

import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu

XY = 64
LINE = 187_500     # x 64 = 12e6
EGO = np.array([0.1, -0.1, 0.3])


@pytest.fixture(scope="module")
def points():
    rng = np.random.default_rng(3)
    az, el, r = (rng.uniform(0, 2 * np.pi, LINE), rng.uniform(-0.4, 0.4, LINE), rng.uniform(1.5, 20.0, LINE))
    return np.stack([r * np.cos(el) * np.cos(az), r * np.cos(el) * np.sin(az), r * np.sin(el)], 1).astype(np.float32)


def _mapper(buffer=2):
    import gvom
    return gvom.Gvom(*synth.gvom_args(0.4, 0.2, XY, 32, buffer))


@pytest.mark.parametrize("config,small,large", [
    (None, "tiled", "azimuth"),                                       # a new handle
    (dict(block=256), "tiled", "azimuth"),
    (dict(tiled=False), "direct", "direct"),
    (dict(tiled=False, azimuth=True), "direct", "azimuth"),
    (dict(tiled=True), "tiled", "tiled"),
    (dict(use_box=True, tiled=False), "direct", "direct"),
    (dict(azimuth=False), "tiled", "tiled"),
])
def test_line(points, config, small, large):
    g = _mapper()
    assert g.last_cast() == "none"
    if config is not None:
        g.set_raycast_config(**config)
    for n, expect in ((LINE - 1, small), (LINE, large), (1, small), (0, small)):
        g.Process_pointcloud(points[:n], EGO, None)
        assert g.last_cast() == expect, (n, g.last_cast())


def test_batches_count_all_points(points):
    g = _mapper(4)
    for split, expect in (((LINE - 10, 9), "tiled"), ((100_000, 87_500), "azimuth"), ((0, LINE), "azimuth")):
        off = np.cumsum([0, *split])
        g.process_batch(points[:off[-1]], off, np.stack([EGO, EGO]), None)
        assert g.last_cast() == expect, split


def test_replayed_and_recorded_scans(points):
    import gvom_native as nat
    g = _mapper()
    dev = nat.DeviceArray(points)
    for k in range(4):      # the third and fourth are replayed
        g.Process_pointcloud(points, EGO, None)
    assert g.last_cast() == "azimuth"
    for k in range(4):
        g.Process_pointcloud(points[:1000], EGO, None)
    assert g.last_cast() == "tiled"
    g.process_pointcloud_device(dev, LINE, EGO)
    assert g.last_cast() == "azimuth"
    g.Process_pointcloud(points[:1000], EGO, None)
    assert g.last_cast() == "tiled"
    g.graph_begin(1)
    g.process_pointcloud_device(dev, LINE, EGO)
    graph = g.graph_end()
    assert g.last_cast() == "azimuth"
    del graph


def test_allocation_free_scans(points):
    import gvom
    import gvom_native as nat
    n = 125_000                      # x 96 = 12e6
    g = gvom.Gvom(*synth.gvom_args(0.4, 0.2, 96, 20, 2))
    dev = nat.DeviceArray(points)
    g.reserve(n, n)
    for count, expect in ((n, "azimuth"), (n - 1, "tiled")):
        nat.check(g._lib.gvom_process_pointcloud_device_noalloc(g._h, dev.ptr, count, nat.GVOM_F32, nat.ptr(EGO), None,
                                                                nat.GVOM_NO_TRANSFORM), g._h)
        assert g.last_cast() == expect
    g.sync()


def test_tuning_on_a_small_scan_leaves_large_ones_alone(points):
    import gvom_native as nat
    g = _mapper()
    dev = nat.DeviceArray(points)
    g.autotune(dev, 5000, EGO)
    g.process_pointcloud_device(dev, LINE, EGO)
    assert g.last_cast() == "azimuth"
