"""The first scan through the tiled cast's scratch with overlap on (runs on an MI355X).

That call allocates the scratch and zeroes it on the main stream, and its stage, on another stream,
counts into it: on memory that held something else before, the counts must be those of a handle
without overlap."""
import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("buffer", [2, 8])
def test_first_overlapped_scan(buffer):
    import gvom
    import gvom_native as nat
    rng = np.random.default_rng(buffer)
    n = 20_000
    az, el, r = rng.uniform(0, 2 * np.pi, n), rng.uniform(-0.4, 0.4, n), rng.uniform(1.5, 40.0, n)
    pts = np.stack([r * np.cos(el) * np.cos(az), r * np.cos(el) * np.sin(az), r * np.sin(el)], 1).astype(np.float32)
    dev = nat.DeviceArray(pts)
    args = synth.gvom_args(0.4, 0.2, 160, 48, buffer)
    ovl, serial = gvom.Gvom(*args), gvom.Gvom(*args)
    ovl.set_overlap(True)
    words = 160 * 160 * 48 * buffer
    used = [nat.DeviceArray(np.full(words, 7, np.int32)) for _ in range(2)]
    del used
    for g in (ovl, serial):
        g.set_raycast_config(128, 1, False, False, True, True, False)
        for k in range(3):
            g.process_pointcloud_device(dev, n, np.array([0.1 + 0.4 * k, -0.1, 0.3]))
    for slot in range(buffer):
        a, b = ovl.slot_state(slot), serial.slot_state(slot)
        assert (a is None) == (b is None), slot
        for f in a or {}:
            assert np.array_equal(a[f], b[f]), f"slot {slot} {f}"
