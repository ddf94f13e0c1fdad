"""gvom_autotune and the azimuth-ordered cast (runs on an MI355X).

A scan below that cast's line cannot be used to time it, so tuning on one leaves the setting
(flag bit 4) as it is, on or off.  After tuning on a scan above the line, which counts azimuth bins
with the cast's own buffers, frames cast in azimuth order equal those of a handle that was never
tuned.
"""
import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu

AZIMUTH = 16


def _scan(rng, n):
    az, el, r = rng.uniform(0, 2 * np.pi, n), rng.uniform(-0.4, 0.4, n), rng.uniform(1.5, 60.0, n)
    return np.stack([r * np.cos(el) * np.cos(az), r * np.cos(el) * np.sin(az), r * np.sin(el)], 1).astype(np.float32)


@pytest.mark.parametrize("on", [True, False])
def test_small_scan_keeps_the_setting(on):
    import gvom
    import gvom_native as nat
    g = gvom.Gvom(*synth.gvom_args(0.4, 0.2, 64, 32, 2))
    if not on:
        g.set_raycast_config(128, 1, False, False, True, True, False)
    pts = nat.DeviceArray(_scan(np.random.default_rng(1), 5000))
    flags = g.autotune(pts, 5000, (0.1, -0.1, 0.3))[2]
    assert bool(flags & AZIMUTH) == on, flags


def test_frames_after_tuning_on_a_large_scan():
    import gvom
    import gvom_native as nat
    n, xy = 60_001, 256   # 15.4e6, above the line
    args = synth.gvom_args(0.4, 0.2, xy, 64, 2)
    rng = np.random.default_rng(2)
    scans = [_scan(rng, n) for _ in range(3)]
    dev = [nat.DeviceArray(s) for s in scans]
    tuned, plain = gvom.Gvom(*args), gvom.Gvom(*args)
    tuned.autotune(dev[0], n, (0.1, -0.1, 0.3))
    block, rpt = 128, 1
    tuned.set_raycast_config(block, rpt, False, False, False, False, True)
    plain.set_raycast_config(block, rpt, False, False, False, False, False)
    for k in range(3):
        ego = np.array([0.1 + 0.5 * k, -0.1, 0.3])
        for g in (tuned, plain):
            g.process_pointcloud_device(dev[k], n, ego)
            g.combine_maps_device()
        for slot in range(args[4]):
            a, b = tuned.slot_state(slot), plain.slot_state(slot)
            assert (a is None) == (b is None), f"frame {k} slot {slot}"
            for f in a or {}:
                assert np.array_equal(a[f], b[f]), f"frame {k} slot {slot} {f}"
        a, b = tuned.combined_state(), plain.combined_state()
        for f in a:
            assert np.array_equal(a[f], b[f], equal_nan=True), f"frame {k} combined {f}"
