"""Overlapped scan calls that outgrow the handle's buffers (runs on an MI355X).

With overlap on, a scan's neighbourhood metrics still run on the stage's stream when the call
returns.  A larger scan right after it, without a combine in between, moves the slot records those
metrics write and the work buffers they read, so the move has to follow them.  Scans that grow
from call to call, alone and as batches, must leave what the same scans leave without overlap.
"""
import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu


def _scan(rng, n):
    az, el, r = rng.uniform(0, 2 * np.pi, n), rng.uniform(-0.4, 0.4, n), rng.uniform(1.5, 20.0, n)
    return np.stack([r * np.cos(el) * np.cos(az), r * np.cos(el) * np.sin(az), r * np.sin(el)], 1).astype(np.float32)


def _same(a, b, label):
    for slot in range(a.buffer_size):
        s, t = a.slot_state(slot), b.slot_state(slot)
        assert (s is None) == (t is None), f"{label} slot {slot}"
        for k in s or {}:
            assert np.array_equal(s[k], t[k]), f"{label} slot {slot} {k}"
    s, t = a.combined_state(), b.combined_state()
    for k in s:
        assert np.array_equal(s[k], t[k], equal_nan=True), f"{label} combined {k}"


@pytest.mark.parametrize("batch", [1, 2])
def test_growing_scans(batch):
    import gvom
    import gvom_native as nat
    rng = np.random.default_rng(batch)
    args = synth.gvom_args(0.4, 0.2, 128, 32, 6)
    ovl, serial = gvom.Gvom(*args), gvom.Gvom(*args)
    ovl.set_overlap(True)
    sizes = [3000, 9000, 26000, 60000]      # past twice the capacity before, each time
    clouds = [np.concatenate([_scan(rng, n) for _ in range(batch)]) for n in sizes]
    dev = [nat.DeviceArray(c) for c in clouds]
    for g in (ovl, serial):
        for k, n in enumerate(sizes):
            ego = np.array([[0.1 + 0.4 * k + 0.2 * b, -0.1, 0.3] for b in range(batch)])
            if batch == 1:
                g.process_pointcloud_device(dev[k], n, ego[0])
            else:
                g.process_batch_device(dev[k], np.arange(batch + 1) * n, ego)
            if k == 2:
                g.combine_maps_device()
        g.combine_maps_device()
    _same(ovl, serial, f"batch {batch}")
