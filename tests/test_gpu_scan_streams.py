"""Scan stages with their sort chain on one stream or on two give the same state.

Eager calls of scans below the azimuth cast's size keep the sort chain on the stage's own stream;
larger ones, and captured sequences of every size, fork it to the side stream.  Frames issued back
to back, eager (overlap off and on) and captured, must leave the ring, every slot, the combined
map and the 2D maps bit-identical to frames with a synchronisation after every call, on both sides
of the line.
"""
import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu

XY = 128
LINE = 12_000_000 // XY   # the smallest scan that forks in an eager call


def _same(a, b, label):
    assert a.ring_state() == b.ring_state(), label
    pairs = [(a.combined_state(), b.combined_state()), (a.maps_state(), b.maps_state())]
    pairs += [(a.slot_state(s), b.slot_state(s)) for s in range(3)]
    for x, y in pairs:
        assert (x is None) == (y is None), label
        for key in x or ():
            assert np.array_equal(x[key], y[key]), (label, key)


@pytest.mark.parametrize("n", [1, 5000, LINE - 1, LINE])
def test_streams_match_synchronised_frames(n):
    import gvom
    import gvom_native as nat
    base = synth.workload(2).map_args
    args = base[:2] + (XY, 32, 3) + base[5:]
    rng = np.random.default_rng(n)
    pts = [np.stack([rng.normal(0, 12, n), rng.normal(0, 12, n), rng.normal(-1, 0.6, n)], 1).astype(np.float32)
           for _ in range(4)]
    dev = [nat.DeviceArray(p) for p in pts]
    egos = np.array([[0.7 * k, -0.4 * k, 0.1 * k] for k in range(4)])

    def frames(g, shift, sync=False):
        for k in range(4):
            g.process_pointcloud_device(dev[k], n, egos[k] + shift, None)
            if sync:
                g.sync()
            g.combine_maps_device()
            if sync:
                g.sync()

    ref, eager, over, cap = (gvom.Gvom(*args) for _ in range(4))
    over.set_overlap(True)
    for r in range(2):
        shift = np.array([0.8, 0.4, -0.2]) * r
        frames(ref, shift, sync=True)
        frames(eager, shift)
        frames(over, shift)
        if r == 0:
            frames(cap, shift)   # buffers grow before the capture
            cap.sync()
            cap.graph_begin(4)
            frames(cap, shift)
            graph = cap.graph_end()
        else:
            graph.launch(egos + shift, None)
        _same(ref, eager, f"eager {r}")
        _same(ref, over, f"overlap {r}")
        _same(ref, cap, f"captured {r}")


# words per table: below, at and above a clearing block's 16384, and not a multiple of four
@pytest.mark.parametrize("xy,z", [(8, 4), (32, 16), (37, 13), (64, 33)])
@pytest.mark.parametrize("scans", [1, 3])
def test_tables_cleared_by_the_sort(xy, z, scans):
    """A direct cast on one stream counts into tables its sort's first pass clears: after frames that
    used every buffer of every slot, the slots equal those of the tiled cast, which writes whole
    tables; an empty scan, which has no sort, leaves an empty slot."""
    import gvom
    import gvom_native as nat
    base = synth.workload(2).map_args
    direct, tiled = (gvom.Gvom(*base[:2], xy, z, 3, *base[5:]) for _ in range(2))
    direct.set_raycast_config(256, 1, False, False, False, False)
    rng = np.random.default_rng(xy)
    reach = 0.25 * xy * base[0]
    for k in range(5):
        n = 0 if k == 4 else 3000 + 100 * k
        p = np.stack([rng.normal(0, reach, n), rng.normal(0, reach, n), rng.normal(-0.5, 0.4, n)], 1)
        p = p.astype(np.float32)
        dev = nat.DeviceArray(p if n else np.zeros((1, 3), np.float32))
        off = np.linspace(0, n, scans + 1).astype(np.int64)
        egos = np.array([[0.5 * k + 0.1 * s, -0.3 * k, 0.1] for s in range(scans)])
        for g in (direct, tiled):
            g.process_batch_device(dev, off, egos, None)
            g.sync()
    for s in range(3):
        a, b = direct.slot_state(s), tiled.slot_state(s)
        assert (a is None) == (b is None)
        for key in a or ():
            assert np.array_equal(a[key], b[key]), (s, key)
