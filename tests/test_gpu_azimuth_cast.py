"""The azimuth-ordered ray cast (the default for large scans) against the linear direct cast.

Pass counts are whole numbers that do not depend on the order or on where a step is counted, so
the slots must be equal bit for bit.  The shapes sit where the wedge layout has its edges: the
smallest scan the rule sends there, a side above twice the layout's rows, rays longer than one
segment count holds, heights and wedges past the LDS counters' room, rays that lead along z,
positions so far from the world's origin that the f32 steps round visibly, several scans sharing a tile, empty scans and scans whose points are all dropped.
"""
import numpy as np
import pytest

import gvom_synth as synth

pytestmark = pytest.mark.gpu

MIN_WORK = 12_000_000   # points x xy_size from which the azimuth order is used


def _points(rng, n, ego, kind, dtype):
    az = rng.uniform(0, 2 * np.pi, n)
    if kind == "sphere":       # every direction, straight up and down among them
        el = np.arcsin(rng.uniform(-1, 1, n))
    elif kind == "narrow":     # all rays in a few wedges around the diagonals and the axes
        el = rng.uniform(-0.2, 0.2, n)
        az = (np.floor(az / (np.pi / 4)) * (np.pi / 4)) + rng.normal(0, 0.01, n)
    else:
        el = rng.uniform(-0.4, 0.4, n)
    r = rng.uniform(0.5, 400.0, n) if kind != "near" else rng.uniform(0.0, 6.0, n)
    p = np.stack([r * np.cos(el) * np.cos(az), r * np.cos(el) * np.sin(az), r * np.sin(el)], 1) + ego
    k = n // 50
    p[:k] = np.round(p[:k] / 0.4) * 0.4                  # on voxel corners
    p[k:k + 20] = ego                                    # no direction at all
    p[k + 20:k + 40, :2] = ego[:2]                       # straight up or down
    p[k + 40:k + 60, 1] = ego[1]                         # along an axis
    p[k + 60:k + 80, 1] = ego[1] + (p[k + 60:k + 80, 0] - ego[0])   # along a diagonal
    p[k + 80:k + 100] = np.nan
    return p.astype(dtype)


def _compare(args, scans, dtype, label, shift=0.0):
    """scans: list of batches (lists of point arrays)."""
    import gvom
    az, lin = gvom.Gvom(*args), gvom.Gvom(*args)
    lin.set_raycast_config(256, 1, False, False, False, False)
    for b, batch in enumerate(scans):
        egos = np.array([[0.13 + 0.9 * b, -0.41 * b, 0.77 + 0.1 * b]] * len(batch))
        egos[:, 0] += 0.3 * np.arange(len(batch))
        egos += shift
        flat = np.concatenate(batch).astype(dtype)
        off = np.cumsum([0] + [len(p) for p in batch])
        for g in (az, lin):
            if len(batch) == 1:
                g.Process_pointcloud(flat, egos[0], None)
            else:
                g.process_batch(flat, off, egos, None)
    for s in range(args[4]):
        a, b = az.slot_state(s), lin.slot_state(s)
        assert (a is None) == (b is None), f"{label}: slot {s}"
        if a is None:
            continue
        for k in a:
            assert np.array_equal(a[k], b[k], equal_nan=True), f"{label}: slot {s} {k}"


@pytest.mark.parametrize("xy,z,n,kind,dtype,shift", [
    (64, 32, MIN_WORK // 64, "sphere", np.float32, 0.0),      # the smallest work the rule takes
    (37, 13, MIN_WORK // 37 + 1, "near", np.float32, 0.0),    # odd sizes, words not a multiple of four
    (1100, 8, 20011, "flat", np.float32, 0.0),                # sides above twice the layout's rows
    (1100, 8, 20011, "narrow", np.float64, 0.0),
    (160, 256, 80001, "sphere", np.float32, 0.0),             # heights past the counters' room
    (250, 60, 49152, "flat", np.float64, 0.0),
    (96, 40, 130000, "narrow", np.float32, 0.0),              # few, dense wedges
    (250, 60, 49152, "sphere", np.float64, 480000.0),         # 1.2e6 and 2.4e6 voxels away: steps of
    (120, 100, 100001, "flat", np.float64, -8.0e5),           # 1/8 and 1/4 voxel are representable
])
def test_azimuth_cast_equals_linear(xy, z, n, kind, dtype, shift):
    assert n * xy >= MIN_WORK
    rng = np.random.default_rng(xy * 1000 + z)
    args = synth.gvom_args(0.4, 0.2, xy, z, 2)
    scans = [[_points(rng, n, np.array([0.13 + 0.9 * b, -0.41 * b, 0.77]) + shift, kind, dtype)]
             for b in range(2)]
    _compare(args, scans, dtype, f"{xy}x{xy}x{z} {kind}", shift)


def test_azimuth_cast_batches():
    """Scans that share tiles and blocks, empty ones between them, one whose points all drop."""
    rng = np.random.default_rng(7)
    ego = np.array([0.13, 0.0, 0.77])
    sizes = [3, 0, 2045, 0, 40000, 1, 2049, 5000]
    batch = [_points(rng, max(n, 8200), ego, "flat", np.float32)[164:164 + n] for n in sizes]
    batch[-1][:] = np.nan
    args = synth.gvom_args(0.4, 0.2, 256, 64, 8)
    assert sum(sizes) * 256 >= MIN_WORK
    _compare(args, [batch], np.float32, "batch")
