"""What the Python mapper makes of the library's answers, on the CPU: a recording stand-in for the
loaded library takes the place of the native one."""
import ctypes

import numpy as np
import pytest

import gvom
import gvom_native as nat


class _Library:
    """Answers the calls a test names; every call is kept."""

    def __init__(self, **answers):
        self.answers, self.calls = answers, []

    def __getattr__(self, name):
        def call(*args):
            self.calls.append((name, args))
            return self.answers[name](*args)
        return call


def _mapper(**answers):
    g = gvom.Gvom.__new__(gvom.Gvom)
    g._lib, g._h, g.xy_size = _Library(**answers), None, 4
    return g


def test_voxel_cloud_of_a_map_that_shrinks_between_the_two_calls():
    """The row count is asked for first and the rows are fetched by a second call; another thread's
    combine in between can leave fewer cells.  Only the rows the second call wrote are returned."""
    counts = [5, 3]

    def debug_voxel_map(h, out, cap, rows):
        n = counts.pop(0)
        rows._obj.value = n
        if out is not None:
            assert cap >= n
            buf = (ctypes.c_float * (8 * n)).from_address(ctypes.cast(out, ctypes.c_void_p).value)
            buf[:] = [float(i) for i in range(8 * n)]
        return nat.GVOM_OK

    cloud = _mapper(gvom_debug_voxel_map=debug_voxel_map).make_debug_voxel_map()
    assert cloud.shape == (3, 8)
    assert np.array_equal(cloud.ravel(), np.arange(24, dtype=np.float32))


@pytest.mark.parametrize("name,rows", [("slot_state", ("hit", "total", "min_h", "metrics")),
                                       ("combined_state", ("hit", "total", "min_h", "metrics", "eigen"))])
def test_state_of_a_map_that_shrinks_between_the_two_calls(name, rows):
    counts = [5, 3]

    def get(h, *args):
        args[-1]._obj.value = counts.pop(0)
        return nat.GVOM_OK

    g = _mapper(gvom_get_slot=get, gvom_get_combined=get)
    g.voxel_count = 64
    state = g.slot_state(0) if name == "slot_state" else g.combined_state()
    for k in rows:
        assert len(state[k]) == 3, k


# flag bits: 1 LDS box, 2 sector order, 4 tiled scratch, 8 spread, 16 azimuth order
@pytest.mark.parametrize("args,kw,expect", [
    ((), {}, (128, 1, 4 + 8 + 16)),                                            # as a new handle starts
    ((64,), {}, (64, 1, 4 + 8 + 16)),                                          # only the launch shape changes
    ((), dict(rays_per_thread=2, spread=False), (128, 2, 4 + 16)),
    ((256, 1, False, False, False, False), {}, (256, 1, 0)),                   # a variant for every scan
    ((128, 1, False, False, True), {}, (128, 1, 4 + 8)),
    ((256, 1), dict(use_box=True, tiled=False), (256, 1, 1 + 8)),
    ((), dict(sector_order=True), (128, 1, 2 + 4 + 8)),
    ((256, 1, False, False, False, False, True), {}, (256, 1, 16)),            # ... for the small ones
    ((), dict(azimuth=False), (128, 1, 4 + 8)),
])
def test_raycast_config_flags(args, kw, expect):
    g = _mapper(gvom_set_raycast_config=lambda h, *a: nat.GVOM_OK)
    g.set_raycast_config(*args, **kw)
    assert g._lib.calls == [("gvom_set_raycast_config", (None,) + expect)]
