"""Reads and synchronising calls when the pinned transfer buffer cannot be had
(forced from the host): the runtime's own copies give the same arrays, the
order's error is still reported, and the next read is back on the buffer."""
import numpy as np
import pytest

from pibiti_amd import scenes, sph

pytestmark = pytest.mark.gpu

ARRAYS = (sph.SPH_ARRAY_POSITION, sph.SPH_ARRAY_VELOCITY, sph.SPH_ARRAY_DENSITY, sph.SPH_ARRAY_PRESSURE,
          sph.SPH_ARRAY_DVEL, sph.SPH_ARRAY_NEIGHBOURS)


def without_buffer(call):
    sph.debug_fail_alloc(1)
    try:
        return call()
    finally:
        sph.debug_fail_alloc(0)


def test_reads_without_the_pinned_buffer():
    p, pos, vel, _ = scenes.scaled_dam_break((9, 7, 11), seed=61)
    print("case: reads without the pinned buffer", flush=True)
    with sph.SphSystem(p, keep_dvel=True) as s:
        s.reset(pos, vel)
        s.update(3)
        for which in ARRAYS:
            plain = without_buffer(lambda: s.get_array(which))
            assert np.array_equal(plain.view(np.uint32), s.get_array(which).view(np.uint32)), which
        without_buffer(s.synchronize)
        s.debug_poke(sph.SPH_DEBUG_ORDER_ERROR)
        with pytest.raises(sph.SphError) as e:
            without_buffer(s.synchronize)
        assert e.value.status == sph.SPH_ERR_ORDER
        s.reset(pos, vel)
        assert np.array_equal(without_buffer(lambda: s.get_array(sph.SPH_ARRAY_POSITION)), pos)
