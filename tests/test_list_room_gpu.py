"""The FAST walk's pair lists at their fullest: 27 cells filled to their cap
around a cell's centre, every group of four candidates with a pair, so that
the particles of the middle cell leave a group more than 27 full cells have
(their own row's run is split at the particle).  Exact: the pair counts; with
one lane per particle (a batch beyond 65,536 particles) the same bits as with
nine, and within the FAST tolerances of the oracle at the largest cap."""
import numpy as np
import pytest

from pibiti_amd import scenes, sph
from test_fast_gpu import check_fast_step

pytestmark = pytest.mark.gpu

FAST = sph.SPH_PREC_FAST


def crowd(p, pos, cap):
    """cap particles close together in each of the 27 cells around a cell's
    centre, all within h of each of the middle cell's."""
    rng = np.random.default_rng(8)
    out = pos.copy()
    lo, hi = np.array(p.world_min[:3]), np.array(p.world_max[:3])
    centre = lo + (np.floor((hi - lo) / 2 / p.h) + 0.5) * p.h
    for k, d in enumerate(np.ndindex(3, 3, 3)):
        out[k * cap:(k + 1) * cap, :3] = centre + ((np.array(d) - 1) * 0.52 + rng.uniform(-0.01, 0.01, (cap, 3))) * p.h
    assert 27 * cap == len(out)
    return out


def same_bits(a, b):
    return np.array_equal(a.view(np.uint32), b.view(np.uint32))


def test_full_lists_one_lane_equal_nine_lanes():
    p, pos, vel, _ = scenes.scaled_dam_break((12, 6, 6), seed=31, precision=FAST)
    assert p.max_par_in_cell == 16
    pos, vel = crowd(p, pos, 16), np.zeros_like(vel)
    big = scenes.scaled_dam_break((41, 41, 41), seed=3, precision=FAST)[:3]
    which = (sph.SPH_ARRAY_NEIGHBOURS, sph.SPH_ARRAY_DENSITY, sph.SPH_ARRAY_VELOCITY, sph.SPH_ARRAY_DVEL)
    print("case: full FAST lists, cap 16, one lane and nine", flush=True)
    with sph.SphBatch([big[0], p], keep_dvel=True) as b:
        assert b.info()["particles"] > 65536
        b.reset(0, *big[1:])
        b.reset(1, pos, vel)
        b.update(1)
        with sph.SphSystem(p, keep_dvel=True) as s:
            s.reset(pos, vel)
            s.update(1)
            assert s.get_array(sph.SPH_ARRAY_NEIGHBOURS).max() == 431
            for w in which:
                assert same_bits(s.get_array(w), b.get_array(1, w)), w
        with sph.SphSystem(big[0], keep_dvel=True) as s:
            s.reset(*big[1:])
            s.update(1)
            for w in which:
                assert same_bits(s.get_array(w), b.get_array(0, w)), w


def test_full_lists_at_the_largest_cap():
    p, pos, vel, _ = scenes.scaled_dam_break((12, 12, 12), seed=32, max_par_in_cell=64)
    print("case: full FAST lists, cap 64", flush=True)
    g = check_fast_step(p, crowd(p, pos, 64), np.zeros_like(vel), "cap 64")
    assert g["nnb"].max() == 1727
