"""The full sort inside the place kernel over many tiles (4,096 pairs each),
on consecutive steps: its blocks hand their tiles to each other within one
launch, through the input, the digit counts and two or three passes, and the
look-back crosses spans of 16 tiles.  Exact: the sorted keys, the permutation
and the cell ranges against a host sort of the positions after each step, and
the positions against the oracle's integration."""
import numpy as np
import pytest

import oracle
from pibiti_amd import scenes, sph
from test_resort_gpu import assert_sorted_like_oracle

pytestmark = pytest.mark.gpu


def many_cells():  # 320,000 particles: 79 tiles; 19 key bits, three passes
    return scenes.scaled_dam_break((80, 50, 80), seed=51, vel_sigma=2.0)[:3]


def few_cells():  # 216,000 particles: 53 tiles; 14 key bits, two passes
    return scenes.dam_break(60, 60, 60, spacing=0.004, h=0.02, world_max=(0.5, 0.5, 0.5), dt=5e-5, viscosity=0.1,
                            vel_sigma=2.0, seed=52)[:3]


@pytest.mark.parametrize("make, passes", [(many_cells, 3), (few_cells, 2)])
def test_full_sorts_over_many_tiles(make, passes):
    p, pos, vel = make()
    assert (p.key_bits + 7) // 8 == passes and p.num_particles > 33 * 4096
    # 5,000 particles in one cell: the full sort on every step
    wmin, cs = np.array(p.world_min, np.float64), np.array(p.cell_size, np.float64)
    centre = wmin + (np.floor((pos[0, :3] - wmin) / cs) + 0.5) * cs
    rng = np.random.default_rng(6)
    crowd = rng.permutation(p.num_particles)[:5000]
    pos[crowd, :3] = (centre + rng.uniform(-0.002, 0.002, (5000, 3))).astype(np.float32)
    vel[crowd] = 0
    print("case: full sorts over many tiles,", p.num_particles, "particles,", passes, "passes", flush=True)
    with sph.SphSystem(p) as s:
        s.reset(pos, vel)
        for step in range(5):
            s.update(1)
            st = s.stats()
            assert st["full_sort"] == 1 and st["sort_errors"] == 0, step
            assert_sorted_like_oracle(s, p)
            if step == 0:
                o = oracle.step_f32(p, pos, vel)
                assert np.array_equal(s.get_array(sph.SPH_ARRAY_POSITION), o["pos"])


def test_more_tiles_than_blocks_at_once():
    """2,195,200 particles: 536 tiles a stage, more than the 512 blocks that
    run at a time, on two consecutive steps."""
    p, pos, vel = scenes.scaled_dam_break((140, 112, 140), seed=53, vel_sigma=2.0)[:3]
    wmin, cs = np.array(p.world_min, np.float64), np.array(p.cell_size, np.float64)
    centre = wmin + (np.floor((pos[0, :3] - wmin) / cs) + 0.5) * cs
    rng = np.random.default_rng(7)
    pos[:5000, :3] = (centre + rng.uniform(-0.002, 0.002, (5000, 3))).astype(np.float32)
    vel[:5000] = 0
    print("case: full sort, 536 tiles", flush=True)
    with sph.SphSystem(p) as s:
        s.reset(pos, vel)
        for step in range(2):
            s.update(1)
            st = s.stats()
            assert st["full_sort"] == 1 and st["sort_errors"] == 0, step
            assert_sorted_like_oracle(s, p)
