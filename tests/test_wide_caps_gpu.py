"""The pair-entry gathers at caps of 17 to 64, whose entry ring is looked at
after every group of candidates: cells filled below, to and beyond the cap.
The reference order bit for bit against the oracle, FAST within its tolerances
(and its pair counts exact), compensated sums and FAST in a batch the same
bits as alone."""
import numpy as np
import pytest

import oracle
from pibiti_amd import scenes, sph
from test_fast_gpu import check_fast_step

pytestmark = pytest.mark.gpu

ARRAYS = (sph.SPH_ARRAY_POSITION, sph.SPH_ARRAY_VELOCITY, sph.SPH_ARRAY_DENSITY, sph.SPH_ARRAY_DVEL)


def scene(cap, spacing, seed=71, prec=sph.SPH_PREC_REFERENCE):
    """h = 0.02: 15 particles to a cell at spacing 0.008, 37 at 0.006, 125 at 0.004."""
    return scenes.dam_break(15, 13, 14, spacing=spacing, h=0.02, world_max=(0.3, 0.3, 0.3), dt=5e-5, viscosity=0.1,
                            vel_sigma=0.05, seed=seed, max_par_in_cell=cap, precision=prec)[:3]


def run(p, pos, vel, steps):
    with sph.SphSystem(p, keep_dvel=True) as s:
        s.reset(pos, vel)
        s.update(steps)
        return [s.get_array(w) for w in ARRAYS]


@pytest.mark.parametrize("spacing", [0.008, 0.006, 0.004])
@pytest.mark.parametrize("cap", [17, 40, 64])
def test_reference_and_fast_orders_at_wide_caps(cap, spacing):
    print("case: wide cap", cap, "spacing", spacing, flush=True)
    p, pos, vel = scene(cap, spacing)
    got = run(p, pos, vel, 2)
    o = oracle.run_f32(p, pos, vel, 2)
    for a, k in zip(got, ("pos", "vel", "dens")):
        assert np.array_equal(a, o[k]), k
    # (its check of the fluid's bulk needs particles of half the rest density,
    # which a cap far below a cell's particles leaves none)
    if np.any(oracle.step_f32(p, pos, vel)["dens"] >= 0.5 * p.rest_density):
        check_fast_step(p, pos, vel, f"cap {cap} spacing {spacing}")
    else:
        assert (cap, spacing) == (17, 0.004)


@pytest.mark.parametrize("prec", [sph.SPH_PREC_REFERENCE, sph.SPH_PREC_KAHAN, sph.SPH_PREC_FAST])
@pytest.mark.parametrize("cap", [17, 64])
def test_batch_equals_alone_at_wide_caps(cap, prec):
    print("case: wide cap", cap, "batch, precision", prec, flush=True)
    sc = [scene(cap, d, seed=72 + k, prec=prec) for k, d in enumerate((0.008, 0.004))]
    with sph.SphBatch([p for p, _, _ in sc], keep_dvel=True) as b:
        for k, (_, pos, vel) in enumerate(sc):
            b.reset(k, pos, vel)
        b.update(2)
        for k, (p, pos, vel) in enumerate(sc):
            for w, a in zip(ARRAYS, run(p, pos, vel, 2)):
                assert np.array_equal(a, b.get_array(k, w)), (k, w)
