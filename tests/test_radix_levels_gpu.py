"""The radix sort where its look-back gets a further level of sums: 16, 256
and 4,096 tiles of 4,096 pairs and one tile more, against numpy's stable
sort; random keys, and all of a tile in one digit."""
import numpy as np
import pytest

from pibiti_amd import sph
from test_radix_sort_gpu import run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "nearly one key"])
@pytest.mark.parametrize("tiles, extra", [(16, 0), (16, 1), (256, 0), (256, 1), (4096, 0), (4096, 1), (4353, 77)])
def test_sort_at_the_levels_of_the_look_back(tiles, extra, kind):
    n = 4096 * tiles + extra
    print("case: radix sort,", tiles, "tiles and", extra, kind, flush=True)
    rng = np.random.default_rng(n)
    keys = rng.integers(0, 2 ** 16, n, dtype=np.uint16)
    if kind != "random":
        keys[rng.random(n) < 0.999] = 0x80FF
    vals = np.arange(n, dtype=np.uint32)
    st, k, v = run(sph.lib().sph_radix_sort, keys.astype(np.uint32), vals, 16)
    order = np.argsort(keys, kind="stable")
    assert st == sph.SPH_OK and np.array_equal(k, keys[order]) and np.array_equal(v, vals[order])
