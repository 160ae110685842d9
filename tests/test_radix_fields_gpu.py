"""The radix sort where a tile's count and a span's sum are at their largest
(4,096 and 65,536, every key of 16 tiles in one digit) and at their smallest,
beside each other, against numpy's stable sort; the call that allocates its
scratch and the one that does not."""
import numpy as np
import pytest

from pibiti_amd import sph
from test_radix_sort_gpu import expected, run

pytestmark = pytest.mark.gpu


def keys_of(kind, n):
    k = np.arange(n, dtype=np.uint32)
    if kind == "one key":
        return np.full(n, 0x2FF01, np.uint32)
    if kind == "a digit per span":  # 16 tiles of one key each
        return (k // 65536 * 0x1357) & np.uint32(0x3FFFF)
    return np.where(k % 4096 == 4095, 0x30000, 0x2FFFF).astype(np.uint32)  # all but one of a tile


@pytest.mark.parametrize("kind", ["one key", "a digit per span", "one of a tile apart"])
@pytest.mark.parametrize("n", [16 * 4096, 49 * 4096 + 3, 1_100_000])
def test_sort_at_the_largest_counts(kind, n):
    print("case: radix sort,", kind, n, flush=True)
    keys, vals = keys_of(kind, n), np.arange(n, dtype=np.uint32)[::-1].copy()
    ek, ev = expected(keys, vals, 18)
    for fn in (sph.lib().sph_radix_sort, sph.lib().sph_radix_sort_noalloc):
        if fn is sph.lib().sph_radix_sort_noalloc and n > 1 << 20:
            continue
        st, k, v = run(fn, keys, vals, 18)
        assert st == sph.SPH_OK and np.array_equal(k, ek) and np.array_equal(v, ev)
