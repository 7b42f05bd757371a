"""The radix sort behind dCOO::init at sizes where its form changes: pairs per
thread of the one-block sort, its limit per key width, the bucket path's tiles
and its buckets past LDS, uniform and skewed keys, against numpy's stable sort
(repeated pairs carry different costs, so an unstable pass shows)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [2, 1023, 1024, 1025, 3072, 3073, 4096, 4097, 5121, 7169, 8192, 8193, 12289, 65537, 262144, 300001]


@pytest.mark.parametrize("nodes", [11, 700, 70000, 9000000])
@pytest.mark.parametrize("skew", [False, True])
def test_sort_sizes(gpu, nodes, skew):
    for m in SIZES:
        rng = np.random.default_rng(m + nodes)
        u = rng.uniform(size=(2, m))
        i, j = ((u ** (6 if skew else 1)) * nodes).astype(np.int32)
        i[0], j[0] = 0, nodes - 1
        c = rng.normal(size=m).astype(np.float32)
        r, co, v, dims = gpu.dcoo_init(i, j, c)
        lo, hi = np.minimum(i, j), np.maximum(i, j)
        o = np.lexsort((np.arange(m), hi, lo))
        assert np.array_equal(r, lo[o]) and np.array_equal(co, hi[o]) and np.array_equal(v, c[o]), m
        assert dims == (int(lo.max()) + 1, int(hi.max()) + 1)
