"""Row scans, pair lists and masks of the maps against the oracle at the sizes
where their kernels change: rows of 1, 16 and 17 waves' tiles, counts on both
sides of 65536, half maps with and without a centre row, strided maps (whose
masks have no mirrored rows) and targets that end inside a tile."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from spira_amd.nn import functional as F

from helpers import assert_tuple_equal

pytestmark = pytest.mark.gpu


def _keys(n, ext, seed):
    rng = np.random.default_rng(seed)
    c = np.unique(np.stack([rng.integers(1, e, 2 * n) for e in ext], 1), axis=0)
    c = c[np.sort(rng.permutation(len(c))[:n])].astype(np.int32)
    return orc.flatten_sort(c, True)[0]


@pytest.mark.parametrize("df", range(1, 9))
@pytest.mark.parametrize("n,k", [(1, 3), (64, 3), (65, 5), (1023, (3, 1, 3)), (65473, (1, 1, 3)), (65600, 3),
                                 (66500, 5), (66700, 5)])
def test_submanifold(dev, n, k, df):
    if n > 60000 and df not in (1, 2, 5, 6):
        pytest.skip("the same kernels at the larger sizes")
    k = (k,) * 3 if isinstance(k, int) else k
    if df > 4 and np.prod(k) < 9:
        pytest.skip("hybrid maps of 9 offsets and more")
    keys = _keys(n, (120, 90, 60), n)
    t = torch.from_numpy(keys).to(dev)
    got = F.build_kmap(t, t, k, (1, 1, 1), df)
    assert_tuple_equal(got, orc.build_kmap(keys, keys, k, (1, 1, 1), df), f"n={n} k={k} df={df}")


@pytest.mark.parametrize("df", [1, 2])
@pytest.mark.parametrize("n", [1, 100, 5000, 150000])
def test_strided(dev, n, df):
    keys = _keys(n, (150, 120, 90), n + 1)
    down = orc.downsample(keys, (2, 2, 2))
    got = F.build_kmap(torch.from_numpy(keys).to(dev), torch.from_numpy(down).to(dev), (2, 2, 2), (1, 1, 1), df)
    assert_tuple_equal(got, orc.build_kmap(keys, down, (2, 2, 2), (1, 1, 1), df), f"n={n} df={df}")
