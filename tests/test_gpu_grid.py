"""The downsample by occupancy grids against the oracle: single keys, columns
around a 32-cell word, levels whose words end inside a block's share, both key
widths, uneven strides, the fields' ends, and boxes too wide for the grids
(then by merging) or unsorted keys (then by sorting)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from spira_amd.nn import KernelMapCache
from spira_amd.nn import functional as F

from helpers import np_

pytestmark = pytest.mark.gpu

S4 = [(2, 2, 2), (4, 4, 4), (8, 8, 8), (16, 16, 16)]


def _box(n, ext, seed, origin=(0, 0, 0)):
    rng = np.random.default_rng(seed)
    c = np.stack([rng.integers(0, e, n) for e in ext], 1) + np.array(origin)
    return np.unique(c, axis=0).astype(np.int32)


SCENES = {
    "one": (np.array([[5, 6, 7]], np.int32), True, S4),
    "words": (_box(3000, (9, 9, 65), 1), True, S4),
    "full": (_box(200000, (33, 31, 64), 2), True, S4),
    "ragged": (_box(20001, (301, 77, 31), 3, (1, 3, 5)), True, [(1, 1, 2), (2, 1, 2), (4, 4, 16)]),
    "wide_z": (_box(5000, (40, 40, 60000), 4), True, [(2, 2, 2), (8, 8, 2)]),
    "narrow_keys": (_box(9000, (200, 300, 250), 5), False, S4),
    "ends32": (np.array([[0, 4000, 200], [4095, 4095, 255], [4095, 4094, 255]], np.int32), False, S4[:1]),
    "eight": (_box(4000, (500, 500, 300), 6), True, [(2 ** l,) * 3 for l in range(1, 9)]),
    "nine": (_box(4000, (500, 500, 300), 6), True, [(2 ** l,) * 3 for l in range(1, 10)]),
    "sweep": (_box(5000, (3200, 3200, 90), 9), True, S4),
    "too_wide": (_box(700, (60000, 60000, 4000), 7), True, S4),
}


@pytest.mark.parametrize("name", sorted(SCENES))
def test_levels(dev, name):
    c, double, strides = SCENES[name]
    keys, _ = orc.flatten_sort(c, double)
    k = torch.from_numpy(keys).to(dev)
    levels, counts = F.downsample_chain_launch(k, strides, grid=True)
    n = counts.tolist()
    assert n[-1] == (2 if name == "too_wide" else 0)
    outs = F.streamed_output_generate(k, strides)
    for i, s in enumerate(strides):
        ref = orc.downsample(keys, s)
        assert np.array_equal(np_(outs[i]), ref), s
        if n[-1] == 0:
            assert np.array_equal(np_(levels[i][:n[i]]), ref), s


def test_unsorted_is_flagged(dev):
    keys, _ = orc.flatten_sort(_box(5000, (60, 60, 60), 8), True)
    k = torch.from_numpy(keys[::-1].copy()).to(dev)
    assert F.downsample_chain_launch(k, S4, grid=True)[1].tolist()[-1] == 1
    for o, s in zip(F.streamed_output_generate(k, S4), S4):
        assert np.array_equal(np_(o), orc.downsample(keys, s)), s


@pytest.mark.parametrize("name", ["words", "sweep", "too_wide"])
def test_network_levels(dev, name):
    """The levels that a network's map build takes, by grids or by merging; a
    build after one that was too wide merges straight away, for a while."""
    c, double, strides = SCENES[name]
    keys, _ = orc.flatten_sort(c, double)
    k = torch.from_numpy(keys).to(dev)
    cache = KernelMapCache()
    n = len(strides)
    for i in range(3):
        cache.reset()
        cache.add_all_kernel_maps(k, [3] * (2 * n + 1), [(1, 1, 1)] * 2 + [s for s in strides for _ in range(2)],
                                  strides, (1, 1, 1), [0] * (2 * n + 1))
        for s in strides:
            assert np.array_equal(np_(cache.get_target_coordinates(k, (1, 1, 1), s)), orc.downsample(keys, s)), s
        assert cache._merge_builds == (max(0, cache.MERGE_BUILDS - i) if name == "too_wide" else 0)
