"""Which maps of a network are put in row order with its map build, and what its
layers then find."""
import copy
import gc
import pickle

import pytest
import torch

from spira_amd import nn as spnn
from spira_amd import scenes
from spira_amd.networks import kmap_schedule
from spira_amd.nn import functional as F
from spira_amd.nn.functional import _native

from helpers import np_, rel_err

pytestmark = pytest.mark.gpu


def _maps(dev, sizes, seed=0):
    g = torch.Generator().manual_seed(seed)
    maps = []
    for T in sizes:
        m = torch.randint(-1000, 1000, (T, 27), generator=g, dtype=torch.int32).clamp_(min=-1)
        maps.append(torch.nn.functional.pad(m, (0, 0, 0, -T % 128), value=-1).to(dev))
    return maps


def test_maps_of_inference_mode(dev):
    """27-offset maps below 100k rows, 150k together, made under inference
    mode: no order is kept for them, and layers read them as they are."""
    sizes = (70000, 80000, 20000)
    plain = _maps(dev, sizes)
    with torch.inference_mode():
        maps = [m.clone() for m in plain]
        F.prepare_row_orders(maps, list(sizes), [-1] * 3)
        for dtype in (torch.float16, torch.float32):
            X, W = torch.randn(1000, 32, device=dev).to(dtype), torch.randn(27, 32, 32, device=dev).to(dtype)
            if dtype == torch.float16:
                with torch.inference_mode(False):
                    X, W = X.clone(), W.clone()  # (prepared weights go by their version)
            for a, b, T in zip(maps, plain, sizes):
                y = F.sparse_convolution_forward_os(1000, T, a, X, W)
                y0 = F.sparse_convolution_forward_os(1000, T, b, X, W, tuning=(0, 0, 0, 0, 0, 0))
                assert rel_err(np_(y.float()), np_(y0.float())) <= (4e-3 if dtype == torch.float16 else 1e-5)


def test_one_map_left_over(dev):
    """17 maps, sorted as 16 and one: layers find every order, and none counts
    as free of the sort."""
    sizes = (12000,) * 17
    maps = _maps(dev, sizes, 1)
    F.prepare_row_orders(maps, list(sizes), [-1] * 17)
    for m, T in zip(maps, sizes):
        assert _native._C.finds_row_order(m, T) and not _native._C.has_free_row_order(m, T)
    other = _maps(dev, (12000,), 2)[0]
    assert not _native._C.finds_row_order(other, 12000)


def test_only_for_layers_that_read_them(dev):
    """A network's map build orders maps of a cache attached to an fp16 layer, or
    to none that it knows of; not those of a network in float32, nor its copy's."""
    coords = scenes.indoor(target=120_000, seed=3)
    keys, _ = F.flat_sort(torch.from_numpy(coords).to(dev), True)
    ts, ks, ss = kmap_schedule("UNet")

    def build(cache):
        """(27-offset maps in row order, their rows) of a build."""
        cache.reset()
        cache.add_all_kernel_maps(keys, ks, ss, ts, (1, 1, 1), [0] * len(ks))
        maps = [e for key, e in cache._kernel_maps_cache.items() if key[2] == (3, 3, 3)]
        return sum(_native._C.cached_row_order(e[3], e[2]) for e in maps)

    cache = spnn.KernelMapCache()
    orders = build(cache)
    assert orders >= 2
    a, b = spnn.SparseConv(4, 8, 3).to(dev), spnn.SparseConv(8, 8, 3).to(dev)
    a.set_kernel_map_cache(cache)
    b.set_kernel_map_cache(cache)
    assert build(cache) == 0
    a.half()
    assert build(cache) == orders
    other = spnn.KernelMapCache()
    a.set_kernel_map_cache(other)
    assert build(cache) == 0 and build(other) == orders
    twin = copy.deepcopy(b)
    assert twin._kernel_map_cache is not cache and build(twin._kernel_map_cache) == orders
    assert build(pickle.loads(pickle.dumps(spnn.KernelMapCache()))) == orders
    del b
    gc.collect()
    assert build(cache) == orders  # (attached to none again)
