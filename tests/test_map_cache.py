"""Map caches as programs keep them: classes of their own, copies and pickles
(host only)."""
import copy
import pickle

from spira_amd import nn as spnn


class NamedCache(spnn.KernelMapCache):
    def __init__(self, name):
        super().__init__()
        self.name = name


class OwnCache:
    """Any class with the methods that layers call."""


def test_copies_of_a_subclass():
    cache, conv = NamedCache("a"), spnn.SparseConv(4, 8, 3)
    conv.set_kernel_map_cache(cache)
    cache.row_order_requests[1] = 1
    for c in (copy.copy(cache), copy.deepcopy(cache), pickle.loads(pickle.dumps(cache))):
        assert c.name == "a" and c.row_order_requests == {1: 1} and c._orders_read()
        conv.set_kernel_map_cache(c)
        assert not c._orders_read()  # (a float32 layer alone)
    assert copy.deepcopy(conv)._kernel_map_cache.name == "a"


def test_cache_of_another_class():
    own, conv = OwnCache(), spnn.SparseConv(4, 8, 3)
    conv.set_kernel_map_cache(own)
    assert conv._kernel_map_cache is own
    conv.set_kernel_map_cache(spnn.KernelMapCache())
    conv.set_kernel_map_cache(own)
    conv.set_kernel_map_cache(None)
    assert conv._kernel_map_cache is None
