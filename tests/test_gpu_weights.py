"""Weights that change between two calls of a layer: every dataflow computes
with the values the weights hold when it is called, float32 also where nothing
tells of the change (writes through ``.data``, inference tensors, a captured
graph's replays, another stream).  float32 outputs are compared with the same
layer on a fresh copy of the weights: one kernel, one order of sums, equal bits
(dataflows 1 and 3, whose small lists take the pass with atomics, to 1e-5 of
the RMS)."""
import numpy as np
import pytest
import torch

from oracle import oracle as orc
from spira_amd import nn as spnn
from spira_amd import scenes
from spira_amd.nn import functional as F

from helpers import np_, rel_err

DATAFLOWS = [0, 1, 2, 3, 5, 6]


def test_reset_parameters_is_seen():
    """A reset counts as a change of the parameters (their version)."""
    m = spnn.SparseConv(4, 8, 3, bias=True)
    before = m.kernel._version, m.bias._version
    m.reset_parameters()
    assert m.kernel._version > before[0] and m.bias._version > before[1]
    assert m.kernel.requires_grad


@pytest.fixture(scope="module")
def keys(dev):
    k, _ = orc.flatten_sort(1 + scenes.spheres_planes(n=6000, grid=64, seed=3), True)
    return torch.from_numpy(k).to(dev)


def _layer(keys, d, cin=32, cout=48, dtype=torch.float32):
    g = torch.Generator().manual_seed(d)
    conv = spnn.SparseConv(cin, cout, 3).to(device=keys.device, dtype=dtype)
    conv.tunable_config["map_dataflow"] = d
    cache = spnn.KernelMapCache()
    conv.set_kernel_map_cache(cache)
    x = torch.randn(len(keys), cin, generator=g).to(dtype).to(keys.device)
    import spira_amd
    return conv, spira_amd.SparseTensor(keys, x, stride=1)


def _same(d, y, ref):
    if d % 2:
        return rel_err(np_(y.float()), np_(ref.float())) <= 1e-5
    return torch.equal(y, ref)


@pytest.mark.gpu
@pytest.mark.parametrize("d", DATAFLOWS)
def test_float32_weights_changed_in_place(dev, keys, d):
    conv, x = _layer(keys, d)
    fresh, _ = _layer(keys, d)

    def check():
        y = conv(x).features
        fresh.kernel = torch.nn.Parameter(conv.kernel.detach().clone())
        assert _same(d, y, fresh(x).features)
        return y

    with torch.no_grad():
        seen = [check()]
        conv.kernel.data.mul_(-0.5)  # (no version, no pointer changes)
        seen.append(check())
        conv.kernel.data.copy_(torch.randn_like(conv.kernel))
        seen.append(check())
        conv.reset_parameters()
        seen.append(check())
        conv.kernel.add_(1.0)
        seen.append(check())
    assert all(not torch.equal(a, b) for a, b in zip(seen, seen[1:]))


@pytest.mark.gpu
@pytest.mark.parametrize("d", [0, 1, 2])
def test_float16_reset_parameters(dev, keys, d):
    conv, x = _layer(keys, d, dtype=torch.float16)
    fresh, _ = _layer(keys, d, dtype=torch.float16)
    with torch.no_grad():
        for _ in range(2):
            y = conv(x).features
            fresh.kernel = torch.nn.Parameter(conv.kernel.detach().clone())
            assert rel_err(np_(y.float()), np_(fresh(x).features.float())) <= 4e-3
            conv.reset_parameters()


@pytest.mark.gpu
@pytest.mark.parametrize("d", DATAFLOWS)
def test_float32_inference_tensors(dev, keys, d):
    """A float32 layer built under inference mode, whose tensors have no
    version, computes what the same layer does outside it."""
    ref, x = _layer(keys, d)
    with torch.inference_mode():
        conv, xi = _layer(keys, d)
        conv.kernel.copy_(ref.kernel)
        y = conv(xi).features
    with torch.no_grad():
        assert _same(d, y, ref(x).features)


@pytest.mark.gpu
@pytest.mark.parametrize("d", DATAFLOWS)
def test_float32_on_two_streams(dev, keys, d):
    conv, x = _layer(keys, d)
    with torch.no_grad():
        want = conv(x).features  # (the map is made here)
        for _ in range(3):
            conv.kernel.data.copy_(conv.kernel.data.clone())
            torch.cuda.synchronize()
            streams = [torch.cuda.Stream(), torch.cuda.Stream()]
            ys = []
            for s in streams:
                with torch.cuda.stream(s):
                    ys.append(conv(x).features)
            torch.cuda.synchronize()
            assert all(_same(d, y, want) for y in ys)


@pytest.mark.gpu
@pytest.mark.parametrize("d", [0, 2, 6])
def test_float32_captured(dev, keys, d):
    """Captured on its first call, replayed after eager work and after its
    weights changed in place: each replay equals the eager result."""
    conv, x = _layer(keys, d)
    twin, _ = _layer(keys, d)
    twin.set_kernel_map_cache(conv._kernel_map_cache)
    with torch.no_grad():
        twin(x)  # makes the map
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = conv(x).features
        for i in range(4):
            graph.replay()
            torch.cuda.synchronize()
            got = y.clone()
            assert torch.equal(got, conv(x).features)
            conv.kernel.data.mul_(1.0 + i)
            torch.cuda.synchronize()


@pytest.mark.gpu
@pytest.mark.parametrize("d", DATAFLOWS)
def test_float16_prepared_for_another_stream(dev, keys, d):
    """Weights prepared on a busy stream are waited for by the stream that
    reads them next."""
    conv, x = _layer(keys, d, dtype=torch.float16)
    twin, _ = _layer(keys, d, dtype=torch.float16)
    twin.set_kernel_map_cache(conv._kernel_map_cache)
    twin.kernel = torch.nn.Parameter(conv.kernel.detach().clone())
    with torch.no_grad():
        want = twin(x).features  # (the map is made here)
        torch.cuda.synchronize()
        a, b = torch.cuda.Stream(), torch.cuda.Stream()
        with torch.cuda.stream(a):
            torch.cuda._sleep(20_000_000)  # ~10 ms
            ya = conv(x).features
        with torch.cuda.stream(b):
            yb = conv(x).features
        torch.cuda.synchronize()
    for y in (ya, yb):
        assert rel_err(np_(y.float()), np_(want.float())) <= 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("d", [0, 1, 2, 6])
def test_float16_captured_first(dev, keys, d):
    """A layer whose first call is captured: eager calls before a replay and
    after it, and every replay, compute the same."""
    conv, x = _layer(keys, d, dtype=torch.float16)
    twin, _ = _layer(keys, d, dtype=torch.float16)
    for m in (conv, twin):  # (one part: no workspace shared by the stream's calls)
        m.tunable_config["os_tuning"] = (0, 0, 1, 0, 0, 0)
    twin.set_kernel_map_cache(conv._kernel_map_cache)
    twin.kernel = torch.nn.Parameter(conv.kernel.detach().clone())
    with torch.no_grad():
        want = np_(twin(x).features.float())
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            y = conv(x).features
        for _ in range(3):
            assert rel_err(np_(conv(x).features.float()), want) <= 4e-3
            y.zero_()
            graph.replay()
            torch.cuda.synchronize()
            assert rel_err(np_(y.float()), want) <= 4e-3
