"""Which maps of a network are put in row order with its map build, and what its
layers then find."""
import pytest
import torch

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
