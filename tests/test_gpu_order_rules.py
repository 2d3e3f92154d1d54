"""Which maps of a network are put in row order with its map build: what the
layers then find, for maps without a version (inference tensors)."""
import pytest
import torch

from spira_amd.nn import functional as F

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
