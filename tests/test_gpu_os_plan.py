"""Column tiles and offset splits of the output-stationary kernel on both
sides of the lines where they change (256 CUs): the plan, and the layer's
output against a float64 sum over the map.

Tolerance, max |error| / RMS(reference): the fp16 store rounds to 2^-11 of a
value that may be 6 x RMS (3e-3), and the fp32 sums of the splits add far less
-> 4e-3."""
import itertools

import numpy as np
import pytest
import torch

from spira_amd.nn import functional as F
from spira_amd.nn.functional import _native

from helpers import np_, rel_err

#         T    K  cin cout  (column tile, splits)
PLANS = [(400, 8, 32, 128, 64, 8), (16300, 27, 32, 32, 32, 2), (16500, 27, 32, 32, 32, 1),
         (12900, 27, 128, 128, 64, 1), (16500, 27, 128, 128, 128, 1), (7000, 27, 128, 128, 32, 1),
         (19400, 27, 64, 96, 32, 1), (19600, 27, 64, 96, 96, 1),
         (12900, 27, 96, 96, 32, 1), (13100, 27, 96, 96, 96, 1), (20000, 27, 64, 256, 96, 1),
         (20600, 27, 64, 256, 128, 1), (700, 125, 16, 16, 32, 42), (16200, 125, 16, 16, 32, 5),
         (16300, 125, 16, 16, 32, 2),
         (22800, 125, 32, 64, 32, 1), (23100, 125, 32, 64, 64, 1), (8000, 125, 96, 128, 64, 4),
         (8300, 125, 96, 128, 64, 2), (17212, 125, 128, 128, 64, 1), (40900, 125, 96, 64, 64, 1)]


@pytest.mark.parametrize("T,K,cin,cout,tile,splits", PLANS)
def test_plan(T, K, cin, cout, tile, splits):
    if torch.cuda.is_available() and torch.cuda.get_device_properties(0).multi_processor_count != 256:
        pytest.skip("the lines are stated for 256 CUs")
    plan = _native._C.conv_os_plan(T, K, cin, 0, cout, True)
    assert (plan[0], plan[2]) == (tile, splits)


@pytest.mark.parametrize("K", [8, 27, 28, 64, 125])
def test_parts_of_grids_of_half_the_chip(K):
    """Three parts or more add in no fixed order: none where the grid, its
    tile narrowed once, holds half a block per CU or more; there a kernel of
    more than 27 offsets is split in two below one block per CU, else not."""
    for rows, cin, cout in itertools.product((1, 5, 31, 33, 42, 43, 63, 65, 127, 128, 135, 158, 255, 257, 319),
                                             (8, 16, 32, 48, 64, 96, 128, 256), (16, 32, 48, 64, 96, 128, 256, 384)):
        plan = _native._C.conv_os_plan(128 * rows, K, cin, 0, cout, True)
        wide = 32 * min(4, -(-cout // 32))
        narrow = wide if wide == 32 or rows * -(-cout // wide) >= 256 else 32 if wide == 96 else wide // 2
        if rows * -(-cout // narrow) >= 128:
            assert plan[2] <= 2, (rows, cin, cout, plan)
            if K > 27:
                assert plan[2] == (2 if rows * -(-cout // narrow) < 256 else 1), (rows, cin, cout, plan)


@pytest.mark.gpu
@pytest.mark.parametrize("T,K,cin,cout,tile,splits", PLANS)
def test_output(dev, T, K, cin, cout, tile, splits):
    g = torch.Generator().manual_seed(T)
    S = T // 2 + 1
    m = torch.randint(-2 * S, S, (T, K), generator=g, dtype=torch.int32).clamp_(min=-1)
    m[T - 130:T - 1] = -1  # an empty row group and more
    X = torch.randn(S, cin, generator=g).half().to(dev)
    W = (torch.randn(K, cin, cout, generator=g) / np.sqrt(9 * cin)).half().to(dev)
    m = torch.nn.functional.pad(m, (0, 0, 0, -T % 128), value=-1).to(dev)
    y = F.sparse_convolution_forward_os(S, T, m, X, W)
    rows = torch.cat([torch.arange(0, min(T, 400)), torch.arange(max(0, T - 400), T)]).unique().to(dev)
    Xz = torch.cat([X.double(), torch.zeros(1, cin, device=dev, dtype=torch.float64)])
    ref = torch.zeros(len(rows), cout, device=dev, dtype=torch.float64)
    for k in range(K):
        ref += Xz[m[rows, k].long()] @ W[k].double()
    assert rel_err(np_(y[rows].float()), np_(ref)) <= 4e-3
    if splits <= 2:  # one sum on every call
        for _ in range(3):
            assert torch.equal(y, F.sparse_convolution_forward_os(S, T, m, X, W))
    # a concatenated input plans by the channels of both parts
    if cin > 32 and cin % 32 == 0:
        y2 = F.sparse_convolution_forward_os(S, T, m, X[:, :32].contiguous(), W, sources2=X[:, 32:].contiguous())
        assert rel_err(np_(y2[rows].float()), np_(ref)) <= 4e-3


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(70000, 80000, 20000, 12000, 11999), (149000, 999), (12000,) * 13])
def test_orders_made_together(dev, sizes):
    """A network's 27-offset maps ordered by one batch, on both sides of its
    lines (150k rows together, 12k rows each): every layer equals the one
    that is told to take no order, in fp16 and float32, with and without a
    split of the offsets."""
    g = torch.Generator().manual_seed(len(sizes))
    maps = []
    for T in sizes:
        m = torch.randint(-1000, 1000, (T, 27), generator=g, dtype=torch.int32).clamp_(min=-1)
        maps.append(torch.nn.functional.pad(m, (0, 0, 0, -T % 128), value=-1).to(dev))
    F.prepare_row_orders(maps, list(sizes), [-1] * len(sizes))
    for m, T in zip(maps[-3:], sizes[-3:]):
        for cin, cout, dtype in ((32, 32, torch.float16), (64, 256, torch.float16), (32, 32, torch.float32)):
            X = torch.randn(1000, cin, generator=g).to(dtype).to(dev)
            W = (torch.randn(27, cin, cout, generator=g) / np.sqrt(9 * cin)).to(dtype).to(dev)
            y = F.sparse_convolution_forward_os(1000, T, m, X, W)
            y0 = F.sparse_convolution_forward_os(1000, T, m, X, W, tuning=(0, 0, 0, 0, 0, 0))
            assert rel_err(np_(y.float()), np_(y0.float())) <= (4e-3 if dtype == torch.float16 else 1e-5)


@pytest.mark.parametrize("T,cin,cout", [(1, 128, 96), (129, 96, 96), (4097, 128, 64), (70001, 112, 96)])
def test_pointwise_plan(T, cin, cout):
    assert _native._C.conv_os_plan(T, 1, cin, 0, cout, False)[1] <= 64
    assert _native._C.conv_os_plan(T, 1, cin, 0, cout, False, (0, 128, 0, 0, 0, -1))[1] == 128


@pytest.mark.gpu
@pytest.mark.parametrize("T,cin,cout", [(1, 128, 96), (129, 96, 96), (4097, 128, 64), (70001, 112, 96)])
def test_pointwise_output(dev, T, cin, cout):
    g = torch.Generator().manual_seed(T)
    X = torch.randn(T, cin, generator=g).half().to(dev)
    W = (torch.randn(1, cin, cout, generator=g) / np.sqrt(cin)).half().to(dev)
    assert rel_err(np_(F.dense_forward(X, W).float()), np_(X.double() @ W[0].double())) <= 4e-3
