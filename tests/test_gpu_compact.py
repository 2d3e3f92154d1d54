"""The compacted convolution kernels (masks, pair lists, fp32 maps) at the
edges of their tiles: targets around a block of 64, offsets around a chunk of
32, channels around the 16-byte row and the column tiles, empty and full maps,
pairs in any order and repeated pairs.  Against a float64 sum over the pairs.

Tolerance, max |error| / RMS(reference): fp16 stores round to 2^-11 of a value
that may be 6 x RMS (3e-3) -> 4e-3; fp32 sums of up to 8000 products, error
growth ~ sqrt(n) 2^-24 of the terms' norm -> 1e-5 (the fp32 bar)."""
import ctypes
import os

import numpy as np
import pytest
import torch

from spira_amd.nn import functional as F
from spira_amd.nn.functional import _native

from helpers import np_, rel_err

pytestmark = pytest.mark.gpu

TOL = {torch.float16: 4e-3, torch.float32: 1e-5}
#        S    T    K  cin cout  density
SHAPES = [(1, 1, 1, 3, 1, 1.0), (70, 63, 8, 4, 16, 0.5), (70, 64, 27, 16, 17, 0.3), (90, 65, 33, 20, 48, 0.4),
          (130, 129, 31, 33, 64, 0.0), (200, 128, 32, 64, 65, 1.0), (300, 200, 65, 96, 97, 0.2),
          (64, 190, 125, 24, 40, 0.3), (150, 100, 27, 160, 130, 0.5), (150, 100, 27, 256, 48, 0.6)]


def _lists(S, T, K, density, seed):
    """Per offset: distinct sources and distinct targets, paired at random."""
    rng = np.random.default_rng(seed)
    out = []
    for _ in range(K):
        n = int(round(density * min(S, T)))
        out.append((rng.permutation(S)[:n].astype(np.int32), rng.permutation(T)[:n].astype(np.int32)))
    return out


def _data(S, T, K, cin, cout, dtype, seed):
    g = torch.Generator().manual_seed(seed)
    X = torch.randn(S, cin, generator=g).to(dtype)
    W = (torch.randn(K, cin, cout, generator=g) / np.sqrt(cin)).to(dtype)
    epi = (torch.rand(cout, generator=g) + 0.5, torch.randn(cout, generator=g),
           torch.randn(T, cout, generator=g).to(dtype), True)
    return X, W, epi


def _ref(lists, T, X, W, epi=None):
    X, W = X.double().numpy(), W.double().numpy()
    y = np.zeros((T, W.shape[2]))
    for k, (s, t) in enumerate(lists):
        np.add.at(y, t, X[s] @ W[k])
    if epi is not None:
        scale, shift, res, _ = epi
        y = np.maximum(y * scale.double().numpy() + shift.double().numpy() + res.double().numpy(), 0)
    return y


def _dev(epi, dev):
    return tuple(v.to(dev) if isinstance(v, torch.Tensor) else v for v in epi)


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("S,T,K,cin,cout,density", SHAPES)
def test_masks(dev, dtype, S, T, K, cin, cout, density):
    lists = _lists(S, T, K, density, S + K)
    X, W, epi = _data(S, T, K, cin, cout, dtype, K)
    sm, tm = np.full((K, S), -1, np.int32), np.full((K, T), -1, np.int32)
    for k, (s, t) in enumerate(lists):
        sm[k, s] = tm[k, t] = np.arange(len(s))
    sizes = torch.tensor([len(s) for s, _ in lists], dtype=torch.int32, device=dev)
    args = (S, T, X.to(dev), W.to(dev), torch.from_numpy(sm).to(dev), torch.from_numpy(tm).to(dev), sizes, 16, 16)
    y = F.sparse_convolution_forward_ws(*args)
    assert rel_err(np_(y.float()), _ref(lists, T, X, W)) <= TOL[dtype]
    y2 = F.sparse_convolution_forward_ws(*args, epilogue=_dev(epi, dev))
    assert rel_err(np_(y2.float()), _ref(lists, T, X, W, epi)) <= TOL[dtype]
    assert torch.equal(y, F.sparse_convolution_forward_ws(*args))  # (sums in a fixed order)


@pytest.mark.parametrize("S,T,K,cin,cout,density", SHAPES)
def test_fp32_map(dev, S, T, K, cin, cout, density):
    lists = _lists(S, T, K, density, S + K)
    X, W, epi = _data(S, T, K, cin, cout, torch.float32, K)
    m = np.full(((T + 127) // 128 * 128, K), -1, np.int32)
    for k, (s, t) in enumerate(lists):
        m[t, k] = s
    y = F.sparse_convolution_forward_os(S, T, torch.from_numpy(m).to(dev), X.to(dev), W.to(dev),
                                        epilogue=_dev(epi, dev))
    assert rel_err(np_(y), _ref(lists, T, X, W, epi)) <= TOL[torch.float32]


@pytest.mark.parametrize("S,T,K,cin,cout", [(2999, 1000, 8, 32, 32), (3000, 1000, 8, 32, 32), (3000, 1000, 9, 32, 32),
                                            (3000, 1000, 8, 36, 32), (3000, 1000, 8, 32, 33), (3000, 1000, 8, 5, 7),
                                            (75000, 24999, 8, 16, 20), (75000, 25000, 8, 16, 20)])
def test_fp32_map_of_a_solid_scene(dev, S, T, K, cin, cout):
    """Nearly full maps of three sources per target: both sides of each line of
    the rule that keeps narrow layers on small ones from the compacted kernel."""
    m = np.random.default_rng(K).integers(-S // 15, S, (T, K)).clip(-1).astype(np.int32)
    lists = [(m[m[:, k] >= 0, k], np.nonzero(m[:, k] >= 0)[0]) for k in range(K)]
    X, W, epi = _data(S, T, K, cin, cout, torch.float32, K)
    dm = torch.nn.functional.pad(torch.from_numpy(m), (0, 0, 0, -T % 128), value=-1).to(dev)
    y = F.sparse_convolution_forward_os(S, T, dm, X.to(dev), W.to(dev), epilogue=_dev(epi, dev))
    assert rel_err(np_(y), _ref(lists, T, X, W, epi)) <= TOL[torch.float32]


def _pair_list(lists, dev, unused=0):
    """(naddrs, qnaddrs, nbmaps) on the device; with `unused` every 40th entry
    -1 on one side and that many entries past the last row's."""
    sizes = np.array([len(s) for s, _ in lists])
    naddrs = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    qn = np.concatenate([[0], np.cumsum((sizes + 127) // 128 * 128)]).astype(np.int32)
    nb = np.stack([np.concatenate([s for s, _ in lists]), np.concatenate([t for _, t in lists])]).astype(np.int32)
    if unused:
        nb[0, 7::80] = -1
        nb[1, 47::80] = -1
        nb = np.concatenate([nb, np.zeros((2, unused), np.int32)], 1)
    return [torch.from_numpy(np.ascontiguousarray(a)).to(dev) for a in (naddrs, qn, nb)]


#                S     T    K  cin cout  compacted (fp16, fp32)
PAIR_SHAPES = [(2100, 2000, 27, 64, 64, True, True), (2600, 2500, 8, 96, 100, True, True),
               (900, 901, 40, 128, 64, True, True), (1500, 1400, 8, 96, 100, True, False),
               (900, 901, 40, 128, 48, False, True)]


@pytest.mark.parametrize("repeat", [0, 50, 1])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("S,T,K,cin,cout,half,full", PAIR_SHAPES)
def test_pairs(dev, dtype, S, T, K, cin, cout, half, full, repeat):
    """Lists on both sides of the compacted kernel's rule (repeats aside); rows
    of pairs shuffled, and with `repeat` every so many-th pair given twice (both
    count)."""
    lists = _lists(S, T, K, 0.6, S + K)
    compacted = half if dtype == torch.float16 else full
    X, W, epi = _data(S, T, K, cin, cout, dtype, K)
    pairs = sum(len(s) for s, _ in lists)
    assert _native._C.pairs_compact_pays(pairs, T, K, W) == compacted
    assert _native._C.pairs_compact_pays(pairs, S, K, W) == compacted
    assert not _native._C.pairs_compact_pays(T * K + 1, T, K, W)  # (some must be repeated)
    if repeat:
        lists = [(np.concatenate([s, s[::repeat]]), np.concatenate([t, t[::repeat]])) for s, t in lists]
    naddrs, qn, nb = _pair_list(lists, dev)
    y = F.sparse_convolution_forward_ws_merged(S, T, X.to(dev), W.to(dev), naddrs, qn, nb, nb.shape[1], int(qn[-1]),
                                               epilogue=_dev(epi, dev))
    assert rel_err(np_(y.float()), _ref(lists, T, X, W, epi)) <= TOL[dtype]
    # transposed: sources and targets exchanged
    back = [(t, s) for s, t in lists]
    X2, _, _ = _data(T, S, K, cin, cout, dtype, K + 1)
    y = F.sparse_convolution_forward_ws_merged(T, S, X2.to(dev), W.to(dev), naddrs, qn, nb, nb.shape[1], int(qn[-1]),
                                               True)
    assert rel_err(np_(y.float()), _ref(back, S, X2, W)) <= TOL[dtype]


@pytest.mark.parametrize("unused", [0, 100])
@pytest.mark.parametrize("repeat", [0, 7])
@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("dense", [-1, 0, 3])
def test_mirrored_pairs(dev, dtype, dense, repeat, unused):
    """Half a submanifold layer's pairs, each counted for its mirrored offset
    too: alone (dense -1; the centre row once), or as a hybrid beside an identity
    or a map of dense offsets.  Repeated pairs count twice, entries of -1 and
    past the last row's not at all."""
    S = T = 2501
    K, cin, cout = 27, 64, 64
    rows = 14 if dense < 0 else 12
    rng = np.random.default_rng(dense + 5)
    lists = _lists(S, T, rows, 0.6, 11)
    if repeat:
        lists = [(np.concatenate([s, s[::repeat]]), np.concatenate([t, t[::repeat]])) for s, t in lists]
    naddrs, qn, nb = _pair_list(lists, dev, unused)
    ends = np_(naddrs)
    kept = []
    for r in range(rows):
        s, t = np_(nb)[:, ends[r]:ends[r + 1]]
        ok = (s >= 0) & (t >= 0)
        kept.append((s[ok], t[ok]))
    Kos = {-1: 0, 0: 1, 3: 3}[dense]
    Kw = 27 if dense < 0 else 2 * rows
    full = kept + [(t, s) for s, t in kept[::-1]][Kw % 2:]
    X, W, epi = _data(S, T, Kw + Kos, cin, cout, dtype, 1)
    assert bool(_native._C.pairs_compact_pays(nb.shape[1] * 2 - 2 * T, T, Kw + Kos, W))
    args = (X.to(dev), W.to(dev), naddrs, qn, nb)
    if dense < 0:
        y = F.sparse_convolution_forward_ws_merged(S, T, *args, nb.shape[1], int(qn[-1]), epilogue=_dev(epi, dev))
    else:
        m, first = None, [(np.arange(T), np.arange(T))]
        if dense:
            m = np.maximum(rng.integers(-S, S, (T, Kos)), -1).astype(np.int32)
            first = [(m[m[:, k] >= 0, k], np.nonzero(m[:, k] >= 0)[0]) for k in range(Kos)]
            m = torch.from_numpy(m).to(dev)
        y = F.sparse_convolution_forward_hs_merged(S, T, *args, m, nb.shape[1], int(qn[-1]), epilogue=_dev(epi, dev))
        full = first + full
    assert rel_err(np_(y.float()), _ref(full, T, X, W, epi)) <= TOL[dtype]


def test_values_stay_in_their_rows(dev):
    """An infinity and a NaN reach exactly the targets that have them as a
    neighbour, and unaligned views of the features are taken as they are."""
    S = T = 150
    lists = _lists(S, T, 27, 0.2, 5)
    X, W, _ = _data(S, T, 27, 40, 36, torch.float32, 3)
    m = np.full((256, 27), -1, np.int32)
    for k, (s, t) in enumerate(lists):
        m[t, k] = s
    md = torch.from_numpy(m).to(dev)
    flat = torch.empty(S * 40 + 1, device=dev)
    view = flat[1:].view(S, 40)
    view.copy_(X)
    assert rel_err(np_(F.sparse_convolution_forward_os(S, T, md, view, W.to(dev))), _ref(lists, T, X, W)) <= 1e-5
    X[7], X[90] = float("inf"), float("nan")
    y = np_(F.sparse_convolution_forward_os(S, T, md, X.to(dev), W.to(dev)))
    touched = np.zeros(T, bool)
    for s, t in lists:
        touched[t[(s == 7) | (s == 90)]] = True
    assert not np.isfinite(y[touched]).any(axis=1).any() or np.isnan(y[touched]).any(axis=1).all()
    assert np.isfinite(y[~touched]).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.float32])
@pytest.mark.parametrize("Kd", [1, 2, 8])
def test_hybrid_without_masked_offsets(dev, dtype, Kd):
    """A hybrid of dense offsets alone (Kd 1: the identity), through the C entry
    with the null workspace that its query allows and through the torch layer."""
    lib = ctypes.CDLL(os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "spira_amd",
                                   "libspira_hip.so"))
    S = T = 130
    g = torch.Generator().manual_seed(Kd)
    m = torch.randint(-S, S, (T, Kd), generator=g, dtype=torch.int32).clamp_(min=-1)
    if Kd == 1:
        m = torch.arange(T, dtype=torch.int32)[:, None]
    X, W, _ = _data(S, T, Kd, 32, 48, dtype, Kd)
    lists = [(m[m[:, k] >= 0, k].numpy(), torch.nonzero(m[:, k] >= 0)[:, 0].numpy()) for k in range(Kd)]
    Xd, Wd = X.to(dev), W.to(dev)
    dense = None if Kd == 1 else torch.nn.functional.pad(m, (0, 0, 0, -T % 128), value=-1).to(dev)
    none = torch.empty(0, S, dtype=torch.int32, device=dev)
    y = F.sparse_convolution_forward_hs(S, T, Xd, Wd, none, none, torch.empty(0, dtype=torch.int32, device=dev), dense,
                                        16, 16)
    assert rel_err(np_(y.float()), _ref(lists, T, X, W)) <= TOL[dtype]
    size = ctypes.c_size_t()
    code = 0 if dtype == torch.float16 else 1
    assert lib.spira_hip_fragments_bytes(Kd, 32, 48, code, ctypes.byref(size)) == 0
    frag = torch.empty(max(size.value, 1), dtype=torch.uint8, device=dev)
    out = torch.empty(T, 48, dtype=dtype, device=dev)
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    ptr = lambda t: ctypes.c_void_p(None if t is None else t.data_ptr())
    assert lib.spira_hip_prepare_fragments(ptr(Wd), Kd, 32, 48, code, ptr(frag), stream) == 0
    assert lib.spira_hip_conv_masks(ctypes.c_int64(S), ctypes.c_int64(T), 0, None, None, Kd, ptr(dense), ptr(Xd), 32,
                                    32, ptr(Wd), ptr(frag), 48, code, ptr(out), None, None, None, 0, None,
                                    ctypes.c_size_t(0), stream) == 0
    assert rel_err(np_(out.float()), _ref(lists, T, X, W)) <= TOL[dtype]
