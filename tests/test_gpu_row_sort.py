"""The batched row orders' own sort at the edges of its 2048-key tiles and of
its size limit, against each map's order alone (which another sort makes):
random rows, rows that are all alike (stability) and few distinct rows."""
import pytest
import torch

from spira_amd.nn.functional import _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["random", "alike", "few"])
@pytest.mark.parametrize("Ts", [(1, 1), (2047, 1), (1000, 1049), (2048,) * 16, (4000, 97, 2048, 300), (300000, 250001),
                                (400000, 299999), (400000, 300001)])
def test_batch_equals_single(dev, Ts, kind):
    C = _native._C
    g = torch.Generator(device=dev).manual_seed(len(Ts))
    maps = []
    for q, T in enumerate(Ts):
        K = (27, 9, 18)[q % 3]
        if kind == "random":
            m = torch.randint(-3, 3, (T, K), generator=g, device=dev, dtype=torch.int32).clamp_(min=-1)
        elif kind == "alike":
            m = torch.arange(K, device=dev, dtype=torch.int32).sub_(q % 5).clamp_(min=-1).expand(T, K).contiguous()
        else:
            few = torch.randint(-1, 1, (7, K), generator=g, device=dev, dtype=torch.int32)
            m = few[torch.randint(0, 7, (T,), generator=g, device=dev)]
        maps.append(torch.nn.functional.pad(m, (0, 0, 0, -T % 128), value=-1))
    C.prepare_row_orders(maps, list(Ts), [1] * len(Ts))
    for m, T in zip(maps, Ts):
        for a, b in zip(C.kmap_row_order(m, T), C.kmap_row_order(m.clone(), T)):
            assert torch.equal(a, b), (T, m.shape)
