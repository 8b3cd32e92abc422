"""The radix sort's scan of each digit's tile counts at its edges: one tile, a tile and a key, a
round of tiles and one more, against torch's stable sort; keys that fill one digit, or all."""
import pytest
import torch

from dynamis_amd.dynamis_state import dynamis_state_impl as impl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("span", [1, 3, 256, 70000, 2 ** 62])
@pytest.mark.parametrize("n", [1, 2047, 2048, 2049, 5000, 2048 * 1024, 2048 * 1024 + 1])
def test_order_of_n_keys(cuda, n, span):
    print(f"\n[case] order n={n} span={span}", flush=True)
    g = torch.Generator().manual_seed(n + span)
    keys = torch.randint(-(span // 2), span - span // 2, (n,), generator=g)
    got = impl.sfc_order(keys.to(cuda))
    assert torch.equal(got.cpu(), torch.sort(keys, stable=True).indices)
