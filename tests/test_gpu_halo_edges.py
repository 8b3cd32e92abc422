"""The halo plan's edge pass with the local atoms' bits in LDS and not: atom counts at the two
lines between (262144 and 1310720 atoms; fewer than 4M edges), a last word and a last round of
edges that are partial, against the halo oracle; indices out of range are refused by both."""
import numpy as np
import pytest
import torch

from oracle import halo
from dynamis_amd.dynamis_state import dynamis_state_impl as impl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,E,W", [(262_145, 4_000_001, 3), (262_144, 4_000_001, 3), (1_310_720, 4_194_304, 8),
                                   (1_310_721, 4_000_000, 8), (300_003, 3_999_999, 70), (77, 1, 1)])
def test_edges_around_the_lines(cuda, N, E, W):
    print(f"\n[case] halo edges N={N} E={E} W={W}", flush=True)
    rng = np.random.default_rng(N + E)
    # slabs of ids, so that most sources are the rank's own; a few far ones, in runs of one target
    pid = np.arange(N) * W // N
    R = W // 2
    my = np.nonzero(pid == R)[0]
    dst = np.sort(rng.choice(my, E))
    src = rng.choice(my, E)
    far = rng.random(E) < 0.1
    src[far] = rng.integers(0, N, int(far.sum()))
    src[-1] = N - 1
    edges = torch.from_numpy(np.stack([src, dst])).to(cuda)
    p, m = torch.from_numpy(pid).to(cuda), torch.from_numpy(my).to(cuda)
    got = impl.extract_halo_info(edges, p, m, R, W, N)
    want = halo.extract_halo_info(src, dst, pid, my, R, W, N)
    for g, w in zip(got, want):
        assert np.array_equal(g.cpu().numpy(), w)
    for bad in (N, -1):
        e2 = edges.clone()
        e2[0, E // 2] = bad
        with pytest.raises(RuntimeError, match="out of range"):
            impl.extract_halo_info(e2, p, m, R, W, N)
    p[N - 1] = W  # (the last edge's source)
    with pytest.raises(RuntimeError, match="out of range"):
        impl.extract_halo_info(edges, p, m, R, W, N)
