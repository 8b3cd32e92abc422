"""num_neighbors_image is written by the build's last kernel: grid and all-pairs builds, with and
without vectors, targets and edges."""
import pytest
import torch

from dynamis_amd import configs
from dynamis_amd.dynamis_state import dynamis_state_impl as impl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vectors", [False, True])
@pytest.mark.parametrize("n,length,r,nt", [(3000, 31.0, 6.0, None), (3000, 31.0, 6.0, 17), (4, 3.0, 6.0, None),
                                           (2, 200.0, 3.0, None), (40000, 74.0, 5.0, 20011)])
def test_number_of_edges(cuda, n, length, r, nt, vectors):
    box = configs.uniform(n, seed=3)
    pos = torch.from_numpy(box.pos).double()
    pos = (pos / pos.max() * length).float().to(cuda)
    cell, pbc = torch.eye(3, dtype=torch.float64) * length, torch.tensor([True] * 3)
    t = None if nt is None else torch.arange(nt, device=cuda)
    for _ in range(2):
        if vectors:
            out = impl.radius_graph_pbc_vectors(pos, cell, pbc, r, t)
        else:
            out = impl.radius_graph_pbc_ex(pos, cell, pbc, r, 0, False, t)
        ei, nn = out[0], out[2]
        assert nn.dtype == torch.int64 and nn.shape == (1,) and int(nn) == ei.shape[1]
