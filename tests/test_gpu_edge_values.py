"""The frames of a graph's edges from its row offsets (mlcg_edge_values):
whole numbers, equal to the index lookup they replace."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 32, 33, 4099])
@pytest.mark.parametrize("longest", [0, 3, 64, 200])
def test_edge_values_equals_lookup(n, longest):
    from mlcg_amd import ops

    g = torch.Generator().manual_seed(n + longest)
    count = torch.randint(0, longest + 1, (n,), generator=g)  # rows without edges among them
    rowptr = torch.cat([torch.zeros(1, dtype=torch.long), count.cumsum(0)]).int().cuda()
    values = torch.randint(-2 ** 40, 2 ** 40, (n,), generator=g).cuda()
    rows = torch.repeat_interleave(torch.arange(n), count).cuda()
    graph = ops.PairGraph(edge_index=None, rowptr=rowptr, col=None, pair_ij=None, pairptr=None,
                          eid2pair=None, frame_ptr=None, num_nodes=n, num_edges=rows.numel(),
                          num_pairs=0)
    assert torch.equal(ops.edge_values(graph, values), values[rows])
