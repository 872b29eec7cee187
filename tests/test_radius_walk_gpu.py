"""The neighbour walk at the edges of its tiles: one target to several waves of
sixteen, one source to more than 64 boxes of 64."""

import pytest
import torch

from gm_attention_amd import _native

pytestmark = pytest.mark.gpu


def unit(n, seed):
    x = torch.randn(n, 3, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    x = x / x.norm(dim=1, keepdim=True)
    return x / x.norm(dim=1, keepdim=True)


@pytest.mark.parametrize("n_targets", [1, 15, 16, 17, 65, 1025, 16385])
@pytest.mark.parametrize("n_sources", [1, 63, 64, 65, 4096, 4097])
def test_walk_is_bit_exact_at_tile_edges(n_targets, n_sources, cuda):
    """Integers: equal to every pair tested by the same float64 rule; a row of
    every source, one of none, and the prefix sums over each share of the scan."""
    targets, sources = unit(n_targets, 1), unit(n_sources, 2)
    for limit in (0.05, 0.9) if n_targets < 5000 else (0.05,):
        edge_index, row_ptr = _native.radius_edges(targets.to(cuda), sources.to(cuda), limit)
        p, q = targets.to(cuda)[:, None], sources.to(cuda)[None]
        member = torch.cat([torch.atan2(torch.linalg.cross(*torch.broadcast_tensors(a, q)).norm(dim=-1),
                                        (a * q).sum(-1).clamp(-1, 1)) <= limit for a in p.split(512)])
        want = member.nonzero().t()
        assert torch.equal(edge_index, want)
        assert torch.equal(row_ptr[1:], member.sum(1).cumsum(0)) and int(row_ptr[0]) == 0
