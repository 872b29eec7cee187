"""Radius subsets decided from lattice distances kept on the GPU that computed them."""

import math

import pytest
import torch

from gm_attention_amd.discretization.discretization import SphericalDiscretization
from gm_attention_amd.discretization.grid import build_equiangular_grid



def test_samples_share_their_distances_and_follow_a_move():
    one = SphericalDiscretization.from_grid(build_equiangular_grid(9, 16), 0.9)
    two = one.tile(2)
    six = two.to("cpu", torch.float32).tile(3)
    assert two._exact_distances.data_ptr() == one._exact_distances.data_ptr()
    assert six._exact_distances.numel() == one.n_edges
    for union, count in ((two, 2), (six, 6)):
        want = one.edges_within(0.5).tile(count, n_sources=one.n_nodes)
        got = union.edges_within(0.5)
        assert torch.equal(got.edge_index, want.edge_index) and torch.equal(got.row_ptr, want.row_ptr)

    saved = two.__getstate__() if hasattr(two, "__getstate__") else None
    saved = dict(saved or two.__dict__)  # as pickled before distances were shared: repeated, and no count
    saved["_exact_distances"] = saved["_exact_distances"].repeat(saved.pop("_exact_copies"))
    older = SphericalDiscretization.__new__(SphericalDiscretization)
    older.__dict__.update(saved, _radius_cache={})
    assert torch.equal(older.edges_within(0.5).edge_index, two.edges_within(0.5).edge_index)

    class OnAnotherGpu:
        device = torch.device("cuda:0")
        moved_to = None

        def detach(self):
            return self

        def to(self, where):
            if isinstance(where, str):
                self.moved_to = where
            return self

    one._exact_distances = held = OnAnotherGpu()
    one.to(dtype=torch.float32)
    assert held.moved_to is None
    one.to("cpu")
    assert held.moved_to == "cpu"


@pytest.mark.gpu
@pytest.mark.parametrize("nlat,nlon", [(16, 32), (19, 36)])
def test_radius_subsets_are_the_same_wherever_the_distances_live(nlat, nlon, cuda):
    """Whole shells (radii on the lattice's own spacing) chosen on the GPU, on the
    host copy, after a move back, and tiled: the same edges bit for bit, and
    nothing of a discretization on the host left on the GPU."""
    step = math.pi / (nlat - 1)
    here = SphericalDiscretization.from_grid(build_equiangular_grid(nlat, nlon, device=cuda), 4 * step)
    assert here._exact_distances.device.type == "cuda" and here._exact_distances.dtype == torch.float64
    host = here.to("cpu")
    back = host.to(cuda)
    assert host._exact_distances.device.type == "cpu"
    for k in (1, 2, 3):
        want = host.edges_within(k * step)
        assert want.edge_index.device.type == "cpu" and 0 < want.n_edges < host.n_edges
        for disc in (here, back):
            got = disc.edges_within(k * step)
            assert got.edge_index.device.type == "cuda"
            assert torch.equal(got.edge_index.cpu(), want.edge_index) and torch.equal(got.row_ptr.cpu(), want.row_ptr)
            assert torch.equal(got.distances.cpu(), want.distances)
    pair, pair_host = here.tile(2).edges_within(1.5 * step), host.tile(2).edges_within(1.5 * step)
    assert torch.equal(pair.edge_index.cpu(), pair_host.edge_index)
