"""Several heads of the grouped factored kernels in one launch
(gm_factored_{forward,backward}_heads_f32) against a launch a head: the same
kernels on the same streams, so every output and gradient is the same, bit
for bit.  Over compiled-in lane slots, runtime slots and the generic kernels,
heads cut into shares (accumulating dh), odd head counts and group counts that
are no multiple of the eight XCDs."""

import pytest
import torch

import problems
from gm_attention_amd.nn import fused_factored
from gm_attention_amd.nn.attention import SO2MHSA
from gm_attention_amd.representations.field_type import SO2FeatureField, SO2FieldType

pytestmark = pytest.mark.gpu

CASES = [  # field, heads, grid
    ({0: 8, 1: 8, 2: 8}, 2, (9, 17)),  # compiled-in slots, frequencies 0..2; 153 groups
    ({0: 12, 1: 12}, 3, (8, 16)),  # compiled-in slots, frequencies 0..1; an odd head count
    ({0: 16, 1: 8}, 2, (9, 16)),  # runtime slots
    ({0: 6, 1: 4, 2: 2}, 2, (7, 15)),  # the generic kernels
    ({0: 32, 1: 32, 2: 32}, 4, (7, 14)),  # two shares a head
    ({0: 64, 1: 64, 2: 64}, 16, (6, 13)),  # sixteen heads
]


@pytest.mark.parametrize("field,heads,grid", CASES)
def test_heads_in_one_launch_equal_a_launch_a_head(field, heads, grid, cuda, monkeypatch):
    print(f"heads in one launch {field} x{heads} {grid}", flush=True)
    disc = problems.discretization(*grid)
    edges = disc.edge_geometry.to(cuda, torch.float32)
    ft = SO2FieldType(field)
    torch.manual_seed(0)
    mhsa = SO2MHSA(ft, heads, cutoff=disc.coverage_radius, batched=True, dtype=torch.float32, device=cuda)
    x = problems.normal((edges.row_ptr.shape[0] - 1, ft.dimension), 1).float().to(cuda).requires_grad_(True)
    probe = problems.normal(tuple(x.shape), 2).float().to(cuda)
    params = [x, *mhsa.parameters()]

    def run():
        out = mhsa(SO2FeatureField.from_flat(ft, x), edges).to_flat()
        return [out.detach(), *torch.autograd.grad(out, params, probe)]

    used = []
    real = fused_factored._together
    monkeypatch.setattr(fused_factored, "_together", lambda *a: used.append(real(*a)) or used[-1])
    together = run()
    assert used == [True, True]
    monkeypatch.setattr(fused_factored, "_together", lambda *a: False)
    for a, b in zip(together, run(), strict=True):
        assert torch.equal(a, b)
