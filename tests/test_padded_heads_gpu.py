"""Heads padded to the compiled-in lane slots' four copies a frequency
(fused_factored.PaddedHead) against the heads' own plans (no padding: the
generic grouped kernels, runtime lane slots or the kernels that are not
grouped), float32 and bfloat16 rows: the same sums in another order.

The bound: both sides are float32 evaluations of one function, so within a few
times sqrt(depth) 2^-24 of each other in norm; the deepest chain of a value is
17 x 2 b products, then the neighbourhood's edges (up to 96 here), then 12 to
32 columns of the projection, some 300 additions: 4 sqrt(300) 2^-24 = 4e-6.
Bfloat16 rows share their rounded inputs, and round their gradient: 2^-8."""

import pytest
import torch

import problems
from gm_attention_amd.nn import fused_factored
from gm_attention_amd.nn.attention import SO2MHSA
from gm_attention_amd.representations.field_type import SO2FeatureField, SO2FieldType

pytestmark = pytest.mark.gpu

CASES = [  # field, heads, shares a head
    ({0: 6, 1: 4, 2: 2}, 2, 1),
    ({0: 1, 1: 1, 2: 1}, 1, 1),
    ({0: 4, 1: 2}, 2, 1),
    ({0: 10, 1: 6, 2: 2}, 2, 2),  # (5, 3, 1): copies that no split divides
    ({0: 16, 1: 8, 2: 4}, 2, 2),
    ({0: 8, 1: 4, 2: 4}, 1, 2),  # runtime lane slots on their own
    ({0: 27, 1: 3, 2: 3}, 3, 3),
]


@pytest.mark.parametrize("bf16", [False, True])
@pytest.mark.parametrize("field,heads,shares", CASES)
def test_padded_heads_equal_their_own_plans(field, heads, shares, bf16, cuda, monkeypatch):
    print(f"padded heads {field} x{heads} bf16={bf16}", flush=True)
    disc = problems.discretization(9, 17)
    edges = disc.edge_geometry.tile(2, n_sources=disc.n_nodes).to(cuda, torch.float32)
    ft = SO2FieldType(field)
    torch.manual_seed(0)
    mhsa = SO2MHSA(ft, heads, cutoff=disc.coverage_radius, batched=True, dtype=torch.float32, device=cuda)
    n = edges.row_ptr.shape[0] - 1
    x = problems.normal((n, ft.dimension), 1).to(cuda, torch.bfloat16 if bf16 else torch.float32).requires_grad_(True)
    probe = problems.normal(tuple(x.shape), 2).float().to(cuda)
    values = [h.value for h in mhsa.heads]
    if bf16 and fused_factored.declined(values[0], SO2FeatureField.from_flat(ft, x), edges):
        pytest.skip("the value kernel does not take bfloat16 rows")
    if bf16 and (heads not in (1, 2, 4, 8, 16)
                 or any(m // heads * (1 if f == 0 else 2) % 4 for f, m in field.items())):
        pytest.skip("the scores take bfloat16 rows of a power of two heads of whole quads of reals")

    def run():
        out = mhsa(SO2FeatureField.from_flat(ft, x), edges).to_flat()
        grads = torch.autograd.grad(out.float(), [x, *mhsa.parameters()], probe)
        return out.detach().float(), grads[0].float(), torch.cat([g.reshape(-1) for g in grads[1:]])

    def layout():
        return fused_factored.heads_layout(values, torch.float32, None, (n, edges.n_edges), x.device)

    assert layout().padded and layout().split == shares
    got = run()
    monkeypatch.setattr(fused_factored, "PADDED_SHARE", 0.0)  # no memory for padding: the heads' own plans
    assert not layout().padded
    for name, a, b in zip(("out", "dx", "dparameters"), got, run(), strict=True):
        err = float((a - b).norm() / b.norm())
        assert err <= (2.0 ** -8 if bf16 and name == "dx" else 4e-6), f"{name}: {err:.2e}"


@pytest.mark.parametrize("field,heads", [({0: 8, 1: 8, 2: 8}, 2), ({0: 32, 1: 32, 2: 32}, 4), ({0: 8, 1: 8}, 2)])
def test_heads_of_the_compiled_in_slots_are_not_padded(field, heads, cuda):
    mhsa = SO2MHSA(SO2FieldType(field), heads, cutoff=0.3, batched=True, dtype=torch.float32, device=cuda)
    layout = fused_factored.heads_layout([h.value for h in mhsa.heads], torch.float32, None, (100, 4000), cuda)
    assert layout.grouped and not layout.padded
