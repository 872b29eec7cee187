"""Several heads of the grouped factored kernels in one launch
(gm_factored_{forward,backward}_heads_f32) against a launch a head: the same
kernels on the same streams, so every output and gradient is the same, bit
for bit.  Over compiled-in lane slots, runtime slots and the generic kernels,
heads cut into shares (accumulating dh), odd head counts and row widths, and
group counts that are no multiple of the eight XCDs.  Each case names the
kernels it is there for and checks that they run."""

import pytest
import torch

import problems
from gm_attention_amd import _native
from gm_attention_amd.nn import fused_factored
from gm_attention_amd.nn.attention import SO2MHSA
from gm_attention_amd.representations.field_type import SO2FeatureField, SO2FieldType

pytestmark = pytest.mark.gpu

CASES = [  # field, heads, grid, the kernels that run, shares a head
    ({0: 8, 1: 8, 2: 8}, 2, (9, 17), "compiled-in", 1),  # frequencies 0..2; 153 groups
    ({0: 12, 1: 12}, 3, (8, 16), "compiled-in", 1),  # frequencies 0..1; an odd head count
    ({0: 16, 1: 8}, 2, (9, 16), "runtime", 1),
    ({0: 6, 1: 4, 2: 2}, 2, (7, 15), "generic", 1),  # nine reals a row, 105 targets
    ({0: 9, 1: 6, 2: 3}, 3, (7, 13), "generic", 1),  # and an odd head count
    ({0: 32, 1: 32, 2: 32}, 4, (7, 14), "compiled-in", 2),
    ({0: 64, 1: 64, 2: 64}, 16, (6, 13), "compiled-in", 1),
]


def _layer(field, heads, grid, form, shares, cuda, monkeypatch):
    """The layer with its heads on their own plans (no memory for padding), on the kernels the case names."""
    monkeypatch.setattr(fused_factored, "PADDED_SHARE", 0.0)
    disc = problems.discretization(*grid)
    edges = disc.edge_geometry.to(cuda, torch.float32)
    ft = SO2FieldType(field)
    torch.manual_seed(0)
    mhsa = SO2MHSA(ft, heads, cutoff=disc.coverage_radius, batched=True, dtype=torch.float32, device=cuda)
    x = problems.normal((edges.row_ptr.shape[0] - 1, ft.dimension), 1).float().to(cuda).requires_grad_(True)
    probe = problems.normal(tuple(x.shape), 2).float().to(cuda)
    params = [x, *mhsa.parameters()]
    size = (x.shape[0], edges.n_edges)
    layout = fused_factored.heads_layout([h.value for h in mhsa.heads], torch.float32, None, size, cuda)
    assert layout.grouped and not layout.padded and layout.split == shares
    lanes = fused_factored._lanes_apply(layout.unit, layout.hp, layout.pa, layout.pt)
    fixed = fused_factored._lanes_fixed(layout.unit, layout.hp, layout.pa, layout.pt)
    assert form == ("compiled-in" if fixed else "runtime" if lanes else "generic")

    def run():
        out = mhsa(SO2FeatureField.from_flat(ft, x), edges).to_flat()
        return [out.detach(), *torch.autograd.grad(out, params, probe)]

    return run


@pytest.mark.parametrize("field,heads,grid,form,shares", CASES)
def test_heads_in_one_launch_equal_a_launch_a_head(field, heads, grid, form, shares, cuda, monkeypatch):
    print(f"heads in one launch {field} x{heads} {grid}", flush=True)
    run = _layer(field, heads, grid, form, shares, cuda, monkeypatch)
    used = []
    real = fused_factored._together
    monkeypatch.setattr(fused_factored, "_together", lambda *a: used.append(real(*a)) or used[-1])
    together = run()
    assert used == [True, True]
    monkeypatch.setattr(fused_factored, "_together", lambda *a: False)
    for a, b in zip(together, run(), strict=True):
        assert torch.equal(a, b)


@pytest.mark.parametrize("together", [True, False])
@pytest.mark.parametrize("field,heads,grid,form,shares", [CASES[0], CASES[2], CASES[3], CASES[5]])
def test_phase_rows_are_absent_where_nothing_reads_them(field, heads, grid, form, shares, together, cuda, monkeypatch):
    """Plans on compiled-in slots run without phase rows, bit for bit as with
    them; the entries refuse the other plans' calls without them, before any
    launch."""
    print(f"phase rows {field} x{heads} {grid} together={together}", flush=True)
    run = _layer(field, heads, grid, form, shares, cuda, monkeypatch)
    monkeypatch.setattr(fused_factored, "_STREAMS", type(fused_factored._STREAMS)())
    if not together:
        monkeypatch.setattr(fused_factored, "_together", lambda *a: False)
    forward, backward, calls = _native.factored_forward_grouped, _native.factored_backward_grouped, []

    def refused(call, at, args, kwargs):
        phases = args[at]
        calls.append(phases is None)
        if phases is not None and form != "compiled-in":
            with pytest.raises(RuntimeError, match="phase rows"):
                call(*args[:at], None, *args[at + 1:], **kwargs)

    monkeypatch.setattr(_native, "factored_forward_grouped",
                        lambda *a, **k: (refused(forward, 3, a, k), forward(*a, **k))[1])
    monkeypatch.setattr(_native, "factored_backward_grouped",
                        lambda *a, **k: (refused(backward, 7, a, k), backward(*a, **k))[1])
    got = run()
    assert calls and all(absent == (form == "compiled-in") for absent in calls)
    streams = fused_factored.grouped_streams
    monkeypatch.setattr(fused_factored, "grouped_streams", lambda *a: streams(*a[:6], True))
    calls.clear()
    want = run()
    assert calls and not any(calls)
    for a, b in zip(got, want, strict=True):
        assert torch.equal(a, b)
