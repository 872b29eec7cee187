"""Assembled parameter forms (nn/assembly.py): the plan's gather and its
transposed gather against the construction itself and its autograd gradient,
by evaluating the codes in torch on the CPU, and the HIP launch on the GPU
(moves and sign changes: bit for bit; gradients: the uses of an entry added)."""

import copy
import gc
import inspect
import pickle
import threading
import time
import weakref

import pytest
import torch

from gm_attention_amd.nn import assembly
from gm_attention_amd.nn.attention import SO2MHSA, _LayerForms
from gm_attention_amd.nn.linear import complex_as_real
from gm_attention_amd.representations.field_type import SO2FieldType


def _build(ps):
    """Stacks, transposes, negated entries, repeats, zeros, an unused and a repeatedly used parameter."""
    a, b, c, _unused, d = ps
    m = a.new_zeros(9, 8)
    m[:4, :6] = complex_as_real(a)
    m[5:, 2:5] = b.t()
    return [m, torch.cat([c, -c, c.new_zeros(3)]), torch.stack([d] * 5), d.reshape(1, 1)]


SHAPES = [(3, 2, 2), (3, 4), (7,), (5, 5), (1,)]


def _params(device="cpu", dtype=torch.float32):
    g = torch.Generator().manual_seed(3)
    return [torch.randn(s, generator=g).to(device, dtype) for s in SHAPES]


def _gather(sources, codes):
    """What gm_signed_gather_f32 computes, by its definition."""
    out = torch.zeros(codes.shape[1], dtype=torch.float64)
    for row in codes.cpu():
        for e, code in enumerate(row.tolist()):
            if code >= 0 and sources[code >> 40] is not None:
                x = float(sources[code >> 40].reshape(-1)[(code >> 1) & ((1 << 39) - 1)])
                out[e] += -x if code & 1 else x
    return out


def test_plan_codes_restate_the_construction_and_its_gradient():
    params = [p.double().requires_grad_(True) for p in _params()]
    plan = assembly.Plan(tuple(p.shape for p in params), _build, torch.device("cpu"))
    want = _build(params)
    flat = _gather([p.detach() for p in params], plan.codes)
    for w, start, shape in zip(want, plan.out_starts, plan.form_shapes):
        assert torch.equal(flat[start:start + shape.numel()].view(shape), w.detach())
    up = [torch.randn_like(w) for w in want]
    up[1] = None  # a form nothing reads has no gradient
    grads = torch.autograd.grad([w for w, u in zip(want, up) if u is not None], params,
                                [u for u in up if u is not None], allow_unused=True)
    back = _gather(up, plan.gradient_codes())
    for p, g, start in zip(params, grads, plan.in_starts):
        got = back[start:start + p.numel()].view(p.shape)
        assert torch.allclose(got, torch.zeros_like(p) if g is None else g, rtol=0, atol=1e-14)


def test_parameters_the_kernel_does_not_take_go_through_the_construction():
    class Owner:
        pass

    params = [p.requires_grad_(True) for p in _params()]
    got = assembly.assembled(Owner(), "x", params, _build)  # CPU
    for g, w in zip(got, _build(params)):
        assert torch.equal(g, w) and g.grad_fn is not None


class _Owner:
    pass


@pytest.fixture
def on_cpu(monkeypatch):
    """Assembly on the CPU: the launch replaced by its definition."""
    monkeypatch.setattr(assembly, "takes", lambda params: True)
    monkeypatch.setattr(assembly, "_gather", lambda sources, codes, made_on: _gather(sources, codes).float())
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def test_the_gradients_table_is_there_before_any_backward(on_cpu, monkeypatch):
    """A backward runs on a thread, and perhaps a stream, of its own: it finds its table complete."""
    owner, params, plans = _Owner(), [p.requires_grad_(True) for p in _params()], []
    find = assembly.Plan.__init__
    monkeypatch.setattr(assembly.Plan, "__init__", lambda self, *a: (find(self, *a), plans.append(self))[0])
    with torch.no_grad():
        assembly.assembled(owner, "x", params, _build)
    assert plans[0].back is None  # inference needs none
    got = assembly.assembled(owner, "x", params, _build)
    assert len(plans) == 1 and plans[0].back is not None
    up = [torch.randn_like(g) for g in got]
    want = torch.autograd.grad(_build(params), params, up, allow_unused=True)
    for g, w in zip(torch.autograd.grad(got, params, up), want):
        assert torch.allclose(g, torch.zeros_like(g) if w is None else w, rtol=0, atol=1e-6)


def test_threads_finding_one_table_agree(monkeypatch):
    plan = assembly.Plan(tuple(p.shape for p in _params()), _build, torch.device("cpu"))
    want = assembly.Plan(plan.shapes, _build, torch.device("cpu")).gradient_codes()
    code = assembly.Plan._code

    def slowly(*args):
        time.sleep(0.05)
        return code(*args)

    monkeypatch.setattr(assembly.Plan, "_code", staticmethod(slowly))
    start, got = threading.Barrier(8), []

    def find():
        start.wait()
        time.sleep(0.01 * len(got))
        got.append(plan.gradient_codes())

    threads = [threading.Thread(target=find) for _ in range(8)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert len(got) == 8 and all(g is got[0] for g in got) and torch.equal(got[0], want)


def test_modules_with_plans_list_copy_and_pickle_without_them(on_cpu):
    from gm_attention_amd.nn.normalization import SO2LayerNorm

    field = SO2FieldType({0: 4, 1: 3})
    plain, norm = SO2LayerNorm(field), SO2LayerNorm(field)
    want = norm.gamma_flat(torch.float32)
    assert set(norm.__dict__) == set(plain.__dict__)
    assert len(assembly._PLANS[norm]) == 1
    assert dir(norm) == dir(plain) and len(inspect.getmembers(norm)) == len(inspect.getmembers(plain))
    assert len(pickle.dumps(norm)) == len(pickle.dumps(plain))
    for copied in (copy.deepcopy, lambda m: pickle.loads(pickle.dumps(m))):
        other = copied(norm)
        assert other not in assembly._PLANS
        assert torch.equal(other.gamma_flat(torch.float32), want)
        plan = weakref.ref(next(iter(assembly._PLANS[other].values())))
        del other
        gc.collect()
        assert plan() is None  # gone with its module


def test_shapes_and_devices_have_plans_of_their_own(on_cpu):
    owner = _Owner()
    params = _params()
    wider = [p.repeat(2, *([1] * (p.dim() - 1))) if i == 2 else p for i, p in enumerate(params)]
    for ps in (params, wider, params):
        for g, w in zip(assembly.assembled(owner, "x", ps, _build), _build(ps)):
            assert torch.equal(g, w)
    assert len(assembly._PLANS[owner]) == 2


def test_replicas_of_a_data_parallel_step_find_no_plans(on_cpu):
    from gm_attention_amd.nn.normalization import SO2LayerNorm

    norm = SO2LayerNorm(SO2FieldType({0: 4, 1: 3}))
    replica = norm._replicate_for_data_parallel()
    replica.gamma = norm.gamma
    got = replica.gamma_flat(torch.float32)
    assert replica not in assembly._PLANS and torch.equal(got, norm.gamma_flat(torch.float32))


def test_a_plan_found_in_inference_mode_trains(on_cpu):
    owner, params = _Owner(), [p.requires_grad_(True) for p in _params()]
    with torch.inference_mode():
        assembly.assembled(owner, "x", params, _build)
    got = assembly.assembled(owner, "x", params, _build)
    up = [torch.randn_like(g) for g in got]
    want = torch.autograd.grad(_build(params), params, up, allow_unused=True)
    for g, w in zip(torch.autograd.grad(got, params, up), want):
        assert torch.allclose(g, torch.zeros_like(g) if w is None else w, rtol=0, atol=1e-6)


def test_second_derivatives_are_the_constructions(on_cpu):
    owner, params = _Owner(), [p.requires_grad_(True) for p in _params()]
    torch.manual_seed(2)
    probes = [torch.randn_like(w) for w in _build(params)]
    probes[3] = None  # a form nothing reads

    def twice(forms):
        loss = sum((f ** 3 * p).sum() for f, p in zip(forms, probes) if p is not None)
        first = torch.autograd.grad(loss, params, create_graph=True, allow_unused=True)
        first = [torch.zeros_like(p) if g is None else g for g, p in zip(first, params)]
        second = torch.autograd.grad(sum((g ** 2).sum() for g in first), params, allow_unused=True)
        return [*first, *(torch.zeros_like(p) if g is None else g for g, p in zip(second, params))]

    for g, w in zip(twice(assembly.assembled(owner, "x", params, _build)), twice(_build(params)), strict=True):
        assert torch.allclose(g, w, rtol=1e-5, atol=1e-5)


def test_transforms_are_followed_through_the_construction(monkeypatch):
    from torch.autograd import forward_ad

    seen = []
    look = lambda x: seen.append(assembly._transformed()) or 2 * x  # noqa: E731
    one = torch.ones(2)
    look(one)
    torch.func.grad(lambda x: look(x).sum())(one)
    torch.vmap(look)(one)
    torch.func.jvp(look, (one,), (one,))
    with forward_ad.dual_level():
        look(one)
    before = len(seen)
    torch.jit.trace(look, one, check_trace=False)
    assert seen[:before] == [False, True, True, True, True] and all(seen[before:]) and len(seen) > before


@pytest.mark.gpu
def test_transforms_and_second_derivatives_of_norms_gains_on_the_gpu(cuda):
    from torch.autograd import forward_ad

    from gm_attention_amd.nn.normalization import SO2LayerNorm

    norm = SO2LayerNorm(SO2FieldType({0: 5, 2: 3}), dtype=torch.float32, device=cuda)
    gains = {f"gamma.{f}": torch.randn_like(p) for f, p in norm.gamma.items()}

    def flat(g):
        return torch.func.functional_call(_Gains(norm), {f"norm.{k}": v for k, v in g.items()}, ())

    want = torch.cat([gains["gamma.0"], gains["gamma.2"].repeat_interleave(2)])
    assert torch.equal(flat(gains), want)
    grads = torch.func.grad(lambda g: (flat(g) ** 2).sum())(gains)
    assert torch.allclose(grads["gamma.0"], 2 * gains["gamma.0"]) and torch.allclose(grads["gamma.2"], 4 * gains["gamma.2"])
    many = torch.vmap(flat)({k: torch.stack([v, 2 * v]) for k, v in gains.items()})
    assert torch.equal(many, torch.stack([want, 2 * want]))
    with forward_ad.dual_level():
        out = flat({k: forward_ad.make_dual(v, torch.ones_like(v)) for k, v in gains.items()})
        assert torch.equal(forward_ad.unpack_dual(out).tangent, torch.ones_like(want))
    leaves = [g.clone().requires_grad_(True) for g in gains.values()]
    first = torch.autograd.grad((flat(dict(zip(gains, leaves))) ** 3).sum(), leaves, create_graph=True)
    second = torch.autograd.grad(sum(g.sum() for g in first), leaves)
    assert torch.allclose(second[0], 6 * leaves[0]) and torch.allclose(second[1], 12 * leaves[1])


class _Gains(torch.nn.Module):
    def __init__(self, norm):
        super().__init__()
        self.norm = norm

    def forward(self):
        return self.norm.gamma_flat(torch.float32)


def test_a_captured_stream_without_a_plan_takes_the_construction(on_cpu, monkeypatch):
    owner, params = _Owner(), [p.requires_grad_(True) for p in _params()]
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    for g, w in zip(assembly.assembled(owner, "x", params, _build), _build(params)):
        assert torch.equal(g, w)
    assert owner not in assembly._PLANS
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    with torch.no_grad():
        assembly.assembled(owner, "x", params, _build)
    plan = next(iter(assembly._PLANS[owner].values()))
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assembly.assembled(owner, "x", params, _build)
    assert plan.back is None  # no gradient table is found under capture either


@pytest.mark.gpu
@pytest.mark.parametrize("train", [False, True])
def test_first_calls_of_norm_gate_and_linear_under_capture(train, cuda):
    """Modules that have run nothing yet, captured forward (and backward): replays
    between eager work equal the eager results, bit for bit forward."""
    from gm_attention_amd.nn.linear import SO2Linear, flat_forward
    from gm_attention_amd.nn.nonlinearities import SO2ScalarGatedNonlinearity
    from gm_attention_amd.nn.normalization import SO2LayerNorm

    field = SO2FieldType({0: 8, 1: 4, 2: 4})
    torch.manual_seed(0)
    made = dict(dtype=torch.float32, device=cuda)
    norm, gate, lin = SO2LayerNorm(field, **made), SO2ScalarGatedNonlinearity(field, **made), SO2Linear(field, field, **made)
    params = [p for m in (norm, gate, lin) for p in m.parameters()]
    x = torch.randn(50, field.dimension, device=cuda, requires_grad=train)
    up = torch.randn(50, field.dimension, device=cuda)

    def step(norm, gate, lin, params):
        with torch.set_grad_enabled(train):
            out = flat_forward(lin, gate.forward_flat(norm.forward_flat(x)))
        return (out.detach(), *torch.autograd.grad(out, [x, *params], up)) if train else (out,)

    # the libraries' handles come up on another set of modules
    others = [copy.deepcopy(m) for m in (norm, gate, lin)]
    with torch.cuda.stream(torch.cuda.Stream()):
        want = step(*others, [p for m in others for p in m.parameters()])
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = step(norm, gate, lin, params)
    for value in (x.detach().clone(), torch.randn_like(x), torch.randn_like(x)):
        with torch.no_grad():
            x.copy_(value)
        graph.replay()
        torch.cuda.synchronize()
        want = step(*others, [p for m in others for p in m.parameters()])
        assert torch.equal(got[0], want[0])
        for g, w in zip(got[1:], want[1:], strict=True):
            assert torch.allclose(g, w, rtol=1e-5, atol=1e-5)
        torch.cuda.synchronize()


@pytest.mark.gpu
def test_tables_found_behind_a_busy_stream_are_complete_for_another(cuda):
    owner, params = _Owner(), [p.requires_grad_(True) for p in _params(cuda)]
    want = _build(params)
    up = [torch.randn_like(w) for w in want]
    ref = torch.autograd.grad(want, params, up, allow_unused=True)
    first, second = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(first):
        torch.cuda._sleep(100_000_000)  # some tens of milliseconds ahead of the tables
        assembly.Plan(tuple(p.shape for p in params), _build, cuda)
        assert first.query()
        torch.cuda._sleep(100_000_000)
        got = assembly.assembled(owner, "x", params, _build)
    with torch.cuda.stream(second):  # while `first` may still gather its forms
        again = assembly.assembled(owner, "x", params, _build)
        grads = torch.autograd.grad(again, params, up)
    torch.cuda.synchronize()
    for a, b, w in zip(got, again, want):
        assert torch.equal(a, w) and torch.equal(b, w)
    for g, r in zip(grads, ref):
        assert torch.allclose(g, torch.zeros_like(g) if r is None else r, rtol=0, atol=1e-6)


@pytest.mark.gpu
def test_forms_and_gradients_on_the_gpu(cuda):
    class Owner:
        pass

    owner = Owner()
    base = torch.empty(64, device=cuda)
    params = _params(cuda)
    params[2] = base[1:8].copy_(params[2])  # a view that starts off any alignment
    params = [p.requires_grad_(True) for p in params]
    got = assembly.assembled(owner, "x", params, _build)
    want = _build(params)
    for g, w in zip(got, want):
        assert torch.equal(g, w)
    up = [torch.randn_like(w) for w in want]
    grads = torch.autograd.grad(got, params, up)
    ref = torch.autograd.grad([w.double() for w in want], params, [u.double() for u in up], allow_unused=True)
    for g, r in zip(grads, ref):
        assert torch.allclose(g, torch.zeros_like(g) if r is None else r, rtol=0, atol=1e-6)
    few = assembly.assembled(owner, "x", [p.detach() for p in params], _build)
    assert not any(f.requires_grad for f in few)
    wider = [p.repeat(2, *([1] * (p.dim() - 1))) if i == 2 else p for i, p in enumerate(params)]
    again = assembly.assembled(owner, "x", wider, _build)  # other shapes under the same name: a plan of their own
    for g, w in zip(again, _build(wider)):
        assert torch.equal(g, w)


@pytest.mark.gpu
@pytest.mark.parametrize("field,heads,bias", [({0: 16, 1: 16, 2: 16}, 4, True), ({0: 6, 1: 4, 2: 2}, 2, False),
                                              ({0: 4, 1: 4}, 2, True)])
def test_layer_forms_equal_the_layers_own_constructions(field, heads, bias, cuda):
    from gm_attention_amd.nn import fused_factored, radial
    from gm_attention_amd.nn.attention import _heads_permutation, _stacked_matrix
    from gm_attention_amd.nn.linear import linear_parameters, matrix_and_bias

    torch.manual_seed(1)
    mhsa = SO2MHSA(SO2FieldType(field), heads, cutoff=0.3, bias=bias, batched=True, dtype=torch.float32, device=cuda)
    values = [h.value for h in mhsa.heads]
    layout = fused_factored.heads_layout(values, torch.float32)
    forms = _LayerForms(mhsa, values, layout, True)
    assert forms.served
    for form, lins in ((forms.query, [h.query for h in mhsa.heads]), (forms.key, [h.key for h in mhsa.heads])):
        want = _stacked_matrix(lins, mhsa.field_type_in, [linear_parameters(lin) for lin in lins])
        assert torch.equal(form[0], want[0])
        assert torch.equal(form[1], want[1]) if bias else form[1] is None
    m, *b = matrix_and_bias(mhsa.output_projection, linear_parameters(mhsa.output_projection))
    assert torch.equal(forms.projection[0], m.index_select(0, _heads_permutation(mhsa, m.device)))
    assert torch.equal(forms.projection[1], b[0]) if bias else forms.projection[1] is None
    for got, want in zip(forms.mixing, fused_factored.mixing_forms(values, layout,
                                                                   [k.readout_parameters() for k in values])):
        assert torch.equal(got, want)
    for got, want in zip(forms.trunk, radial.stacked_forms([radial.trunk_parameters(k) for k in values]), strict=True):
        assert torch.equal(got, want)
