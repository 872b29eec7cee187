"""A layer's parameters in the forms its kernels read, in one launch each way.

The layers' kernels take block matrices, mixing matrices and stacked trunks
whose every entry is one parameter entry, possibly negated, or zero (the
reference concatenates and stacks them per head and block on every call,
nn/attention.py:653-669, nn/kernels.py:506-546).  :func:`assembled` runs such a
construction once on the parameters' positions in place of their values, keeps
where every entry comes from, and from then on fills every form with one
``gm_signed_gather_f32`` launch; the gradient is the transposed gather, each
parameter entry's uses added in a fixed order.  The numbers are the
construction's own, bit for bit (moves and sign changes only).

Parameters the kernel does not take -- CPU tensors, other types and subclasses,
parameters on several devices or another than the current one, or not
contiguous -- go through the construction itself, as do parameters without a
plan on a stream under capture or in a replica of a data-parallel step, and all
of them under functorch transforms, forward-mode derivatives, tracing and
compiling.
"""

from __future__ import annotations

import itertools
import weakref
from collections.abc import Callable, Sequence
from typing import Any

import torch
from torch import Tensor, nn
from torch.autograd import forward_ad

from gm_attention_amd import _native

MAX_SOURCES = 256  # tensors a launch reads
MAX_USES = 16  # uses of one parameter entry the gradient's padded table holds
_ALIGN = 64  # entries a form starts at a multiple of (256 bytes: whole cache lines)
_PLAIN = (Tensor, nn.Parameter)  # subclasses may hold their numbers elsewhere
_OFFSET = (1 << 39) - 1  # of a code: its entry's offset in the tensor
#: Plans by the module whose parameters they assemble, then by name, device and
#: shapes: beside the modules, so that these copy, pickle and list as if there
#: were none, and gone with them.
_PLANS: weakref.WeakKeyDictionary[Any, dict[tuple, Plan]] = weakref.WeakKeyDictionary()


def _starts(sizes: Sequence[int], align: int) -> list[int]:
    """Starts of consecutive ranges of ``sizes``, each rounded up to ``align``, then the total."""
    return list(itertools.accumulate((-(-n // align) * align for n in sizes), initial=0))


class Plan:
    """Where every entry of a construction's forms comes from, found on the
    parameters' device and complete on return."""

    def __init__(self, shapes: tuple[torch.Size, ...], build: Callable[[list[Tensor]], list[Tensor]],
                 device: torch.device) -> None:
        self.shapes = shapes
        sizes = [s.numel() for s in shapes]
        self.in_starts = _starts(sizes, 4)  # a gradient starts on 16 bytes
        at = torch.arange(1, self.in_starts[-1] + 1, dtype=torch.float64, device=device)
        with torch.no_grad():
            forms = build([at[a:a + n].view(s) for a, n, s in zip(self.in_starts, sizes, shapes)])
        self.form_shapes = [m.shape for m in forms]
        self.out_starts = _starts([m.numel() for m in forms], _ALIGN)
        flat = torch.zeros(self.out_starts[-1], dtype=torch.float64, device=device)
        for a, m in zip(self.out_starts, forms):
            flat[a:a + m.numel()] = m.reshape(-1)
        position = flat.abs().long() - 1  # -1: zero
        self.codes = torch.where(position < 0, -1, self._code(self.in_starts, position, flat < 0)).reshape(1, -1)
        counts = torch.bincount(position.clamp_min(-1) + 1, minlength=2)[1:]
        self.most = int(counts.max())  # uses of one parameter entry
        self.made_on = _native.stream_handle(device)
        self.back: Tensor | None = None
        self.back_made_on = 0
        _native.complete(device)

    @staticmethod
    def _code(starts: list[int], position: Tensor, negative: Tensor) -> Tensor:
        edges = torch.tensor(starts[:-1], dtype=torch.int64, device=position.device)
        tensor = torch.searchsorted(edges, position, right=True) - 1
        # an empty tensor shares its start with the next one: searchsorted takes the last of them, which holds it
        offset = position - edges[tensor.clamp_min(0)]
        return (tensor << 40) | (offset << 1) | negative.long()

    def gradient_codes(self) -> Tensor:
        """``(uses, parameter entries)``: entry p's j-th use among the forms' entries."""
        if self.back is None:
            with _native.LOCK:
                if self.back is None:
                    codes = self.codes[0]
                    used = torch.nonzero(codes >= 0).squeeze(1)
                    codes = codes[used]
                    starts = torch.tensor(self.in_starts, dtype=torch.int64, device=codes.device)
                    at, order = torch.sort(starts[codes >> 40] + ((codes >> 1) & _OFFSET), stable=True)
                    rank = torch.arange(at.numel(), device=at.device) - torch.searchsorted(at, at)
                    table = torch.full((max(self.most, 1), self.in_starts[-1]), -1, dtype=torch.int64,
                                       device=at.device)
                    table[rank, at] = self._code(self.out_starts, used[order], (codes[order] & 1) == 1)
                    _native.complete(table.device)
                    self.back_made_on = _native.stream_handle(table.device)
                    self.back = table
        return self.back


def _gather(tensors: Sequence[Tensor | None], codes: Tensor, made_on: int) -> Tensor:
    """``signed_gather`` on the current stream; a table made on another one outlives what this has queued."""
    if _native.stream_handle(codes.device) != made_on:
        codes.record_stream(torch.cuda.current_stream(codes.device))
    return _native.signed_gather(tensors, codes)


def _forms(plan: Plan, *params: Tensor | None) -> tuple:
    out = _gather(params, plan.codes, plan.made_on)
    return tuple(out[a:a + s.numel()].view(s) for a, s in zip(plan.out_starts, plan.form_shapes))


def _gradients(plan: Plan, *grads: Tensor | None) -> tuple:
    out = _gather(_held(grads), plan.gradient_codes(), plan.back_made_on)
    return tuple(out[a:a + s.numel()].view(s) for a, s in zip(plan.in_starts, plan.shapes))


class _Assemble(torch.autograd.Function):
    """The forms from the parameters; its gradient is :class:`_Transposed`, and that one's is this one."""

    @staticmethod
    def forward(ctx: Any, plan: Plan, *params: Tensor | None) -> tuple:
        ctx.plan = plan
        ctx.set_materialize_grads(False)
        return _forms(plan, *params)

    @staticmethod
    def backward(ctx: Any, *grads: Tensor | None) -> tuple:
        if all(g is None for g in grads):
            return (None,) * len(ctx.needs_input_grad)
        out = (_Transposed.apply if torch.is_grad_enabled() else _gradients)(ctx.plan, *grads)
        return (None, *(g if need else None for g, need in zip(out, ctx.needs_input_grad[1:])))


class _Transposed(torch.autograd.Function):
    @staticmethod
    def forward(ctx: Any, plan: Plan, *grads: Tensor | None) -> tuple:
        ctx.plan = plan
        ctx.set_materialize_grads(False)
        return _gradients(plan, *grads)

    @staticmethod
    def backward(ctx: Any, *grads: Tensor | None) -> tuple:
        if all(g is None for g in grads):
            return (None,) * len(ctx.needs_input_grad)
        out = (_Assemble.apply if torch.is_grad_enabled() else _forms)(ctx.plan, *_held(grads))
        return (None, *(g if need else None for g, need in zip(out, ctx.needs_input_grad[1:])))


def _held(tensors: Sequence[Tensor | None]) -> list[Tensor | None]:
    """The tensors as the kernel reads them."""
    return [None if t is None else t.to(torch.float32).resolve_neg().contiguous() for t in tensors]


def _transformed() -> bool:
    """Whether something follows torch's own operations here that an autograd
    function with a launch of its own in it would hide from it: a functorch
    transform, forward-mode derivatives, tracing or compiling."""
    return (torch._C._are_functorch_transforms_active() or forward_ad._current_level >= 0 or torch.jit.is_tracing()
            or torch.compiler.is_compiling())


def takes(params: Sequence[Tensor]) -> bool:
    """Whether :func:`assembled` fills the forms of ``params`` in one launch."""
    if not 0 < len(params) <= MAX_SOURCES:
        return False
    device = params[0].device
    if device.type != "cuda" or device.index != torch.cuda.current_device() or _transformed():
        return False
    for p in params:  # a loop of cheap tests: small layers have sixty parameters and half a millisecond
        if (p.dtype is not torch.float32 or p.get_device() != device.index or not p.is_contiguous() or p.is_neg()
                or type(p) not in _PLAIN):
            return False
    return True


def assembled(owner: Any, name: str, params: Sequence[Tensor], build: Callable[[list[Tensor]], list[Tensor]],
              taken: bool | None = None) -> list:
    """``build(params)``, a list of forms whose every entry is an entry of
    ``params``, negated or not, or zero.  The plan is kept for ``owner`` under
    ``name`` (which also names whatever else ``build`` depends on) and the
    parameters' device and shapes.  ``taken``: :func:`takes` of ``params`` where
    the caller has it."""
    if not (takes(params) if taken is None else taken):
        return build(list(params))
    key = (name, params[0].device, tuple(p.shape for p in params))
    plan = _PLANS.get(owner, {}).get(key)
    graded = torch.is_grad_enabled() and any(p.requires_grad for p in params)
    if (plan is None or (graded and plan.back is None)) and (
            torch.cuda.is_current_stream_capturing() or owner.__dict__.get("_is_replica")):
        # finding a plan waits on the host, which a captured stream cannot, and a replica of a
        # data-parallel step is gone after it: these take the construction
        return build(list(params))
    if plan is None:
        with _native.LOCK:
            plans = _PLANS.setdefault(owner, {})
            plan = plans.get(key)
            if plan is None:
                plan = plans[key] = Plan(key[2], build, key[1])
    if plan.most > MAX_USES:
        return build(list(params))
    if graded:
        plan.gradient_codes()  # found here: the backward runs on a thread and perhaps a stream of its own
    return list(_Assemble.apply(plan, *params))
