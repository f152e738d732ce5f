"""clip_grad_norm_ with torch.nn.utils.clip_grad_norm_'s signature and result.

Called by the reference's loop at train.py:486 on model.parameters().  When
those parameters are exactly the ones (with grads) of one of this package's
AdamW optimizers, the norm pass runs on the optimizer's plan and the clip
coefficient stays on the GPU for the AdamW pass to apply in registers: the
gradients are read once here and once in the step, never rewritten.  Any other
parameter list goes through a grads-only plan and is scaled in place, as
torch/nn/utils/clip_grad.py:120-182 does.
"""

from __future__ import annotations

import ctypes
import struct
import sys
import threading
import types
import warnings
import weakref
from typing import Iterable

import torch

from . import _native as N
from .adamw import _OWNER, engine_of

class _GradPlan:
    """A plan of gradients no engine owns, for the set of `key`.  Whoever holds
    it keeps it alive, so a call may use the plan it looked up whatever other
    threads remember meanwhile; its lock is held from a gradient table to the
    last launch that reads it."""

    __slots__ = ("handle", "lock")

    def __init__(self, key: bytes):
        self.handle, self.lock = None, threading.Lock()
        index, = struct.unpack_from("<q", key)
        sets = list(struct.iter_unpack("<qb", key[8:]))
        descs = (N.TensorDesc * len(sets))()
        for d, (numel, code) in zip(descs, sets):
            d.numel = numel
            d.group = 0
            d.grad_dtype = code
            d.lowp_dtype = N.NONE
        # a chunk-table entry per 4 KB of gradients, four work-groups of the in-place scaling (mgopt.hip,
        # scale_grads_kernel)
        chunk = 1024 if any(code == N.F32 for _, code in sets) else 2048
        plan = ctypes.c_void_p()
        with torch.cuda.device(index):
            N.check(N.lib().mgopt_plan_create(descs, len(sets), 1, None, chunk, ctypes.byref(plan)),
                    "mgopt_plan_create")
        self.handle = plan.value

    def __del__(self, _finalizing=sys.is_finalizing):
        # bound at class definition: at interpreter shutdown the process releases everything itself
        if self.handle is not None and not _finalizing():
            N.load_library().mgopt_plan_destroy(ctypes.c_void_p(self.handle))


#: plans of gradient sets no engine owns, by the set's key (the device index, then each gradient's length in 8 bytes
#: and dtype code in 1) and by stream: a plan holds the gradient table, the partials and the ticket counter of the call
#: in flight, so calls on two streams need one each.  A plan's tables take about 0.3 % of the gradients' bytes and
#: 120-250 bytes per tensor, outside torch's allocator.
_GRAD_PLANS: dict[bytes, dict[int, _GradPlan]] = {}
MAX_SETS = 17
MAX_STREAMS = 33       # per set: torch's pool of 32 and the default stream
#: the plans that captured calls use, by the set's key: a graph holds the addresses of a plan's device tables, so a plan
#: once captured is never given back, and calls outside a capture leave it to the replays (its gradient table is then
#: the graph's).  One per set, shared by all captures of it.
_CAPTURED_PLANS: dict[bytes, _GradPlan] = {}
_PLANS_LOCK = threading.Lock()   # changes of these two
_last_fast: tuple[tuple, weakref.ref] | None = None   # (id tuple, engine) of the last fused-path call


def _grad_table(grads: list[torch.Tensor]) -> tuple[bytes, bytes, int]:
    """What the host helper's clip_table returns, for gradients it leaves to
    Python: the checks here name what is wrong with them."""
    dev = grads[0].device
    if dev.type != "cuda":
        raise RuntimeError("clip_grad_norm_ runs on the GPU only; there is no CPU path")
    for g in grads:
        if g.device != dev:
            raise RuntimeError("clip_grad_norm_ needs all gradients on one GPU")
        if not g.is_contiguous():
            raise RuntimeError("clip_grad_norm_ needs contiguous gradients")
    key = struct.pack("<q", dev.index) + b"".join(struct.pack("<qb", g.numel(), N.dtype_code(g.dtype)) for g in grads)
    return key, struct.pack(f"<{len(grads)}Q", *(g.data_ptr() for g in grads)), dev.index


def _capturing(index: int) -> bool:
    """Whether torch's current stream on GPU `index` is capturing a graph."""
    if index == torch.cuda.current_device():
        return torch.cuda.is_current_stream_capturing()
    with torch.cuda.device(index):
        return torch.cuda.is_current_stream_capturing()


def _plan_for(key: bytes, index: int, stream: int) -> _GradPlan:
    if _capturing(index):
        return _captured_plan(key, stream)
    by_stream = _GRAD_PLANS.get(key)
    plan = by_stream.get(stream) if by_stream is not None else None
    return _new_plan(key, stream) if plan is None else plan


def _new_plan(key: bytes, stream: int) -> _GradPlan:
    """A new plan, remembered for calls on `stream`; the set's oldest plan, and
    the oldest set's plans, are given back above the limits."""
    plan, old = _GradPlan(key), []
    with _PLANS_LOCK:
        by_stream = _GRAD_PLANS.setdefault(key, {})
        old.append(by_stream.pop(stream, None))      # another thread's, made meanwhile
        by_stream[stream] = plan
        if len(by_stream) > MAX_STREAMS:
            old.append(by_stream.pop(next(iter(by_stream))))
        if len(_GRAD_PLANS) > MAX_SETS:
            old.append(_GRAD_PLANS.pop(next(iter(_GRAD_PLANS))))
    return plan                                      # `old` goes here, outside the lock: that waits for the GPU


def _captured_plan(key: bytes, stream: int) -> _GradPlan:
    with _PLANS_LOCK:
        plan = _CAPTURED_PLANS.get(key)
        if plan is None:
            by_stream = _GRAD_PLANS.get(key)
            if not by_stream:
                raise RuntimeError("run clip_grad_norm_ once on gradients of these lengths and dtypes outside graph "
                                   "capture before capturing it")
            # a capture has a stream of its own as a rule: the set's newest plan then
            plan = by_stream.pop(stream if stream in by_stream else next(reversed(by_stream)))
            _CAPTURED_PLANS[key] = plan
    return plan


def _norm_only(table: tuple[bytes, bytes, int], max_norm: float, error_if_nonfinite: bool) -> torch.Tensor:
    key, ptrs, index = table
    N.lib()
    stream = N.stream_handle(index)
    plan = _plan_for(key, index, stream)
    # torch checks finiteness (clip_grad.py:110-116) before it scales (:232)
    scale = 0 if error_if_nonfinite else N.entry_address("mgopt_scale_grads")
    with plan.lock:
        rc, norm, coef = N.host().clip_launch(N.entry_address("mgopt_plan_set_grads"),
                                              N.entry_address("mgopt_grad_norm"), scale, plan.handle, ptrs, max_norm,
                                              index, stream)
        N.check(rc, "clip_grad_norm_")
    if error_if_nonfinite:
        _check_finite(norm, error_if_nonfinite)
        grads = ctypes.cast(ctypes.c_char_p(ptrs), ctypes.POINTER(ctypes.c_void_p))
        with plan.lock:
            # once more: another thread's call may have used the plan while this one waited
            N.check(N.lib().mgopt_plan_set_grads(plan.handle, grads, stream), "mgopt_plan_set_grads")
            N.check(N.lib().mgopt_scale_grads(plan.handle, coef.data_ptr(), stream), "mgopt_scale_grads")
    return norm


# (no no_grad wrapper: nothing here records autograd history, the kernels
# write through raw pointers, and the decorator costs ~2.5 us per call)
def clip_grad_norm_(
    parameters: torch.Tensor | Iterable[torch.Tensor],
    max_norm: float,
    norm_type: float = 2.0,
    error_if_nonfinite: bool = False,
    foreach: bool | None = None,
) -> torch.Tensor:
    """Total L2 norm of the gradients (as one vector), clipping them to
    max_norm: coefficient min(1, max_norm / (norm + 1e-6)), applied with no
    host branch (clip_grad.py:185-233).  Returns the pre-clip norm as a 0-dim
    float32 tensor on the GPU.

    In a graph capture, a list that is not an optimizer's needs one call
    before it, on gradients of the same lengths and dtypes.  Graphs that clip
    such sets share one plan: their replays must not overlap, nor the first
    of them a call that began before the capture."""
    if float(norm_type) != 2.0:
        raise NotImplementedError("only norm_type=2.0 is implemented")
    if isinstance(parameters, torch.Tensor):
        parameters = [parameters]
    else:
        is_generator = isinstance(parameters, types.GeneratorType)
        parameters = list(parameters)
        if is_generator and len(parameters) == 0:
            warnings.warn("`parameters` is an empty generator, no gradient clipping will occur.", stacklevel=3)
    max_norm = float(max_norm)

    # Fast path: this exact parameter list was seen before and is the whole
    # parameter set of one optimizer (the train.py:486 call, every step).  The
    # last such list is remembered with its engine, which holds the
    # parameters (so their ids cannot be reused while it lives).
    global _last_fast
    key = tuple(map(id, parameters))
    if _last_fast is not None and _last_fast[0] == key and (eng := _last_fast[1]()) is not None:
        total = eng.norm(max_norm)
        _check_finite(total, error_if_nonfinite, eng)
        return total
    eng = engine_of(parameters[0]) if parameters else None
    if eng is not None and key in eng.complete_keys:
        _last_fast = (key, weakref.ref(eng))
        total = eng.norm(max_norm)
        _check_finite(total, error_if_nonfinite, eng)
        return total

    engines = {id(e): e for p in parameters if (e := engine_of(p)) is not None} if _OWNER else {}
    if len(engines) == 1:
        eng = next(iter(engines.values()))
        grads = eng.current_grads()
        mine = {id(p) for p, g in zip(eng.params, grads) if g is not None}
        given = {id(p) for p in parameters if engine_of(p) is eng}
        given_with_grad = {i for i in given if i in mine}
        if len(given) == len(parameters) and given_with_grad == mine:
            if not mine:
                return torch.tensor(0.0)
            if given == {id(p) for p in eng.params} and len(eng.complete_keys) < 8:
                eng.complete_keys.add(key)
            total = eng.norm(max_norm)
            _check_finite(total, error_if_nonfinite, eng)
            return total
    for e in engines.values():
        if e.scale_src is not None:
            raise RuntimeError(
                "clip_grad_norm_ on a parameter list that is not exactly an optimizer's parameters "
                "cannot follow GradScaler.unscale_ of that optimizer"
            )
    table = N.host().clip_table(parameters)
    if table is None:
        grads = [p.grad for p in parameters if p.grad is not None]
        if not grads:
            return torch.tensor(0.0)
        table = _grad_table(grads)
    return _norm_only(table, max_norm, error_if_nonfinite)


def _check_finite(total: torch.Tensor, error_if_nonfinite: bool, eng=None) -> None:
    if error_if_nonfinite and not bool(torch.isfinite(total)):
        if eng is not None:
            # torch raises before clipping, so a step taken anyway uses the
            # unclipped gradients: withdraw the pending coefficient
            eng.clip_pending = False
        raise RuntimeError(
            "The total norm of order 2.0 for gradients from `parameters` is non-finite, so it cannot be "
            "clipped. To disable this error and scale the gradients by the non-finite norm anyway, "
            "set `error_if_nonfinite=False`"
        )
