"""mgopt_plan_set_grads and stream capture, through the C ABI: a captured call
sets the gradients of each replay, and calls outside the graph set their own,
in whatever order captures, replays and eager calls come.  Sets of one kernel
argument block (up to 480 tensors), of one tensor more and of several blocks."""

from __future__ import annotations

import ctypes

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log
from tests.test_gpu_c_abi import DEV, F32, NONE, TensorDesc, _lib, _ok, _stream

pytestmark = pytest.mark.gpu


class _Plan:
    """A plan over `sets[0]`'s shapes, without optimizer state."""

    def __init__(self, grads):
        self.lib, self.plan = _lib(), ctypes.c_void_p()
        descs = (TensorDesc * len(grads))()
        for d, g in zip(descs, grads):
            d.numel, d.grad_dtype, d.lowp_dtype = g.numel(), F32, NONE
        _ok(self.lib.mgopt_plan_create(descs, len(grads), 1, None, 1024, ctypes.byref(self.plan)), self.lib, "create")

    def norm(self, grads):
        out = torch.empty((), dtype=torch.float32, device=DEV)
        table = (ctypes.c_void_p * len(grads))(*[g.data_ptr() for g in grads])
        _ok(self.lib.mgopt_plan_set_grads(self.plan, table, _stream()), self.lib, "set_grads")
        _ok(self.lib.mgopt_grad_norm(self.plan, None, 1.0, out.data_ptr(), None, None, _stream()), self.lib, "norm")
        return out

    def close(self):
        torch.cuda.synchronize()
        self.lib.mgopt_plan_destroy(self.plan)


def _grads(n, seed, sigma):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return [torch.empty(1 + i % 37, device=DEV).normal_(0.0, sigma, generator=gen) for i in range(n)]


def _want(grads):
    return O.norm_from_sumsq(sum(O.sumsq(g.cpu().numpy()) for g in grads))


@pytest.mark.parametrize("n", [3, 480, 481, 1500])
def test_captured_and_eager_tables_stay_apart(n):
    a, b = _grads(n, 1, 1.0), _grads(n, 2, 3.0)
    want_a, want_b = _want(a), _want(b)
    assert want_a != want_b
    log(f"case: captured gradient table of {n}")
    plan = _Plan(a)
    try:
        assert float(plan.norm(a)) == want_a
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = plan.norm(b)
        assert float(plan.norm(b)) == want_b         # nothing has replayed: the table still held a
        assert float(plan.norm(a)) == want_a
        for _ in range(3):
            graph.replay()
            assert float(captured) == want_b
            assert float(plan.norm(a)) == want_a     # the replay left b in the table
        with torch.cuda.graph(graph := torch.cuda.CUDAGraph()):
            captured = plan.norm(a)                  # the pointers of the last eager call
        for _ in range(2):
            assert float(plan.norm(b)) == want_b
            graph.replay()
            assert float(captured) == want_a
    finally:
        plan.close()


@pytest.mark.parametrize("n", [480, 481, 1000])
def test_replaced_buffers_are_followed(n):
    """Outside a capture: new buffers each call, and the same ones twice."""
    log(f"case: replaced gradient buffers, {n} tensors")
    sets = [_grads(n, seed, 1.0 + seed) for seed in range(6)]     # more sets than pinned slots
    plan = _Plan(sets[0])
    try:
        got = [(plan.norm(g), plan.norm(g)) for g in sets + sets]
        for (x, y), g in zip(got, sets + sets):
            assert float(x) == float(y) == _want(g)
    finally:
        plan.close()
