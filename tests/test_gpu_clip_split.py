"""clip_grad_norm_ over parameters no AdamW of the package owns: the in-place
scaling in work-groups of 1 KB, with ordinary accesses up to 96 MiB of gradients and
nontemporal ones above, 16-byte, 8-byte and single-element forms by alignment.
Expected: each gradient times the returned norm's coefficient in fp32, rounded
once to its dtype (what the kernel computes, so the comparison is exact)."""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"
F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16


def _grads(spec, seed):
    """Gradients (dtype, length, elements past a 512-byte boundary) as views of buffers of their own."""
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return [torch.empty(n + at, dtype=dt, device=DEV).normal_(0.0, 1e-2, generator=gen)[at:] for dt, n, at in spec]


@pytest.mark.parametrize("spec", [
    [(dt, n, 0) for dt in (F32, F16, BF16) for n in (1, 7, 8, 2047, 2048, 2049, 1024, 1025, 16385)],
    [(dt, 5000, at) for dt in (F32, F16, BF16) for at in (1, 2, 3, 4, 6, 8)],
    [(BF16, 0, 0), (BF16, 4097, 0), (BF16, 0, 0), (BF16, 3, 1)],
    [(BF16, (96 << 19) - 5, 0), (BF16, 5, 0)],          # 96 MiB: the largest with ordinary accesses
    [(BF16, (96 << 19) - 5, 0), (BF16, 6, 0)],          # two bytes more
    [(F32, 60_000_001, 0), (F16, 1_000_003, 4)],        # mixed, above every cache rule
], ids=["sizes", "offsets", "empty", "96MiB", "above-96MiB", "mixed-large"])
def test_scaled_in_place(spec):
    log(f"case: clip split {spec[:3]} of {len(spec)}")
    grads = _grads(spec, 9)
    params = [torch.nn.Parameter(torch.zeros_like(g)) for g in grads]
    for p, g in zip(params, grads):
        p.grad = g
    before = [g.clone() for g in grads]
    norm = mg.clip_grad_norm_(params, 0.25)
    sumsq = sum(O.sumsq(g.float().cpu().numpy()) for g in before if g.numel())
    assert float(norm) == O.norm_from_sumsq(sumsq)
    coef = torch.tensor(O.clip_coef(float(norm), 0.25), dtype=F32, device=DEV)
    assert float(coef) < 1.0
    for p, g in zip(params, before):
        assert torch.equal(p.grad, (g.float() * coef).to(g.dtype))
