"""Pass 2's split of each chunk-table entry over work-groups: every chunk size
must give the same bits, whether its parts are 256 elements, longer (sizes that
are no power of two of 256, or above 65,536) or end beyond a tensor's last
element."""

from __future__ import annotations

import importlib

import pytest
import torch

from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"
SHAPES = [(1,), (255,), (256,), (257,), (1023,), (1025,), (4, 1024), (3, 1536), (70_001,), (2, 65536), (300_007,)]


def _run(dtype, chunk):
    gen = torch.Generator(device=DEV).manual_seed(4)
    params = []
    for k, shape in enumerate(SHAPES):
        n = torch.Size(shape).numel()
        at = k % 3                       # every third tensor aligned, the others one or two elements off
        p = torch.nn.Parameter(torch.empty(n + at, dtype=dtype, device=DEV).normal_(0.0, 0.02, generator=gen)[at:].view(shape))
        p.grad = torch.empty(shape, dtype=dtype, device=DEV).normal_(0.0, 1e-2, generator=gen)
        params.append(p)
    opt = mg.AdamW(params, lr=1e-2, weight_decay=0.1, chunk_elems=chunk, state_layout="separate")
    for _ in range(2):
        mg.clip_grad_norm_(params, 1.0)
        opt.step()
    return params, [opt.state[p] for p in params]


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("chunk", [512, 1536, 2560, 65536, 131072, 1 << 20])
def test_chunk_sizes_agree(chunk, dtype, monkeypatch):
    monkeypatch.setenv("MGOPT_FOLD", "0")
    log(f"case: chunk {chunk} {dtype}")
    want_p, want_s = _run(dtype, 1024)
    got_p, got_s = _run(dtype, chunk)
    for a, b, sa, sb in zip(got_p, want_p, got_s, want_s):
        assert torch.equal(a, b)
        for key in sb:
            assert torch.equal(sa[key], sb[key]), key
