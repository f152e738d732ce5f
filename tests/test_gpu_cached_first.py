"""Gradient sets larger than the Infinity Cache: pass 1 reads the last 256 MiB
of them (512 MiB of a set of at least 640 MiB) with loads that allocate there,
and pass 2 starts with those chunks, then does the rest.  Each chunk must be
updated exactly once wherever the split falls."""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"


def _params(sizes, dtype, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    params = []
    for n in sizes:
        p = torch.nn.Parameter(torch.empty(n, dtype=dtype, device=DEV).normal_(0.0, 0.02, generator=gen))
        p.grad = torch.empty(n, dtype=dtype, device=DEV).normal_(0.0, 1e-2, generator=gen)
        params.append(p)
    return params


@pytest.mark.parametrize("sizes,dtype", [
    ((1000, 70_000_003, 12_345), torch.float32),            # the split falls inside one tensor
    ((40_000_000, 40_000_000, 1025, 7), torch.float32),     # on another tensor than the last
    ((67_108_865,), torch.float32),                         # one element more than fits
    ((90_000_001, 30_000_000, 30_000_001), torch.bfloat16),
    ((100_000_001, 67_772_159, 3), torch.float32),          # 640 MiB less 4 bytes: the last with 256 MiB
    ((100_000_001, 67_772_159, 4), torch.float32),          # 640 MiB: 512 MiB from here on
], ids=["inside", "between", "one-over", "bf16", "below-long", "long"])
def test_every_chunk_is_updated_once(sizes, dtype):
    log(f"case: cached first {sizes} {dtype}")
    whole, single = _params(sizes, dtype, 3), _params(sizes, dtype, 3)
    opts = [mg.AdamW(whole, lr=1e-2, weight_decay=0.1, writeback_grads=dtype == torch.float32)]
    opts += [mg.AdamW([p], lr=1e-2, weight_decay=0.1) for p in single]
    for opt in opts:
        opt.step()          # no clip call: nothing couples the tensors
    for a, b in zip(whole, single):
        assert torch.equal(a, b)
        assert torch.equal(a.grad, b.grad)
        sa, sb = opts[0].state[a], opts[1 + [id(p) for p in single].index(id(b))].state[b]
        for key in sb:
            assert torch.equal(sa[key], sb[key]), key
    want = O.norm_from_sumsq(sum(O.sumsq(p.grad.float().cpu().numpy()) for p in whole))
    assert float(mg.clip_grad_norm_(whole, 1e9)) == want
