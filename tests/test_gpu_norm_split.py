"""The split of pass 1 into chunks: norms of sets on both sides of each size
at which the chunk length changes, with whole and ragged last chunks, against
the oracle's compensated sum of squares.  The GPU's fp64 sums differ from it by
under n * 2**-53 relative, far inside half an fp32 unit, so the rounded norms
are equal."""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"
GROUPS, SHORTEST = 2048, 16384      # chunks a set is split into, shortest chunk


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sizes", [
    (2_097_153,),                                       # the smallest set with a finalize of its own
    (SHORTEST * (GROUPS - 1),),                         # the last with the shortest chunks, all whole
    (SHORTEST * GROUPS * 2 - SHORTEST * 2,),            # one chunk short of the next length
    (SHORTEST * GROUPS * 2 - 1,),                       # the next length, a ragged last chunk
    (3_000_000, 1, 8191, SHORTEST + 3, 2 * SHORTEST, 5),
], ids=lambda s: "+".join(map(str, s)))
def test_norm_is_the_oracles_for_every_chunk_length(sizes, dtype):
    gen = torch.Generator(device=DEV).manual_seed(sum(sizes))
    params = []
    for n in sizes:
        p = torch.nn.Parameter(torch.empty(n, dtype=dtype, device=DEV))
        p.grad = torch.empty(n, dtype=dtype, device=DEV).normal_(0.0, 1e-2, generator=gen)
        params.append(p)
    want = O.norm_from_sumsq(sum(O.sumsq(p.grad.float().cpu().numpy()) for p in params))
    log(f"case: norm of {sizes} {dtype}")
    got = mg.clip_grad_norm_(params, 1e9)
    assert float(got) == want, (sizes, dtype, float(got), want)
