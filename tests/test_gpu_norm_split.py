"""The split of pass 1 into chunks: norms of sets on both sides of each size
at which the chunk length changes, with whole and ragged last chunks, and of
flat buffers of the same lengths, against the oracle's compensated sum of
squares.  The GPU adds at most 256 squares per thread of a chunk, 8 partials per
thread of the finalize and 14 terms in the tree behind each, so its fp64 sums
are off by under 320 * 2**-53 = 4e-14 relative, and the fp32 norms equal unless
one lies that close to a rounding boundary."""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log
from tests.test_zz_no_alloc import _lib, _noalloc_norm

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"
GROUPS, SHORTEST = 2048, 16384      # chunks a set is split into, shortest chunk


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("sizes", [
    (2_097_152,),                                       # the largest whose pass 1 finalizes
    (2_097_153,),                                       # the smallest set with a finalize of its own
    (SHORTEST * (GROUPS - 1),),                         # the last with the shortest chunks, all whole
    (SHORTEST * GROUPS * 2 - SHORTEST * 2,),            # one chunk short of the next length
    (SHORTEST * GROUPS * 2 - 1,),                       # the next length, a ragged last chunk
    (3_000_000, 1, 8191, SHORTEST + 3, 2 * SHORTEST, 5),
], ids=lambda s: "+".join(map(str, s)))
def test_norm_is_the_oracles_around_the_shorter_chunk_lengths(sizes, dtype):
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
    if len(sizes) == 1:
        assert _noalloc_norm(_lib(), params[0].grad, sizes[0], None, 1e9)[0] == want


@pytest.mark.parametrize("length,dtype", [(65536, torch.float16), (131072, torch.bfloat16)])
def test_the_longer_chunk_lengths(length, dtype):
    """The two longest, each from 2,048 chunks of that length on: one chunk
    fewer (the length before), and the first set with a ragged last one."""
    full = length * GROUPS - 1
    gen = torch.Generator(device=DEV).manual_seed(length)
    p = torch.nn.Parameter(torch.empty(full, dtype=dtype, device=DEV))
    g = torch.empty(full, dtype=dtype, device=DEV).normal_(0.0, 1e-2, generator=gen)
    for n in (full - length + 1, full):
        log(f"case: norm of {n} {dtype}")
        q = torch.nn.Parameter(p.detach()[:n])
        q.grad = g[:n]
        want = O.norm_from_sumsq(O.sumsq(g[:n].float().cpu().numpy()))
        assert float(mg.clip_grad_norm_([q], 1e9)) == want
        assert _noalloc_norm(_lib(), g, n, None, 1e9)[0] == want
