"""Gradient sets larger than the Infinity Cache: pass 1 reads the last 256 MiB
of them (512 MiB of a set of at least 640 MiB) with loads that allocate there,
and pass 2 starts with those chunks, then does the rest.  Each chunk must be
updated exactly once wherever the split falls.  The reference updates the same
tensors in pieces, one optimizer each, small enough that pass 1 reads all of a
piece the one way and pass 2 runs it in order."""

from __future__ import annotations

import importlib

import pytest
import torch

from oracle import oracle as O
from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
DEV = "cuda:0"
F32, F16 = torch.float32, torch.float16
PIECE = 1 << 25         # elements: 128 MiB of fp32 gradients


def _params(sizes, pdtype, gdtypes, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    params, grads = [], []
    for k, n in enumerate(sizes):
        params.append(torch.nn.Parameter(torch.empty(n, dtype=pdtype, device=DEV).normal_(0.0, 0.02, generator=gen)))
        grads.append(torch.empty(n, device=DEV).normal_(0.0, 1e-2, generator=gen).to(gdtypes[k % len(gdtypes)]))
    return params, grads


def _step(params, grads, **kw):
    opt = mg.AdamW(params, lr=1e-2, weight_decay=0.1, **kw)
    opt.set_grad_source(grads)
    opt.step()          # no clip call: nothing couples the tensors
    return opt


@pytest.mark.parametrize("sizes,dtype,gdtypes", [
    ((1000, 70_000_003, 12_345), F32, [F32]),            # the split falls inside one tensor
    ((40_000_000, 40_000_000, 1025, 7), F32, [F32]),     # on another tensor than the last
    ((67_108_865,), F32, [F32]),                         # one element more than fits
    ((90_000_001, 30_000_000, 30_000_001), torch.bfloat16, [torch.bfloat16]),
    ((100_000_001, 67_772_159, 3), F32, [F32]),          # 640 MiB less 4 bytes: the last with 256 MiB
    ((100_000_001, 67_772_159, 4), F32, [F32]),          # 640 MiB: 512 MiB from here on
    ((50_000_001, 60_000_001, 1023, 5), F32, [F32, F16]),    # two kernel classes, above 256 MiB
    ((20_000_001, 30_000_001, 1023, 5), F32, [F32, F16]),    # and below
], ids=["inside", "between", "one-over", "bf16", "below-long", "long", "mixed", "mixed-small"])
def test_every_chunk_is_updated_once(sizes, dtype, gdtypes):
    log(f"case: cached first {sizes} {dtype} {gdtypes}")
    whole, grads = _params(sizes, dtype, gdtypes, 3)
    before = [p.detach().clone() for p in whole]
    first = [g.clone() for g in grads]
    opt = _step(whole, grads, writeback_grads=gdtypes == [F32])
    for p, g, p0, g0 in zip(whole, grads, before, first):
        assert torch.equal(g, g0)       # nothing to unscale or clip, written back or not
        for at in range(0, p.numel(), PIECE):
            part = slice(at, at + PIECE)
            q = torch.nn.Parameter(p0[part].clone())
            want = _step([q], [g0[part].clone()]).state[q]
            assert torch.equal(p[part], q), at
            for key in want:
                got = opt.state[p][key]
                assert torch.equal(got if key == "step" else got[part], want[key]), (key, at)
    want = O.norm_from_sumsq(sum(O.sumsq(g.float().cpu().numpy()) for g in first))
    assert float(mg.clip_grad_norm_(whole, 1e9)) == want
