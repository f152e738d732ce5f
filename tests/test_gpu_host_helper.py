"""The host helper's launches of a stand-alone clip: what other Python threads
and callers see of them."""

from __future__ import annotations

import ctypes
import importlib
import threading
import time

import pytest
import torch

from tests._gpu_harness import log

pytestmark = pytest.mark.gpu

mg = importlib.import_module("minigpt-train-infra_amd")
N = importlib.import_module("minigpt-train-infra_amd._native")
DEV = "cuda:0"


def test_other_threads_run_while_an_entry_point_waits():
    """An upload of more than 480 gradients may wait for the GPU inside
    mgopt_plan_set_grads.  A sleep of 0.3 s stands for it (usleep's only
    argument is where the entry points take the plan)."""
    log("case: threads during clip_launch")
    usleep = ctypes.cast(ctypes.CDLL(None).usleep, ctypes.c_void_p).value
    ticks, stop = [], threading.Event()

    def count():
        while not stop.is_set():
            ticks.append(time.monotonic())
            time.sleep(0.005)

    thread = threading.Thread(target=count)
    thread.start()
    try:
        torch.empty((), device=DEV)
        start = time.monotonic()
        rc, norm, coef = N.host().clip_launch(usleep, usleep, 0, 300_000, b"", 1.0, 0, 0)
        end = time.monotonic()
    finally:
        stop.set()
        thread.join()
    assert rc == 0 and end - start >= 0.6
    assert sum(start < t < end for t in ticks) >= 20
