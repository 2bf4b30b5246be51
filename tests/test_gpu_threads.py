"""Calls from one of several Python threads: what waits for the GPU does so without holding up the others."""
import threading
import time

import pytest
import torch

import tome_amd
from tome_amd.logprob import sample_step

pytestmark = pytest.mark.gpu


def _calls(dev):
    g = torch.Generator(device=dev).manual_seed(1)
    x = torch.randn((2, 8, 2000), device=dev, generator=g)
    tg = torch.zeros((2, 8), dtype=torch.int64, device=dev)
    h = torch.randn((2, 8, 128), device=dev, generator=g).to(torch.bfloat16)
    w = torch.randn((2000, 128), device=dev, generator=g).to(torch.bfloat16)
    mask, u = torch.ones((2, 8), dtype=torch.bool), torch.rand(16)                       # in host memory
    active = torch.ones(16, dtype=torch.int32, device=dev)
    host = torch.empty((2, 16), dtype=torch.int32, pin_memory=True)
    return {
        "token_logprobs_lengths": lambda: tome_amd.token_logprobs(x, tg, 1.0, [8, 3]),
        "token_logprobs_mask": lambda: tome_amd.token_logprobs(x, tg, 1.0, row_valid=mask),
        "sample_tokens": lambda: tome_amd.sample_tokens(x, 1.0, uniforms=u),
        "sample_step": lambda: sample_step(x.view(16, -1), 1.0, 20, u, active, host, -1, 0),
        "lmhead": lambda: tome_amd.fused_lmhead_logprobs(h, w, tg, 1.0, [8, 3]),
        "grpo_pair": lambda: tome_amd.grpo_pair_logprobs(h, h, w, tg, 1.0, row_valid=mask),
    }


@pytest.mark.parametrize("name", ["token_logprobs_lengths", "token_logprobs_mask", "sample_tokens", "sample_step", "lmhead", "grpo_pair"])
def test_a_copy_that_waits_lets_other_threads_run(dev, name):
    """Lengths, masks and uniforms in host memory are copied in the call, behind the work already queued on the stream: a
    thread that ticks every millisecond keeps ticking while the call waits (the GIL's switch interval is 5 ms)."""
    call = _calls(dev)[name]
    call()
    a = torch.randn((8192, 8192), device=dev)
    b = torch.empty_like(a)
    torch.mm(a, a, out=b)
    torch.cuda.synchronize()
    ticks, stop = [], threading.Event()

    def tick():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    other = threading.Thread(target=tick)
    other.start()
    try:
        for _ in range(24):                                             # ~10 ms each
            torch.mm(a, a, out=b)
        t0 = time.perf_counter()
        call()
        t1 = time.perf_counter()
        torch.cuda.synchronize()
    finally:
        stop.set()
        other.join()
    inside = [t for t in ticks if t0 <= t <= t1]
    gaps = [y - x for x, y in zip([t0, *inside], [*inside, t1])]
    assert t1 - t0 > 0.06, "the call did not wait for the queued work: nothing was tested"
    assert max(gaps) < (t1 - t0) / 3
