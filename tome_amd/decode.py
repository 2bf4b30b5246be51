"""The policy-side extraction sites of Tome's decode loops, on the batched sampler.

``Rollout`` (mlx-impl/node.py:556-612) and ``Judge`` (node.py:325-374) both run, per generated
token, a full ``fused_log_softmax`` over the batch followed by a Python loop that samples every row
(``_sample_token``, node.py:894-907) and reads its log-prob back with ``float(...)`` - 2·B host round
trips per step.  Here a step is one ``sample_tokens`` call for the whole batch (finished rows are
masked and not read) whose tokens and log-probs land in host memory; the bookkeeping
around it follows the reference line by line, including the two loops' different treatment of EOS.

The model itself (KV cache, attention) is not part of this path: ``model_step(tokens)`` stands for
``self.model(current_tokens, cache=batched_cache)[0][:, 0, :]`` plus ``cache.advance(1)``.
"""
from __future__ import annotations

from typing import Callable, List, Optional

import numpy as np
import torch

from . import _lib
from .logprob import _check_temperature, _stream, sample_tokens

UniformSource = Callable[[int, int], torch.Tensor]


def _uniforms(source, step: int, rows: int, dev: torch.device, generator) -> Optional[torch.Tensor]:
    if source is None:
        return torch.rand(rows, dtype=torch.float32, device=dev, generator=generator)
    u = source(step, rows)
    return torch.as_tensor(u, dtype=torch.float32, device=dev).reshape(rows)


class _Loop:
    """A decode loop's state between its steps.

    On the GPU it stays there: the sampler takes finished rows out of ``active``, forms the next step's input ids and writes
    the step's tokens and log-probs straight into page-locked host memory, so that a step is the sampler's launches and one
    synchronisation (the mask, the ids and the copy back were four launches, a copy each way and their host work: 32 sequences
    x 32 steps 1.97 -> 1.25 ms).  Tensors elsewhere go through ``sample_tokens``, which refuses them."""

    def __init__(self, rows: int, dev: torch.device, stop: int, idle: int):
        self.rows, self.dev, self.stop, self.idle = rows, dev, int(stop), int(idle)
        self.on_gpu = dev.type == "cuda"
        self.mask = None                                                       # off the GPU; None = every row active
        if self.on_gpu:
            self.active = torch.ones(rows, dtype=torch.int32, device=dev)
            self.host = torch.empty((2, rows), dtype=torch.int32, pin_memory=True)
            self.host_np = self.host.numpy()

    def step(self, logits: torch.Tensor, temperature: float, top_k: int, uniforms, active: Optional[np.ndarray] = None):
        """Sample every active row; returns the host (token, lp) arrays after ONE synchronisation and sets ``self.next``.

        ``active`` is the host copy of the mask (None = the loop's first draw: every row, and nothing stops one).  The
        sampler answers -1 for a row it was asked to draw from that holds no logit above -inf (a model that has diverged);
        such an id must not reach the next ``model_step`` as an embedding index, so it is an error here, naming the rows."""
        if temperature <= 0:
            uniforms = None
        if self.on_gpu:
            self.next = _lib.torch_ops().sample_step(logits, _check_temperature(temperature or 1.0), int(top_k), uniforms, self.active,
                                                     self.host, self.stop if active is not None else -1, self.idle, True, _stream(logits))
            torch.cuda.current_stream(self.dev).synchronize()
            host = self.host_np
        else:
            out = sample_tokens(logits, temperature, top_k, uniforms=uniforms, row_valid=self.mask)
            self.next = out.token.reshape(-1).to(torch.int64)
            host = torch.stack([out.token.reshape(-1), out.lp.reshape(-1).view(torch.int32)]).numpy()
        tok = host[0].astype(np.int64)
        bad = tok < 0 if active is None else (tok < 0) & active
        if bad.any():
            raise RuntimeError(f"decode step: no token could be drawn for rows {np.flatnonzero(bad).tolist()} "
                               "(no logit above -inf); the model's logits are degenerate")
        return tok, host[1].view(np.float32).copy()

    def finish(self, active: np.ndarray) -> None:
        """Rows have finished (on the GPU the sampler has seen that for itself)."""
        if not self.on_gpu:
            self.mask = torch.from_numpy(active.astype(np.int32))
            self.next = torch.where(self.mask != 0, self.next, torch.full_like(self.next, self.idle))


def _results(toks: np.ndarray, lps: np.ndarray, lens: np.ndarray) -> List[dict]:
    return [{"tokens": toks[i, :lens[i]].tolist(), "log_probs": [float(v) for v in lps[i, :lens[i]]]}
            for i in range(toks.shape[0])]


def rollout_decode(model_step: Callable[[torch.Tensor], torch.Tensor], last_logits: torch.Tensor, G: int,
                   temperature: float, max_tokens: int, eos_token_id: int, *, top_k: int = 20,
                   uniform_source: Optional[UniformSource] = None,
                   generator: Optional[torch.Generator] = None) -> List[dict]:
    """The sampling half of ``_rollout_batched`` (mlx-impl/node.py:556-612).

    ``last_logits`` [num_prompts, V]: the last prompt position's logits; every prompt gets ``G``
    independent first tokens from its row (node.py:556-571).  Then up to ``max_tokens - 1`` steps
    (node.py:578): ``model_step(tokens int64 [num_prompts * G]) -> logits [num_prompts * G, V]``; a
    finished sequence is fed ``eos_token_id`` (node.py:593-595) and is neither sampled nor read.
    A sequence finishes when it draws EOS - which is kept, with its log-prob (node.py:604-608) - or
    reaches ``max_tokens``.  Returns ``[{"tokens": [...], "log_probs": [...]}]`` in sequence order
    ``p_idx * G + g_idx`` (node.py:574).  ``uniform_source(step, rows)`` supplies the draws' uniforms
    (step 0 = first tokens); by default they come from ``torch.rand`` with ``generator``.

    Per generated token the host does one synchronisation and array bookkeeping; the next step's input ids and the mask of
    finished rows are formed on the device.
    """
    dev = last_logits.device
    total = last_logits.shape[0] * G
    first = last_logits.repeat_interleave(G, dim=0)                            # same row, G independent draws
    loop = _Loop(total, dev, eos_token_id, eos_token_id)                       # a finished row is fed EOS (node.py:593-595)
    tok, lp = loop.step(first, temperature, top_k, _uniforms(uniform_source, 0, total, dev, generator))
    width = max(int(max_tokens), 1)
    toks = np.zeros((total, width), dtype=np.int64)
    lps = np.zeros((total, width), dtype=np.float32)
    lens = np.ones(total, dtype=np.int64)
    toks[:, 0], lps[:, 0] = tok, lp                                            # node.py:574
    finished = np.zeros(total, dtype=bool)                                     # node.py:575: the first token is not checked
    for step in range(max_tokens - 1):                                         # node.py:578
        if finished.all():
            break
        logits = model_step(loop.next)
        tok, lp = loop.step(logits, temperature, top_k, _uniforms(uniform_source, step + 1, total, dev, generator), ~finished)
        act = ~finished
        rows = np.nonzero(act)[0]
        toks[rows, lens[rows]] = tok[rows]                                     # node.py:604-605
        lps[rows, lens[rows]] = lp[rows]
        lens[rows] += 1
        newly = act & ((tok == eos_token_id) | (lens >= max_tokens))           # node.py:607-608
        if newly.any():
            finished |= newly
            loop.finish(~finished)
    return _results(toks, lps, lens)


def judge_decode(model_step: Callable[[torch.Tensor], torch.Tensor], first_logits: torch.Tensor,
                 temperature: float, max_tokens: int, eos_token_id: int, *, top_k: int = 20,
                 uniform_source: Optional[UniformSource] = None,
                 generator: Optional[torch.Generator] = None) -> List[dict]:
    """The sampling half of a ``Judge`` chunk (mlx-impl/node.py:325-374).

    ``first_logits`` [B, V]; the first token of every item is always kept (node.py:334-342).
    In the loop (node.py:346-374) an item that draws EOS becomes inactive and the EOS token is NOT
    recorded (node.py:369-370) - unlike ``rollout_decode`` - and inactive items are fed token 0
    (node.py:350).  Returns ``[{"tokens": [...], "log_probs": [...]}]`` per item.
    """
    dev = first_logits.device
    B = first_logits.shape[0]
    # an inactive item is fed token 0 (node.py:350); without an EOS token (None) nothing ends one
    loop = _Loop(B, dev, -1 if eos_token_id is None else eos_token_id, 0)
    tok, lp = loop.step(first_logits, temperature, top_k, _uniforms(uniform_source, 0, B, dev, generator))
    width = max(int(max_tokens), 1)
    toks = np.zeros((B, width), dtype=np.int64)
    lps = np.zeros((B, width), dtype=np.float32)
    lens = np.ones(B, dtype=np.int64)
    toks[:, 0], lps[:, 0] = tok, lp
    active = np.ones(B, dtype=bool)                                            # node.py:344
    for step in range(max_tokens - 1):                                         # node.py:346
        if not active.any():
            break
        logits = model_step(loop.next)
        tok, lp = loop.step(logits, temperature, top_k, _uniforms(uniform_source, step + 1, B, dev, generator), active)
        ended = active & (tok == loop.stop)                                    # node.py:369-370: EOS is not recorded
        rows = np.nonzero(active & ~ended)[0]
        toks[rows, lens[rows]] = tok[rows]                                     # node.py:371-373
        lps[rows, lens[rows]] = lp[rows]
        lens[rows] += 1
        if ended.any():
            active &= ~ended
            loop.finish(active)
    return _results(toks, lps, lens)
