"""Token-log-prob operators on torch (ROCm) tensors, backed by libtome_logprob.so.

The first two functions keep the reference's names, argument order and meaning:

* ``fused_log_softmax(logits, temperature=1.0)``     mlx-impl/model.py:77-89
* ``local_compute_logprobs(logits, ids, temp)``      mlx-impl/node.py:400-404

The others are the additive, fused forms of the same path: one scalar per row
instead of a [rows, V] matrix (``token_logprobs``), the lm_head matmul of
mlx-impl/model.py:538 folded in (``fused_lmhead_logprobs``), and the GRPO
policy + reference pair with k3 KL and entropy (``grpo_dual_logprobs``).

Launches are asynchronous on the current torch stream, like MLX's lazy graph
(forced by ``mx.eval`` at node.py:456); reading a result on the host synchronises.
"""
from __future__ import annotations

from typing import NamedTuple, Optional

import torch

from . import _lib


class TokenLogprobs(NamedTuple):
    lp: torch.Tensor                    # float32, log-prob of the target id
    lse: Optional[torch.Tensor]         # float32, logsumexp of x / temperature
    entropy: Optional[torch.Tensor]     # float32, entropy of softmax(x / temperature), nats
    argmax: Optional[torch.Tensor]      # int32, first maximum of the row


class SampledTokens(NamedTuple):
    token: torch.Tensor                 # int32, the drawn (or greedy) token id; -1 for masked rows
    lp: torch.Tensor                    # float32, its log-prob under the full softmax
    argmax: torch.Tensor                # int32, first maximum of the row
    topk_idx: Optional[torch.Tensor]    # int32 [..., top_k], candidates by descending logit
    topk_logit: Optional[torch.Tensor]  # float32 [..., top_k], their raw logits


class DualLogprobs(NamedTuple):
    lp: torch.Tensor        # policy log-prob of the target id
    ref_lp: torch.Tensor    # reference-model log-prob of the target id
    k3: torch.Tensor        # exp(ref_lp - lp) - (ref_lp - lp) - 1
    entropy: torch.Tensor   # entropy of the policy distribution


def _check_temperature(temperature: float) -> float:
    temperature = float(temperature)
    if not (temperature > 0.0) or temperature == float("inf"):
        # the reference maps 0 to 1.0 at its call sites (`temperature or 1.0`, node.py:451)
        raise ValueError(f"temperature must be finite and > 0, got {temperature}")
    return temperature


def _tensor(t, like: torch.Tensor, on_device: bool = True):
    """``t`` as a tensor (ids, masks and lengths may also be given as lists)."""
    if t is None or isinstance(t, torch.Tensor):
        return t
    return torch.as_tensor(t, device=like.device) if on_device else torch.as_tensor(t)


def _require_tensor(t, what: str) -> None:
    """For arguments that the native call also takes as None, with another meaning."""
    if not isinstance(t, torch.Tensor):
        raise TypeError(f"{what} must be a tensor, got {type(t).__name__}")


def _rows_view(x: torch.Tensor) -> torch.Tensor:
    """[..., V] -> [rows, V] with unit stride along V, copying only when no such view exists (as every operator does)."""
    return _lib.torch_ops().rows_view(x)


def _row_valid(lead_shape, n_rows: int, lengths, row_valid, dev) -> Optional[torch.Tensor]:
    """int32 row mask from either an explicit mask or per-sequence lengths over a [B, L] leading shape."""
    if lengths is not None and row_valid is not None:
        raise ValueError("pass lengths or row_valid, not both")
    if row_valid is not None:
        rv = row_valid if isinstance(row_valid, torch.Tensor) else torch.as_tensor(row_valid, device=dev)
        if rv.numel() != n_rows:
            raise ValueError(f"row_valid has {rv.numel()} entries, expected {n_rows}")
        return rv.reshape(-1).to(device=dev, dtype=torch.int32).contiguous()
    if lengths is None:
        return None
    if len(lead_shape) != 2:
        raise ValueError("lengths needs inputs shaped [batch, seq, ...]")
    B, L = lead_shape
    ln = lengths if isinstance(lengths, torch.Tensor) else torch.as_tensor(lengths)
    if ln.numel() != B:
        raise ValueError(f"lengths has {ln.numel()} entries, expected {B}")
    ln = ln.to(device=dev, dtype=torch.int64).reshape(B, 1)
    return (torch.arange(L, device=dev).reshape(1, L) < ln).to(torch.int32).reshape(-1).contiguous()


# A fraction of the cost of the Stream object; a torch built without a GPU runtime does not have it, and imports this package for
# the parts that need none.
_current_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def _stream(t: torch.Tensor) -> int:
    """Raw hipStream_t of torch's current stream on ``t``'s GPU (the launch stream of every call); 0 for a CPU tensor,
    which the operators refuse."""
    if not t.is_cuda:
        return 0
    return _current_raw_stream(t.get_device()) if _current_raw_stream else torch.cuda.current_stream(t.device).cuda_stream


def token_logprobs(logits: torch.Tensor, targets, temperature: float = 1.0, lengths=None, *,
                   row_valid=None, want_lse: bool = False, want_entropy: bool = False,
                   want_argmax: bool = False) -> TokenLogprobs:
    """Log-prob of ``targets`` under softmax(logits / temperature), one scalar per row.

    ``logits`` is [..., V] float32 or bfloat16; ``targets`` has the leading shape.
    Rows masked out by ``lengths`` (per sequence, for [B, L, V] inputs) or
    ``row_valid`` are not read; their outputs are 0 (argmax -1).  Outputs are float32
    with the leading shape.
    """
    return TokenLogprobs(*_lib.torch_ops().token_logprobs(
        logits, _tensor(targets, logits), _check_temperature(temperature), _tensor(lengths, logits, False),
        _tensor(row_valid, logits), want_lse, want_entropy, want_argmax, _stream(logits)))


def token_logprobs_rows(logits: torch.Tensor, row_index, targets, temperature: float = 1.0, *,
                        want_lse: bool = False, want_entropy: bool = False, want_argmax: bool = False) -> TokenLogprobs:
    """``token_logprobs`` for a list of rows, packed: entry i scores row ``row_index[i]`` of the flattened
    ``logits`` ([..., V] -> [rows, V]) against ``targets[i]``; every output has ``len(row_index)`` entries.

    This is the slicing of mlx-impl/node.py:449 (the completion rows of each sequence of a padded chunk) and
    local_compute_logprobs on the slices (node.py:400-404) for the whole chunk in one launch; rows that are not
    listed are neither read nor launched.  An index outside the matrix scores NaN (argmax -1).
    """
    return TokenLogprobs(*_lib.torch_ops().token_logprobs_rows(
        logits, _tensor(row_index, logits), _tensor(targets, logits), _check_temperature(temperature), want_lse, want_entropy,
        want_argmax, _stream(logits)))


def _draw(logits: torch.Tensor, temperature: float, uniforms, generator: Optional[torch.Generator]):
    """(temperature, uniforms) of a sampler call: greedy (no uniforms) at temperature 0, else one uniform per row."""
    if float(temperature) == 0.0:
        return 1.0, None
    temperature = _check_temperature(temperature)
    if uniforms is None:
        if not logits.is_cuda:
            raise RuntimeError("tome_amd operators run on a ROCm GPU only (there is no CPU fallback); "
                               f"got a tensor on {logits.device}")
        uniforms = torch.rand(logits.shape[:-1].numel(), dtype=torch.float32, device=logits.device, generator=generator)
    return temperature, uniforms


def sample_tokens(logits: torch.Tensor, temperature: float, top_k: int = 20, *, uniforms=None,
                  generator: Optional[torch.Generator] = None, row_valid=None, lengths=None,
                  want_topk: bool = False) -> SampledTokens:
    """One decode step for a batch of rows: ``_sample_token(logits, temperature, top_k)``
    (mlx-impl/node.py:894-907) for every row at once, with the log-prob of the chosen token that
    the decode loops look up afterwards (node.py:590,605) from the same pass.

    ``temperature == 0`` is greedy (node.py:896-897) and the log-prob then uses temperature 1.0, as
    ``temperature or 1.0`` does at node.py:590.  Otherwise the token is drawn from
    softmax(top-k logits / temperature) by inverse CDF at ``uniforms`` (float32 in [0, 1), one per
    row; drawn with ``torch.rand`` from ``generator`` when omitted) - candidates ordered by
    logit descending, equal logits by ascending id.  MLX's random stream is not reproduced.
    """
    temperature, uniforms = _draw(logits, temperature, uniforms, generator)
    mask = None
    if row_valid is not None or lengths is not None:
        lead = logits.shape[:-1]
        mask = _row_valid(lead, lead.numel(), lengths, row_valid, logits.device)
    return SampledTokens(*_lib.torch_ops().sample_tokens(
        logits, temperature, int(top_k), _tensor(uniforms, logits), mask, want_topk, _stream(logits)))


def sample_step(logits: torch.Tensor, temperature: float, top_k: int, uniforms, active: torch.Tensor, host: torch.Tensor,
                stop_token: int, idle_token: int) -> torch.Tensor:
    """``sample_tokens`` as a step of the decode loops (``tome_amd.decode``): the rows of ``active`` (int32, on the GPU) are
    sampled and leave it when they draw ``stop_token`` (negative: none does); tokens and log-probs go to ``host`` (int32
    [2, rows], page-locked); returns the next input ids, int64, ``idle_token`` for rows that are no longer active.
    ``temperature`` and ``uniforms`` as in ``sample_tokens``: 0 is greedy, uniforms are drawn when omitted."""
    temperature, uniforms = _draw(logits, temperature, uniforms, None)
    return _lib.torch_ops().sample_step(logits, temperature, int(top_k), _tensor(uniforms, logits), active, host, int(stop_token),
                                        int(idle_token), False, _stream(logits))


class DecodeStepGraph:
    """``sample_tokens`` for one fixed decode-batch shape, captured once as a HIP graph and replayed.

    A decode loop (mlx-impl/node.py:575-612) calls the sampler once per generated token with the
    same shapes; replaying a captured graph removes the per-call host work (argument checks, output
    allocation, two kernel launches).  ``logits`` and ``uniforms`` are the static input buffers: write
    the step's logits and fresh uniforms into them (``copy_``, ``uniform_``), call ``replay()``, read
    ``token`` / ``lp`` / ``argmax``.  The kernels allocate nothing and clear nothing with memsets,
    so every replay computes exactly what the eager call does.
    """

    def __init__(self, logits: torch.Tensor, temperature: float, top_k: int = 20, *, uniforms: Optional[torch.Tensor] = None):
        if not logits.is_cuda:
            raise RuntimeError("tome_amd operators run on a ROCm GPU only (there is no CPU fallback); "
                               f"got a tensor on {logits.device}")
        dev = logits.device
        self.logits = logits
        rows = logits.numel() // logits.shape[-1]
        self.uniforms = uniforms if uniforms is not None else torch.rand(rows, dtype=torch.float32, device=dev)
        self.temperature, self.top_k = float(temperature), int(top_k)
        self._stream = torch.cuda.Stream(device=dev)       # default priority
        self._graph = torch.cuda.CUDAGraph()
        self._stream.wait_stream(torch.cuda.current_stream(dev))
        with torch.cuda.stream(self._stream):
            sample_tokens(self.logits, self.temperature, self.top_k, uniforms=self.uniforms)   # warm-up outside capture
        self._stream.synchronize()
        with torch.cuda.graph(self._graph, stream=self._stream):
            out = sample_tokens(self.logits, self.temperature, self.top_k, uniforms=self.uniforms)
        self.token, self.lp, self.argmax = out.token, out.lp, out.argmax

    def replay(self) -> SampledTokens:
        self._graph.replay()
        return SampledTokens(self.token, self.lp, self.argmax, None, None)


def local_compute_logprobs(logits: torch.Tensor, ids: torch.Tensor, temp: float) -> torch.Tensor:
    """Drop-in for the closure at mlx-impl/node.py:400-404.

    ``logits`` [Lc, V] (bf16 or f32), ``ids`` [Lc] token ids, ``temp`` > 0.  Returns
    float32 [Lc]: ``logits[ids]/temp - logsumexp(logits/temp)`` computed in fp32 in one
    pass over the row.
    """
    return token_logprobs(logits, ids, temp).lp


def fused_log_softmax(logits: torch.Tensor, temperature: float = 1.0) -> torch.Tensor:
    """Drop-in for mlx-impl/model.py:77-89: full log-softmax with temperature, same shape and dtype."""
    return _lib.torch_ops().fused_log_softmax(logits, _check_temperature(temperature), _stream(logits))


def fused_lmhead_logprobs(hidden: torch.Tensor, weight: torch.Tensor, targets, temperature: float = 1.0,
                          lengths=None, *, row_valid=None, want_lse: bool = False,
                          want_entropy: bool = False, want_argmax: bool = False,
                          norm_weight: torch.Tensor | None = None, norm_eps: float = 1e-6) -> TokenLogprobs:
    """Log-probs of ``targets`` under softmax((hidden @ weight.T) / temperature) without the logits.

    ``hidden`` [..., H] bf16 (already through the final norm, mlx-impl/model.py:536),
    ``weight`` [V, H] bf16 (the tied embedding matrix, model.py:538).  bf16 products are
    accumulated in fp32; unlike the reference the logits are not rounded to bf16.
    ``want_argmax`` adds the greedy token id (first maximum, as ``int(mx.argmax(logits))`` at
    mlx-impl/node.py:897); logits closer than fp32 accumulation noise may swap.
    With ``norm_weight`` (bf16 [H]) ``hidden`` holds the PRE-norm states and the model's final
    RMSNorm (``mx.fast.rms_norm(x, weight, eps)``, model.py:336-343, :536) is applied to the valid
    rows first.
    """
    return TokenLogprobs(*_lib.torch_ops().lmhead_logprobs(
        hidden, weight, _tensor(targets, hidden), _check_temperature(temperature), _tensor(lengths, hidden, False),
        _tensor(row_valid, hidden), want_lse, want_entropy, want_argmax, norm_weight, float(norm_eps), None, _stream(hidden)))


def _lmhead_logprobs_rows(states: torch.Tensor, weight: torch.Tensor, rows: torch.Tensor, targets: torch.Tensor, temperature: float,
                          norm_weight: torch.Tensor | None, norm_eps: float) -> torch.Tensor:
    """Log-probs of ``targets`` for a packed list of rows (int32, on the device) of ``states`` [n, H], without gathering them where
    the kernels can address the rows in place: the gather's two launches and 2 * n * H * 2 bytes go (passes of 28 sequences at H = 1728
    327 -> 309 us, 6 at 832 194 -> 178, 64 at 1024 2713 -> 2692).  What they could not
    (rows that do not start on 16 bytes, H that only the 32-bit-addressed kernel takes) is gathered."""
    if states.is_contiguous() and states.data_ptr() % 16 == 0 and states.shape[1] % 64 == 0 and rows.numel():
        return _lib.torch_ops().lmhead_logprobs(states, weight, targets, _check_temperature(temperature), None, None, False, False, False,
                                                norm_weight, float(norm_eps), rows, _stream(states))[0]
    picked = states.index_select(0, rows.long())
    return fused_lmhead_logprobs(picked, weight, targets, temperature, norm_weight=norm_weight, norm_eps=norm_eps).lp


def grpo_dual_logprobs(hidden: torch.Tensor, w_policy: torch.Tensor, w_ref: torch.Tensor, targets,
                       temperature: float = 1.0, lengths=None, *, row_valid=None) -> DualLogprobs:
    """Policy and reference log-probs of ``targets`` plus k3 KL and policy entropy, per token.

    The two weight sets share ``hidden`` (in Tome the policy is the reference plus a merged
    LoRA delta, mlx-impl/node.py:102-164).  k3 and entropy have no counterpart in the
    reference node; they are defined by their closed forms.
    """
    _require_tensor(w_ref, "w_ref")
    return DualLogprobs(*_lib.torch_ops().grpo_pair(
        hidden, None, w_policy, w_ref, _tensor(targets, hidden), _check_temperature(temperature),
        _tensor(lengths, hidden, False), _tensor(row_valid, hidden), None, 0.0, _stream(hidden)))


def grpo_pair_logprobs(hidden_policy: torch.Tensor, hidden_ref: torch.Tensor, w_policy: torch.Tensor, targets,
                       temperature: float = 1.0, lengths=None, *, w_ref: torch.Tensor | None = None,
                       row_valid=None, norm_weight: torch.Tensor | None = None,
                       norm_eps: float = 1e-6) -> DualLogprobs:
    """``grpo_dual_logprobs`` for the reference's two-model layout: one hidden-state matrix per model.

    Tome's ``UpdateWeights`` merges LoRA deltas into attention and MLP weights only
    (mlx-impl/node.py:134-151), so policy and reference models differ in their final hidden
    states and share the final norm and the lm_head (mlx-impl/model.py:536-538): ``w_ref``
    defaults to ``w_policy``.  ``norm_weight`` as in ``fused_lmhead_logprobs``, applied to both.
    """
    _require_tensor(hidden_ref, "hidden_ref")
    return DualLogprobs(*_lib.torch_ops().grpo_pair(
        hidden_policy, hidden_ref, w_policy, w_ref, _tensor(targets, hidden_policy), _check_temperature(temperature),
        _tensor(lengths, hidden_policy, False), _tensor(row_valid, hidden_policy), norm_weight, float(norm_eps),
        _stream(hidden_policy)))
