"""The work a user of tome_amd has it do, as cases that can be timed and compared.

``listed()`` names one case per use; ``draw(rng)`` gives more of the same ranges.  Sizes are the benchmark's
(vocabulary 151936, hidden sizes 1024 / 2560 / 4096, the GRPO shapes of bench.py) or generic.  ``prepare`` makes what a
program holds before the call (logits or hidden states a model has just produced, its weights, token ids, adapters as
they came over the wire), ``run`` is one pass through the package's public functions.

  score     token_logprobs: log-prob (and statistics) of one id per row of a logits matrix
  matrix    fused_log_softmax: the whole log-softmax matrix
  lmhead    fused_lmhead_logprobs: hidden states x lm_head -> log-probs, logits never formed
  pair      grpo_pair_logprobs: policy and reference pass of a GRPO step over a shared lm_head
  sample    sample_tokens: one decode step of a batch
  rollout   rollout_decode: a whole decode loop on a given model
  entry     RefLogprobServicer.process_ref_logprobs_batched on hidden states: the reference pass of a rollout batch
  update    WeightUpdateServicer.update_weights: a LoRA request merged into the policy's weights
"""
import math
from types import SimpleNamespace

import numpy as np
import torch

import tome_amd

V = 151936
DEV = "cuda:0"


def listed():
    return [
        # Smallest call: the judge's extraction sites, fp32 logits of a few sequences, one id each.
        {"name": "score_f32_8rows", "kind": "score", "dtype": "f32", "batch": 8, "seq": 1, "V": V, "T": 1.0, "mask": False,
         "entropy": False, "argmax": False},
        # The GRPO reference pass on logits: 8 groups x 512 columns, right-padded, lengths 64..512.
        {"name": "score_bf16_ref_chunk", "kind": "score", "dtype": "bf16", "batch": 8, "seq": 512, "V": V, "T": 1.0, "mask": True,
         "entropy": False, "argmax": False},
        # A vocabulary that is no multiple of a vector: rows start at odd elements.  Policy statistics of a small batch.
        {"name": "score_bf16_odd_vocab", "kind": "score", "dtype": "bf16", "batch": 3, "seq": 131, "V": 50257, "T": 0.7, "mask": False,
         "entropy": True, "argmax": True},
        # fused_log_softmax as the decode loops call it: a decode batch in fp32.
        {"name": "matrix_f32_64rows", "kind": "matrix", "dtype": "f32", "rows": 64, "V": V, "T": 1.0},
        # The same function on the logits of a prefill.
        {"name": "matrix_f32_1024rows", "kind": "matrix", "dtype": "f32", "rows": 1024, "V": V, "T": 1.0},
        # lm_head + log-softmax of a short chunk: a few completions of a few dozen tokens.
        {"name": "lmhead_200x2560", "kind": "lmhead", "n": 200, "H": 2560, "V": V, "T": 0.7, "valid": 1.0, "norm": False, "entropy": False},
        # ... of a full chunk, at the benchmark's shape.
        {"name": "lmhead_4096x1024", "kind": "lmhead", "n": 4096, "H": 1024, "V": V, "T": 1.0, "valid": 1.0, "norm": False, "entropy": False},
        # Largest: policy + reference pass over 16 x 1024 padded tokens, final norm included.
        {"name": "pair_16x1024x2560", "kind": "pair", "batch": 16, "seq": 1024, "H": 2560, "V": V, "T": 0.7, "norm": True},
        # One decode step: top-k 20 sampling of 64 sequences with their log-probs.
        {"name": "sample_f32_64rows", "kind": "sample", "dtype": "f32", "rows": 64, "V": V, "T": 0.8, "k": 20},
        # A decode loop: 4 prompts x 8 completions of up to 32 tokens.
        {"name": "rollout_32seqs", "kind": "rollout", "dtype": "f32", "prompts": 4, "G": 8, "tokens": 32, "V": V, "T": 0.8},
        # The servicer's reference pass on a rollout batch: 8 prompts x 8 completions, in chunks of 32 sequences.
        {"name": "entry_hidden_64seqs", "kind": "entry", "prompts": 8, "G": 8, "most_prompt": 200, "most_completion": 256, "H": 1024, "V": V,
         "T": 1.0, "norm": True},
        # One UpdateWeights request: every layer of a 28-layer model of hidden size 1024, rank 8.
        {"name": "update_28layers_r8", "kind": "update", "layers": 28, "hidden": 1024, "inter": 3072, "heads": 16, "kv_heads": 8,
         "head_dim": 128, "rank": 8, "split_qkv": False},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _vocab(rng):
    """The benchmark's vocabulary, or any size from 32000 up: three in four of those leave rows off 16-byte boundaries."""
    return V if rng.random() < 0.4 else rng.randrange(32000, 160000)


def draw(rng):
    kind = rng.choice(["score", "matrix", "lmhead", "pair", "sample", "rollout", "entry", "update"])
    temp = rng.choice([0.7, 0.8, 1.0, 1.0, 1.3])
    dtype = rng.choice(["f32", "bf16"])
    if kind == "score":
        rows = _log_int(rng, 1, 8192)
        batch = rng.choice([1, 3, 8, 16])
        mask = rows >= 64 and rng.random() < 0.5
        return {"kind": kind, "dtype": dtype, "batch": batch, "seq": max(1, rows // batch), "V": _vocab(rng), "T": temp, "mask": mask,
                "entropy": rng.random() < 0.4, "argmax": rng.random() < 0.4}
    if kind == "matrix":
        return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 1, 3000), "V": _vocab(rng), "T": temp}
    if kind == "lmhead":
        H = 64 * rng.randrange(12, 65)                                    # 768 .. 4096
        n = _log_int(rng, 8, 8192 * 2560 // H)
        return {"kind": kind, "n": n, "H": H, "V": _vocab(rng), "T": temp, "valid": rng.choice([1.0, 1.0, 0.6]), "norm": rng.random() < 0.3,
                "entropy": rng.random() < 0.3}
    if kind == "pair":
        H = 64 * rng.randrange(12, 65)
        batch = rng.choice([2, 4, 8, 16])
        seq = max(4, min(1024, _log_int(rng, 8, 1024)))
        while batch * seq * H > 15000 * 2560:
            seq //= 2
        return {"kind": kind, "batch": batch, "seq": seq, "H": H, "V": _vocab(rng), "T": temp, "norm": rng.random() < 0.5}
    if kind == "sample":
        return {"kind": kind, "dtype": dtype, "rows": _log_int(rng, 1, 1024), "V": _vocab(rng), "T": rng.choice([0.0, 0.7, 0.8, 1.0]),
                "k": rng.choice([5, 20, 20, 32])}
    if kind == "rollout":
        return {"kind": kind, "dtype": dtype, "prompts": rng.randrange(1, 9), "G": rng.choice([2, 4, 8, 16]), "tokens": _log_int(rng, 4, 64),
                "V": _vocab(rng), "T": rng.choice([0.0, 0.7, 0.8, 1.0])}
    if kind == "entry":
        return {"kind": kind, "prompts": rng.randrange(1, 9), "G": rng.choice([2, 4, 8]), "most_prompt": _log_int(rng, 16, 400),
                "most_completion": _log_int(rng, 16, 400), "H": 64 * rng.randrange(12, 41), "V": _vocab(rng), "T": temp,
                "norm": rng.random() < 0.5}
    hidden = 256 * rng.randrange(3, 11)                                   # 768 .. 2560
    return {"kind": "update", "layers": rng.randrange(2, 29), "hidden": hidden, "inter": 256 * rng.randrange(hidden // 128, 3 * hidden // 256 + 1),
            "heads": hidden // 64, "kv_heads": 8, "head_dim": 64, "rank": rng.choice([4, 8, 12, 16, 32, 64]), "split_qkv": rng.random() < 0.4}


# ---- inputs --------------------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed))
    return g


def _logits(g, rows, vocab, dtype):
    """Rows ~ N(0, 3^2) with one likely id each, as a language model's; the likely ids come back too."""
    x = torch.empty((rows, vocab), dtype=torch.float32 if dtype == "f32" else torch.bfloat16, device=DEV)
    for r in range(0, rows, 1024):
        x[r:r + 1024].normal_(0.0, 3.0, generator=g)
    spike = torch.randint(0, vocab, (rows,), device=DEV, generator=g)
    x[torch.arange(rows, device=DEV), spike] += 15.0
    return x, spike


def _targets(g, spike, vocab):
    """Half of the ids are the likely one, half are any."""
    other = torch.randint(0, vocab, spike.shape, device=DEV, generator=g)
    return torch.where(torch.rand(spike.shape, device=DEV, generator=g) < 0.5, spike, other)


def _normal(g, shape, std):
    return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0.0, std, generator=g)


def _lengths(rs, batch, seq):
    return rs.randint(max(1, seq // 8), seq + 1, batch)


def prepare(case, seed):
    rs = np.random.RandomState(seed % (1 << 31))
    g = _gen(seed)
    kind = case["kind"]
    s = SimpleNamespace(case=case)
    if kind == "score":
        x, spike = _logits(g, case["batch"] * case["seq"], case["V"], case["dtype"])
        s.logits = x.view(case["batch"], case["seq"], case["V"])
        s.targets = _targets(g, spike, case["V"]).view(case["batch"], case["seq"])
        s.lengths = torch.from_numpy(_lengths(rs, case["batch"], case["seq"])).to(DEV) if case["mask"] else None
    elif kind == "matrix":
        s.logits, _ = _logits(g, case["rows"], case["V"], case["dtype"])
    elif kind == "sample":
        s.logits, _ = _logits(g, case["rows"], case["V"], case["dtype"])
        s.uniforms = torch.rand(case["rows"], device=DEV, generator=g)
    elif kind == "lmhead":
        s.hidden = _normal(g, (case["n"], case["H"]), 1.0)
        s.weight = _normal(g, (case["V"], case["H"]), 0.02)
        s.norm = _normal(g, (case["H"],), 0.1) + 1.0 if case["norm"] else None
        s.targets = torch.randint(0, case["V"], (case["n"],), device=DEV, generator=g)
        s.valid = None if case["valid"] >= 1.0 else (torch.rand(case["n"], device=DEV, generator=g) < case["valid"]).to(torch.int32)
    elif kind == "pair":
        shape = (case["batch"], case["seq"], case["H"])
        s.policy = _normal(g, shape, 1.0)
        s.ref = s.policy + _normal(g, shape, 0.2)                         # what a LoRA step leaves in the final states
        s.weight = _normal(g, (case["V"], case["H"]), 0.02)
        s.norm = _normal(g, (case["H"],), 0.1) + 1.0 if case["norm"] else None
        s.targets = torch.randint(0, case["V"], shape[:2], device=DEV, generator=g)
        s.lengths = torch.from_numpy(_lengths(rs, case["batch"], case["seq"])).to(DEV)
    elif kind == "rollout":
        rows = case["prompts"] * case["G"]
        s.eos = 7
        s.last, _ = _logits(g, case["prompts"], case["V"], case["dtype"])
        s.steps = []
        for _ in range(8):                                                # a model's answers, one after the other
            x, _spike = _logits(g, rows, case["V"], case["dtype"])
            ends = torch.rand(rows, device=DEV, generator=g) < 0.05
            x[:, s.eos] += torch.where(ends, 30.0, 0.0).to(x.dtype)
            s.steps.append(x)
        s.uniforms = torch.rand((case["tokens"], rows), device=DEV, generator=g)
    elif kind == "entry":
        P, G = case["prompts"], case["G"]
        ls = np.random.RandomState(P * 1000 + case["most_completion"])       # the lengths are the case's, the ids the seed's
        p_len = ls.randint(max(1, case["most_prompt"] // 4), case["most_prompt"] + 1, P)
        c_len = ls.randint(max(1, case["most_completion"] // 8), case["most_completion"] + 1, (P, G))
        s.prompts = [tome_amd.Prompt(str(i), rs.randint(0, case["V"], n).tolist()) for i, n in enumerate(p_len)]
        s.completions = [[rs.randint(0, case["V"], n).tolist() for n in row] for row in c_len]
        most = int((p_len[:, None] + c_len).max())
        s.hidden = _normal(g, (32 * most * case["H"],), 1.0)
        s.weight = _normal(g, (case["V"], case["H"]), 0.02)
        s.norm = _normal(g, (case["H"],), 0.1) + 1.0 if case["norm"] else None

        def model(ids, cache=None):
            b, n = ids.shape
            return s.hidden[:b * n * case["H"]].view(b, n, case["H"]), cache

        s.servicer = tome_amd.RefLogprobServicer(model, device=DEV, lm_head_weight=s.weight, final_norm_weight=s.norm)
    elif kind == "update":
        _prepare_update(s, case, rs, g)
    else:
        raise ValueError(kind)
    return s


def _update_shapes(case):
    q, kv = case["heads"] * case["head_dim"], case["kv_heads"] * case["head_dim"]
    return {"qkv": (q + 2 * kv, case["hidden"]), "gate_up": (2 * case["inter"], case["hidden"]), "down": (case["hidden"], case["inter"])}, q, kv


def _prepare_update(s, case, rs, g):
    shapes, q, kv = _update_shapes(case)
    n = case["layers"]
    ref = {k: _normal(g, (n, *sh), 0.02) for k, sh in shapes.items()}
    s.policy = {k: torch.zeros_like(v) for k, v in ref.items()}

    def model(w):
        return SimpleNamespace(layers=[SimpleNamespace(
            self_attn=SimpleNamespace(num_heads=case["heads"], qkv_proj=SimpleNamespace(weight=w["qkv"][i])),
            mlp=SimpleNamespace(gate_up_proj=SimpleNamespace(weight=w["gate_up"][i]), down_proj=SimpleNamespace(weight=w["down"][i])))
            for i in range(n)])

    def raw(a):
        return torch.from_numpy(a.astype(np.float32)).to(torch.bfloat16).view(torch.int16).numpy().tobytes()

    params = {"mlp.gate_up_proj": shapes["gate_up"], "mlp.down_proj": shapes["down"]}
    if case["split_qkv"]:
        params.update({"self_attn.q_proj": (q, case["hidden"]), "self_attn.v_proj": (kv, case["hidden"])})
    else:
        params["self_attn.qkv_proj"] = shapes["qkv"]
    r = case["rank"]
    updates = [tome_amd.LayerUpdate(i, name, raw(rs.standard_normal((r, cols)) * 0.05), raw(rs.standard_normal((rows, r)) * 0.05),
                                    [r, cols], [rows, r], 2.0)
               for i in range(n) for name, (rows, cols) in params.items()]
    s.request = SimpleNamespace(updates=updates)
    s.servicer = tome_amd.WeightUpdateServicer(model(s.policy), model(ref), head_dim=case["head_dim"], num_kv_heads=case["kv_heads"])


# ---- one pass ------------------------------------------------------------------------------------------------------
def run(s):
    c = s.case
    kind = c["kind"]
    if kind == "score":
        out = tome_amd.token_logprobs(s.logits, s.targets, c["T"], s.lengths, want_entropy=c["entropy"], want_argmax=c["argmax"])
        return {k: v for k, v in out._asdict().items() if v is not None}
    if kind == "matrix":
        return tome_amd.fused_log_softmax(s.logits, c["T"])
    if kind == "sample":
        out = tome_amd.sample_tokens(s.logits, c["T"], c["k"], uniforms=s.uniforms)
        return {"token": out.token, "lp": out.lp, "argmax": out.argmax}
    if kind == "lmhead":
        out = tome_amd.fused_lmhead_logprobs(s.hidden, s.weight, s.targets, c["T"], row_valid=s.valid, want_entropy=c["entropy"],
                                             norm_weight=s.norm)
        return {k: v for k, v in out._asdict().items() if v is not None}
    if kind == "pair":
        return tome_amd.grpo_pair_logprobs(s.policy, s.ref, s.weight, s.targets, c["T"], s.lengths, norm_weight=s.norm)._asdict()
    if kind == "rollout":
        turn = iter(range(1 << 30))
        out = tome_amd.rollout_decode(lambda tokens: s.steps[next(turn) % len(s.steps)], s.last, c["G"], c["T"], c["tokens"], s.eos,
                                      uniform_source=lambda step, rows: s.uniforms[step])
        tokens = np.full((len(out), c["tokens"]), -1, dtype=np.int64)            # as a trainer pads them
        log_probs = np.zeros((len(out), c["tokens"]), dtype=np.float32)
        for i, o in enumerate(out):
            tokens[i, :len(o["tokens"])] = o["tokens"]
            log_probs[i, :len(o["tokens"])] = o["log_probs"]
        return {"tokens": tokens, "log_probs": log_probs}
    if kind == "entry":
        results = [tome_amd.PromptRollout(p.prompt_id, [tome_amd.Completion(tokens=t) for t in row])
                   for p, row in zip(s.prompts, s.completions)]
        s.servicer.process_ref_logprobs_batched(s.prompts, results, c["G"], c["T"])
        return np.array([v for r in results for comp in r.completions for v in comp.ref_log_probs], dtype=np.float32)
    if kind == "update":
        answer = s.servicer.update_weights(s.request)
        return {"success": answer.success, **s.policy}
    raise ValueError(kind)


# ---- what a pass cannot do without ---------------------------------------------------------------------------------
def work(case):
    kind = case["kind"]
    size = {"f32": 4, "bf16": 2}.get(case.get("dtype"), 2)
    if kind == "score":
        rows = case["batch"] * case["seq"] * (0.5625 if case["mask"] else 1.0)   # mean of the padded lengths
        return {"bytes": rows * (case["V"] * size + 16), "flops": rows * case["V"] * 4}
    if kind == "matrix":
        return {"bytes": 2 * case["rows"] * case["V"] * size, "flops": case["rows"] * case["V"] * 5}
    if kind == "sample":
        return {"bytes": case["rows"] * (case["V"] * size + 16), "flops": case["rows"] * case["V"] * 4}
    if kind == "lmhead":
        n = case["n"] * case["valid"]
        return {"bytes": 2 * case["H"] * (n + case["V"]) + 12 * n, "flops": 2 * n * case["H"] * case["V"]}
    if kind == "pair":
        n = case["batch"] * case["seq"] * 0.5625
        return {"bytes": 2 * case["H"] * (2 * n + case["V"]) + 20 * n, "flops": 4 * n * case["H"] * case["V"]}
    if kind == "rollout":
        rows = case["prompts"] * case["G"] * case["tokens"] * 0.9                # most sequences run to the end
        return {"bytes": rows * (case["V"] * size + 16), "flops": rows * case["V"] * 4}
    if kind == "entry":
        n = case["prompts"] * case["G"] * case["most_completion"] * 0.5625
        chunks = -(-case["prompts"] * case["G"] // 32)
        return {"bytes": 2 * case["H"] * (n + chunks * case["V"]) + 8 * n, "flops": 2 * n * case["H"] * case["V"]}
    shapes, q, kv = _update_shapes(case)
    elems = case["layers"] * sum(r * c for r, c in shapes.values())
    adapters = case["layers"] * case["rank"] * sum(r + c for r, c in shapes.values())
    return {"bytes": 4 * elems + 2 * adapters, "flops": 2 * case["rank"] * elems}


def tolerance(case):
    """About four times the distance from the same path with every sum in 64 bits (measured at the listed sizes)."""
    kind = case["kind"]
    if kind == "matrix":                                                  # fp32 5.3e-8; bf16 1.6e-3: the output's own rounding
        return {"rel": 2.5e-7} if case["dtype"] == "f32" else {"rel": 6e-3}
    if kind == "update":                                                  # a product next to a rounding boundary may flip: 1e-4 of
        return {"rel": 1e-4}                                              # the elements, one bf16 step each
    if kind == "pair":                                                    # k3 of nearly equal log-probs: 8e-5
        return {"rel": 3e-4}
    if kind in ("lmhead", "entry") and case["norm"]:                      # one bf16 step in a normalised state: 1e-5 of a short batch
        return {"rel": 4e-5}
    return {"rel": 1e-6}                                                  # 5e-8 .. 1.7e-7
