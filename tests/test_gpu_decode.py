"""The decode loops' extraction sites (Rollout node.py:556-612, Judge node.py:325-374) on the batched sampler,
against the oracle's row-by-row restatement: token lists bit-exact, log-probs to 1e-4."""
import numpy as np
import pytest
import torch

import oracle
import tome_amd

pytestmark = pytest.mark.gpu
V = 3001


def _setup(dev, seed, B):
    rng = np.random.default_rng(seed)
    W = (rng.standard_normal((V, V)) * 2.5).astype(np.float32)        # next-token logits = row of the last token
    first = (rng.standard_normal((B, V)) * 2.5).astype(np.float32)
    Wt = torch.from_numpy(W).to(dev)
    return rng, W, first, (lambda toks: Wt[toks]), (lambda toks: W[np.asarray(toks)])


def _safe(run_oracle, rng, steps, rows, T, k, W, first, tries=50):
    """Uniforms for which no draw of the oracle run sits within 1e-4 of a CDF step (fp32 and fp64 sums may
    disagree there, and one different token changes the rest of the sequence)."""
    for _ in range(tries):
        us = rng.random((steps, rows)).astype(np.float32)
        seq = run_oracle(us)
        ok = True
        for b, s in enumerate(seq):
            rows_seen = [first[b * first.shape[0] // rows]] + [W[t] for t in s["tokens"][:-1]]
            for st, row in enumerate(rows_seen):
                _, val = oracle.top_k_rows(row[None].astype(np.float64), k)
                p = np.exp((val[0] - val[0, 0]) / T); cdf = np.cumsum(p) / p.sum()
                if np.abs(cdf - us[st, b]).min() < 1e-4:
                    ok = False
        if ok:
            return us, seq
    raise AssertionError("no safe uniforms found")


@pytest.mark.parametrize("T,G,eos", [(0.8, 3, 7), (1.0, 1, -1), (0.0, 2, 11)])
def test_rollout_decode_matches_oracle(dev, T, G, eos):
    rng, W, first, model_t, model_np = _setup(dev, 41, 4)
    max_tokens, k = 9, 20
    if eos >= 0:
        W[:, eos] += 4.0                                               # make EOS likely enough to end some sequences early
        model_t = (lambda Wt: (lambda toks: Wt[toks]))(torch.from_numpy(W).to(dev))
    run = lambda us: oracle.rollout_decode(model_np, first, G, T, max_tokens, eos, us, k)
    if T > 0:
        us, want = _safe(run, rng, max_tokens, 4 * G, T, k, W, first)
        src = lambda step, rows: torch.from_numpy(us[step])
    else:
        want, src = run(None), None
    got = tome_amd.rollout_decode(model_t, torch.from_numpy(first).to(dev), G, T, max_tokens, eos, top_k=k, uniform_source=src)
    assert [g["tokens"] for g in got] == [w["tokens"] for w in want]
    for g, w in zip(got, want):
        assert len(g["log_probs"]) == len(g["tokens"])
        np.testing.assert_allclose(g["log_probs"], w["log_probs"], atol=1e-4, rtol=0)
    if eos >= 0:
        assert any(g["tokens"][-1] == eos and len(g["tokens"]) < max_tokens for g in got)   # EOS kept (node.py:604-608)


@pytest.mark.parametrize("T,eos", [(0.9, 5), (0.0, 3)])
def test_judge_decode_matches_oracle(dev, T, eos):
    rng, W, first, _, model_np = _setup(dev, 43, 6)
    W[:, eos] += 4.0
    Wt = torch.from_numpy(W).to(dev)
    model_t = lambda toks: Wt[toks]
    max_tokens, k = 8, 20
    run = lambda us: oracle.judge_decode(model_np, first, T, max_tokens, eos, us, k)
    if T > 0:
        us, want = _safe(run, rng, max_tokens, 6, T, k, W, first)
        src = lambda step, rows: torch.from_numpy(us[step])
    else:
        want, src = run(None), None
    got = tome_amd.judge_decode(model_t, torch.from_numpy(first).to(dev), T, max_tokens, eos, top_k=k, uniform_source=src)
    assert [g["tokens"] for g in got] == [w["tokens"] for w in want]
    for g, w in zip(got, want):
        np.testing.assert_allclose(g["log_probs"], w["log_probs"], atol=1e-4, rtol=0)
    assert all(eos not in g["tokens"][1:] for g in got)                # EOS never recorded after the first token (node.py:369-370)


@pytest.mark.parametrize("rows,V_step", [(1, 5), (33, 3001), (16, 40000), (9, 50257)])
@pytest.mark.parametrize("stop", [-1, 2])
def test_sample_step_keeps_the_loop_state(dev, rows, V_step, stop):
    """tome_row_sample_step in every kernel form: tokens and log-probs (in page-locked memory) as sample_tokens gives them,
    rows leave the mask exactly when they draw the stop token, the next ids are the tokens or the idle one."""
    from tome_amd.logprob import sample_step
    g = torch.Generator(device=dev).manual_seed(rows + V_step)
    active = torch.ones(rows, dtype=torch.int32, device=dev)
    host = torch.empty((2, rows), dtype=torch.int32, pin_memory=True)
    for _ in range(4):
        x = torch.randn((rows, V_step), device=dev, generator=g)
        x[torch.rand(rows, device=dev, generator=g) < 0.4, 2] += 50.0
        u = torch.rand(rows, device=dev, generator=g)
        before = active.clone()
        want = tome_amd.sample_tokens(x, 0.9, 4, uniforms=u, row_valid=before)
        nxt = sample_step(x, 0.9, 4, u, active, host, stop, 77)
        torch.cuda.synchronize()
        tok = want.token.to(torch.int64)
        assert torch.equal(host[0], want.token.cpu()) and torch.equal(host[1].view(torch.float32), want.lp.cpu())
        left = (before != 0) & (tok != stop)
        assert torch.equal(active != 0, left)
        assert torch.equal(nxt, torch.where(left, tok, torch.full_like(tok, 77)))


def test_sample_step_checks_where_the_gpu_writes(dev):
    """`host` and `active` reach the kernel as addresses: memory the GPU must not write, strided tensors, other types and
    sizes are refused before anything is launched, each with a message of its own."""
    from tome_amd.logprob import sample_step
    rows = 4
    x = torch.zeros((rows, 300), device=dev)
    active = torch.ones(rows, dtype=torch.int32, device=dev)
    pinned = torch.empty((2, rows), dtype=torch.int32, pin_memory=True)
    step = lambda a, h: sample_step(x, 0.0, 4, None, a, h, -1, 0)
    with pytest.raises(ValueError, match="page-locked"):
        step(active, torch.empty((2, rows), dtype=torch.int32))
    with pytest.raises(ValueError, match="host must hold"):
        step(active, pinned[:1])
    with pytest.raises(ValueError, match="one row per sequence"):
        step(active[:2], pinned)
    with pytest.raises(ValueError, match="contiguous"):
        step(active, torch.empty((rows, 2), dtype=torch.int32, pin_memory=True).t())
    with pytest.raises(ValueError, match="contiguous"):
        step(torch.ones(2 * rows, dtype=torch.int32, device=dev)[::2], pinned)
    with pytest.raises(TypeError, match="int32"):
        step(active.long(), pinned)
    with pytest.raises(TypeError, match="int32"):
        step(active, torch.empty((2, rows), dtype=torch.float32, pin_memory=True))
    with pytest.raises(RuntimeError, match="CPU fallback"):
        step(active.cpu(), pinned)
    on_gpu = torch.empty((2, rows), dtype=torch.int32, device=dev)                # ... and what may be written still is
    assert torch.equal(step(active, on_gpu), step(active, pinned))
    torch.cuda.synchronize()
    assert torch.equal(on_gpu.cpu(), pinned)


def test_sample_step_draws_as_sample_tokens_does(dev):
    """Temperature 0 is greedy whatever the uniforms; without uniforms they are drawn, from torch's generator of the GPU."""
    from tome_amd.logprob import sample_step
    rows = 512
    x = torch.zeros((rows, 4), device=dev)                             # four equal logits: greedy is always id 0
    active = torch.ones(rows, dtype=torch.int32, device=dev)
    host = torch.empty((2, rows), dtype=torch.int32, pin_memory=True)
    assert not sample_step(x, 0.0, 4, torch.full((rows,), 0.9, device=dev), active, host, -1, 0).any()
    torch.manual_seed(11)
    want = tome_amd.sample_tokens(x, 1.0, 4).token
    torch.manual_seed(11)
    got = sample_step(x, 1.0, 4, None, active, host, -1, 0)
    torch.cuda.synchronize()
    assert torch.equal(got, want.long()) and torch.equal(host[0], want.cpu())
    assert len(got.unique()) == 4


@pytest.mark.parametrize("loop", ["rollout", "judge"])
@pytest.mark.parametrize("temperature", [0.0, 0.8])
def test_decode_loops_on_the_gpu_refuse_a_row_without_a_token(dev, loop, temperature):
    """An active row whose logits are all -inf at the second step: RuntimeError names it, and its -1 has not been fed to the
    model.  A finished row with such logits is not read."""
    B, V_small, eos = 3, 40, 9
    first = torch.zeros((B, V_small), device=dev)
    first[:, 4] = 50.0
    seen = []

    def model_step(tokens, bad, at):
        seen.append(tokens.tolist())
        out = torch.zeros((B, V_small), device=dev)
        out[:, 5] = 50.0
        if len(seen) == 1:
            out[2, eos] = 90.0                                         # row 2 ends at the first step
        if len(seen) == at:
            out[bad] = float("-inf")
        return out

    def run(bad, at):
        seen.clear()
        step = lambda tokens: model_step(tokens, bad, at)
        if loop == "rollout":
            return tome_amd.rollout_decode(step, first, 1, temperature, 5, eos)
        return tome_amd.judge_decode(step, first, temperature, 5, eos)

    with pytest.raises(RuntimeError, match=r"rows \[1\]"):
        run(1, 2)
    idle = eos if loop == "rollout" else 0
    assert seen == [[4, 4, 4], [5, 5, idle]]
    done = run(2, 2)                                                   # the row that has ended
    assert [d["tokens"] for d in done] == [[4, 5, 5, 5, 5]] * 2 + ([[4, eos]] if loop == "rollout" else [[4]])
