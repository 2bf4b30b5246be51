"""Ids, masks and lengths in every element type the operators take, read by the kernels as they are: the same bits as the
call with int32 ids and an int32 mask."""
import ctypes

import numpy as np
import pytest
import torch

import oracle
import tome_amd
from tome_amd import _lib

pytestmark = pytest.mark.gpu

B, L, V = 5, 31, 4099


def _inputs(dev, H=None):
    g = torch.Generator(device=dev).manual_seed(3)
    if H is None:
        x = torch.randn((B, L, V), device=dev, generator=g) * 2
    else:
        x = torch.randn((B, L, H), device=dev, generator=g).to(torch.bfloat16)
    t = torch.randint(0, V, (B, L), device=dev, generator=g)
    t[0, 0], t[4, 30] = V, -1                                          # outside the vocabulary: NaN
    lens = torch.tensor([31, 0, 1, 17, 30], device=dev)
    mask = (torch.arange(L, device=dev)[None] < lens[:, None])
    return x, t, lens, mask


def _same(a, b):
    for u, v in zip(a, b):
        assert (u is None) == (v is None)
        if u is not None:
            assert u.shape == v.shape and torch.equal(u.view(torch.int32), v.view(torch.int32))


MASKS = {"bool": lambda m, ln: {"row_valid": m}, "uint8": lambda m, ln: {"row_valid": m.to(torch.uint8) * 3},
         "int32": lambda m, ln: {"row_valid": m.to(torch.int32)}, "int64": lambda m, ln: {"row_valid": m.long() * 7},
         "float": lambda m, ln: {"row_valid": m.float()}, "strided": lambda m, ln: {"row_valid": m.t().contiguous().t()},
         "cpu": lambda m, ln: {"row_valid": m.cpu()}, "len64": lambda m, ln: {"lengths": ln}, "len32": lambda m, ln: {"lengths": ln.int()},
         "len_list": lambda m, ln: {"lengths": ln.tolist()}, "len_cpu": lambda m, ln: {"lengths": ln.cpu()}}


@pytest.mark.parametrize("form", sorted(MASKS))
@pytest.mark.parametrize("idtype", [torch.int64, torch.int16, torch.int32])
def test_masks_and_ids_in_any_type(dev, form, idtype):
    """Row kernel, fused kernel (small, tiled, with the norm), pair pass: each against int32 ids and an int32 mask."""
    x, t, lens, mask = _inputs(dev)
    plain = {"row_valid": mask.to(torch.int32).contiguous()}
    kw = MASKS[form](mask, lens)
    want = tome_amd.token_logprobs(x, t.int(), 0.9, want_lse=True, want_entropy=True, want_argmax=True, **plain)
    _same(tome_amd.token_logprobs(x, t.to(idtype), 0.9, want_lse=True, want_entropy=True, want_argmax=True, **kw), want)
    m = mask.cpu().numpy()
    ok = m & ((t >= 0) & (t < V)).cpu().numpy()
    ref = oracle.logprob_rows(x.reshape(-1, V).cpu().numpy(), t.clamp(0, V - 1).reshape(-1).int().cpu().numpy(), 0.9).reshape(B, L)
    lp = want.lp.cpu().numpy()
    np.testing.assert_allclose(lp[ok], ref[ok], atol=1e-4, rtol=0)
    assert (lp[~m] == 0).all() and np.isnan(lp[m & ~ok]).all() and (want.argmax.cpu().numpy()[~m] == -1).all()
    h, _, _, _ = _inputs(dev, 256)
    w = (torch.randn((1000, 256), device=dev, generator=torch.Generator(device=dev).manual_seed(4)) * 0.1).to(torch.bfloat16)
    tf = t.clamp(-1, 1000)
    nw = torch.ones(256, dtype=torch.bfloat16, device=dev) + h[0, 0] * 0.1
    for norm in (None, nw):
        want = tome_amd.fused_lmhead_logprobs(h, w, tf.int(), 0.8, want_entropy=True, want_argmax=True, norm_weight=norm, **plain)
        _same(tome_amd.fused_lmhead_logprobs(h, w, tf.to(idtype), 0.8, want_entropy=True, want_argmax=True, norm_weight=norm, **kw), want)
    want = tome_amd.grpo_pair_logprobs(h, h * 1.5, w, tf.int(), 0.8, norm_weight=nw, **plain)
    _same(tome_amd.grpo_pair_logprobs(h, h * 1.5, w, tf.to(idtype), 0.8, norm_weight=nw, **kw), want)


@pytest.mark.parametrize("n,H,norm", [(1, 256, False), (60, 512, False), (100, 320, True), (300, 128, False), (40, 72, True), (16, 1024, True)])
def test_lmhead_on_a_list_of_rows(dev, n, H, norm):
    """tome_lmhead_logprob_sel with a row list (streaming, tiled and generic kernel): the bits of the call on the gathered
    rows, repeats and any order allowed; an entry that names no row scores NaN (argmax -1) and leaves the others alone."""
    lib = tome_amd.load_library()
    g = torch.Generator(device=dev).manual_seed(n + H)
    n_rows, Vs = 77, 1500
    h = torch.randn((n_rows, H), device=dev, generator=g).to(torch.bfloat16)
    w = (torch.randn((Vs, H), device=dev, generator=g) * 0.1).to(torch.bfloat16)
    nw = (torch.rand(H, device=dev, generator=g) + 0.5).to(torch.bfloat16) if norm else None
    idx = torch.randint(0, n_rows, (n,), device=dev, generator=g, dtype=torch.int32)
    t = torch.randint(0, Vs, (n,), device=dev, generator=g)
    want = tome_amd.fused_lmhead_logprobs(h[idx.long()], w, t, 0.9, want_lse=True, want_entropy=True, want_argmax=True, norm_weight=nw)
    for bad in ([], [0], [n - 1]):
        rows = idx.clone()
        for j, b in enumerate(bad):
            rows[b] = n_rows if j % 2 == 0 and b == 0 else -5
        out = [torch.full((n,), 9.0, device=dev) for _ in range(3)] + [torch.zeros(n, dtype=torch.int32, device=dev)]
        sel = _lib.TomeRowSel(targets=t.data_ptr(), target_bytes=8)
        ws_bytes = lib.tome_norm_lmhead_logprob_workspace(n, H, Vs)
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=dev)
        _lib.check(lib.tome_lmhead_logprob_sel(h.data_ptr(), rows.data_ptr(), n_rows, nw.data_ptr() if norm else None, 1e-6, w.data_ptr(), n,
                                               H, Vs, H, H, ctypes.addressof(sel), 0.9, *[o.data_ptr() for o in out], ws.data_ptr(), ws_bytes,
                                               torch.cuda.current_stream(dev).cuda_stream))
        ok = torch.ones(n, dtype=torch.bool, device=dev)
        ok[bad] = False
        for o, e in zip(out, want):
            assert torch.equal(o[ok], e[ok])
        for o in out[:3]:
            assert bool(torch.isnan(o[~ok]).all())
        assert bool((out[3][~ok] == -1).all())
