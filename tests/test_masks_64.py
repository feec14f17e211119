"""Masks at lengths that are multiples of 64 but not of 128 run the 16-bit kernels as they are, with classes, and learned masks of any
kind at lengths that are no multiple of 128 get their gradient from tri_attn_bwd_dmask."""
import ctypes
import math

import pytest
import torch

import trident_amd as trident
from tests import parity
from trident_amd import _lib, operation
from trident_amd.operation import Attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kind", ["dense", "length", "16 bit", "keys", "dense+dropout"])
@pytest.mark.parametrize("dtype,B,H,S,D", [(torch.bfloat16, 2, 3, 64, 64), (torch.float16, 1, 3, 192, 128), (torch.bfloat16, 2, 2, 320, 32),
                                           (torch.float16, 2, 2, 192, 16), (torch.bfloat16, 1, 2, 576, 64), (torch.bfloat16, 2, 1, 448, 128)])
def test_multiples_of_64(dtype, B, H, S, D, kind, device):
    g = torch.Generator().manual_seed(S + D)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4)]
    p, rng = (0.2, (31, 2)) if "dropout" in kind else (0.0, (0, 0))
    mask = 0.5 * torch.randn(1, H, S, S, generator=g) if kind == "16 bit" else torch.randn(B, 1, 1 if kind == "keys" else S, S, generator=g)
    if kind == "length":
        mask = torch.zeros(B, 1, S, S)
        mask[0, ..., S - 70 if S > 70 else 40:] = -math.inf
    mask = mask.to(dtype) if kind == "16 bit" else mask
    tq, tk, tv, tdo, tm = [x.to(device) for x in (q, k, v, d_o, mask)]
    assert operation._prepared_mask(tm, tq) is None
    o, lse = torch.empty_like(tq), torch.empty(B, H, S, device=device)
    args = operation._make_args(tq, tk, tv, o, lse, operation._expand_mask(tm, (B, H, S, S)), p, False, 0.125, 0, 0, tdo, o, o, o, None, lse)
    assert [_lib.lib().tri_attn_uses_matrix_cores(ctypes.byref(args), which) for which in (0, 1, 2)] == [1, 1, 1]
    assert operation._mask_classes(tm, args) is not None
    scale = 1.0 / math.sqrt(D)
    o, lse = Attention._forward(tq, tk, tv, tm, p, False, scale, *rng)
    dq, dk, dv, _ = Attention._backward(tdo, tq, tk, tv, o, lse, tm, scale, p, False, *rng, False)
    kw = dict(mask=mask.float(), dropout_p=p, is_causal=False, scale=scale, seed=rng[0], offset=rng[1])
    parity.close(o, parity.oracle_forward(q, k, v, **kw)[0], dtype, f"{kind} O")
    dq_r, dk_r, dv_r, _, _ = parity.oracle_backward(q, k, v, d_o, o=o, **kw)
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q, k, v, d_o, o=o, **kw)
    parity.close(dq, dq_r, dtype, f"{kind} dQ", a_dq)
    parity.close(dk, dk_r, dtype, f"{kind} dK", a_dk)
    parity.close(dv, dv_r, dtype, f"{kind} dV", a_dv)


@pytest.mark.parametrize("S", [128, 192])
def test_masks_of_fp32_calls_are_not_classified(S, device, monkeypatch):
    """No fp32 kernel looks at classes: a pass over the mask, and memory, for nothing. (The first call with a mask: nothing is cached.)"""
    q = torch.randn(1, 2, S, 64, device=device)
    mask = torch.randn(1, 1, S, S, device=device)
    for dtype, wanted in ((torch.float32, False), (torch.float16, True)):
        x = q.to(dtype)
        args = operation._make_args(x, x, x, x, torch.empty(1, 2, S, device=device), operation._expand_mask(mask, (1, 2, S, S)), 0.0, False, 0.125, 0, 0)
        assert (operation._mask_classes(mask, args) is not None) == wanted and bool(args.mask_classes) == wanted


@pytest.mark.parametrize("S,D", [(1, 64), (63, 32), (64, 64), (130, 128), (192, 16), (260, 64)])
@pytest.mark.parametrize("shape", ["BHSS", "1HSS", "SS"])
@pytest.mark.parametrize("small", [False, True])
def test_learned_masks_at_lengths_that_are_no_multiple_of_128(S, D, shape, small, device, monkeypatch):
    """B = 1, so that [1,H,S,S] is a mask of its own for every head; as a large call has it (padded) and as a small one."""
    monkeypatch.setattr(operation, "_PADS_FROM", 1 << 62 if small else 0)
    monkeypatch.setattr(trident.config, "reference_limits", False)
    B, H = (2, 2) if shape == "BHSS" else (1, 3)
    g = torch.Generator().manual_seed(S)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(torch.bfloat16) for _ in range(4)]
    mask = (0.5 * torch.randn({"BHSS": (B, H, S, S), "1HSS": (1, H, S, S), "SS": (S, S)}[shape], generator=g)).to(torch.bfloat16)
    tq, tk, tv, tm = [x.to(device).requires_grad_() for x in (q, k, v, mask)]
    out = trident.function.scaled_dot_product_attention(tq, tk, tv, tm)
    grads = torch.autograd.grad(out, (tq, tk, tv, tm), d_o.to(device))
    full = mask.float() if mask.dim() == 4 else mask.float()[None, None]
    dq, dk, dv, dm, _ = parity.oracle_backward(q, k, v, d_o, mask=full, want_dmask=True, o=out.detach())
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q, k, v, d_o, mask=full, o=out.detach())
    for name, got, want, terms in (("dQ", grads[0], dq, a_dq), ("dK", grads[1], dk, a_dk), ("dV", grads[2], dv, a_dv)):
        parity.close(got, want, torch.bfloat16, name, terms)
    parity.close(grads[3].reshape(full.shape), dm, torch.bfloat16, "dMask")


@pytest.mark.parametrize("path", ["C++", "Python"])
@pytest.mark.parametrize("moved", ["query", "key", "value", "grad"])
@pytest.mark.parametrize("S,D,from_,pitch", [(64, 64, 4, 72), (192, 128, 0, 129), (260, 32, 4, 40)])
def test_learned_full_masks_beside_rows_off_the_16_byte_boundaries(S, D, from_, pitch, moved, path, device, monkeypatch):
    """tri_attn_bwd_dmask does not take such rows: the dQ pass writes the gradient of a [B,H,S,S] mask, as at multiples of 128. (Memory
    freed before the backward holds NaN: a gradient that nobody writes shows.)"""
    monkeypatch.setattr(operation, "_PADS_FROM", 0)
    monkeypatch.setattr(trident.config, "reference_limits", False)
    B, H = 2, 2
    g = torch.Generator().manual_seed(S)
    given = {n: torch.randn(B, H, S, D, generator=g).to(torch.bfloat16) for n in ("query", "key", "value", "grad")}
    mask = (0.5 * torch.randn(B, H, S, S, generator=g)).to(torch.bfloat16)
    on_gpu = {n: x.to(device) for n, x in given.items()}
    on_gpu[moved] = torch.zeros(B, H, S, pitch, dtype=torch.bfloat16, device=device)[..., from_:from_ + D].copy_(given[moved])
    tq, tk, tv, tm = [x.requires_grad_() for x in (on_gpu["query"], on_gpu["key"], on_gpu["value"], mask.to(device))]
    call = trident.function.scaled_dot_product_attention if path == "C++" else \
        lambda q, k, v, m: operation.Attention.apply(q, k, v, m, 0.0, False, 1.0 / math.sqrt(D), False)
    out = call(tq, tk, tv, tm)
    assert (type(out.grad_fn).__name__ == "AttentionBackward") == (path == "Python")
    stale = [torch.full_like(mask, math.nan, device=device) for _ in range(8)]
    del stale
    grads = torch.autograd.grad(out, (tq, tk, tv, tm), on_gpu["grad"])
    q, k, v, d_o = given.values()
    dq, dk, dv, dm, _ = parity.oracle_backward(q, k, v, d_o, mask=mask.float(), want_dmask=True, o=out.detach())
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q, k, v, d_o, mask=mask.float(), o=out.detach())
    for name, got, want, terms in (("dQ", grads[0], dq, a_dq), ("dK", grads[1], dk, a_dk), ("dV", grads[2], dv, a_dv)):
        parity.close(got, want, torch.bfloat16, name, terms)
    parity.close(grads[3], dm, torch.bfloat16, "dMask")


@pytest.mark.parametrize("p", [0.0, 0.2])
@pytest.mark.parametrize("shape", ["1HSS", "11SS"])
@pytest.mark.parametrize("B,H,S,D,mask_dtype", [(40, 3, 70, 64, torch.bfloat16), (50, 2, 130, 128, torch.float32), (33, 4, 64, 32, torch.bfloat16),
                                                (64, 1, 33, 16, torch.float16), (9, 2, 257, 128, torch.bfloat16), (5, 1, 128, 64, torch.float32)])
def test_pairs_of_a_tile_dealt_to_several_workgroups(B, H, S, D, mask_dtype, shape, p, device):
    """Few tiles under many pairs: parts of unequal length and empty ones, with and without the workspace, against fp64. The sums
    are fp32 in both: apart by the rounding of `pairs` additions at most."""
    g = torch.Generator(device=device).manual_seed(S + D)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g, device=device).to(torch.bfloat16) for _ in range(4)]
    mask = (0.5 * torch.randn(1, H if shape == "1HSS" else 1, S, S, generator=g, device=device)).to(mask_dtype)
    scale, rng, full = 1.0 / math.sqrt(D), ((5, 2) if p else (0, 0)), (B, H, S, S)
    o, lse = Attention._forward(q, k, v, mask, p, False, scale, *rng)
    delta = (o.float() * d_o.float()).sum(-1)
    results = []
    for split in (True, False):
        dmask = torch.full(mask.shape, float("nan"), dtype=mask_dtype, device=device)
        args = operation._make_args(q, k, v, o, lse, mask.expand(full), p, False, scale, *rng, d_o, None, None, None, dmask.expand(full), delta)
        size = _lib.lib().tri_attn_workspace_size(ctypes.byref(args), 4)
        assert size > 0
        if split:
            workspace = torch.full((size,), 255, dtype=torch.uint8, device=device)
            args.workspace, args.workspace_size = workspace.data_ptr(), size
        _lib.check(_lib.lib().tri_attn_bwd_dmask(ctypes.byref(args)))
        results.append(dmask)
    s = q.double() @ k.double().transpose(-1, -2).contiguous() * scale + mask.double()
    dp = d_o.double() @ v.double().transpose(-1, -2).contiguous()
    if p:
        keep = torch.empty(B * H, S, S, dtype=torch.uint8, device=device)
        for bh in range(B * H):
            _lib.check(_lib.lib().tri_attn_dropout_mask(*rng, p, bh, 0, S, 0, S, keep[bh].data_ptr(), torch.cuda.current_stream().cuda_stream))
        dp *= keep.view(full) * (256 / (256 - round(p * 256)))
    ds = torch.exp2(s * math.log2(math.e) - lse.double()[..., None]) * (dp - delta.double()[..., None])
    want = ds.sum((0,) if shape == "1HSS" else (0, 1), keepdim=True).reshape(mask.shape)
    terms = ds.abs().sum((0,) if shape == "1HSS" else (0, 1), keepdim=True).reshape(mask.shape)
    half_ulp = {torch.float32: 0.0, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}[mask_dtype]
    for dmask in results:
        # (scores of D products and their exponentials in fp32: a few 2^-20 of every term)
        assert ((dmask.double() - want).abs() <= half_ulp * want.abs() * 1.01 + 2.0 ** -17 * terms + 1e-7).all()
