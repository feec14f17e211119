"""Masked 16-bit problems up to head size 64, and whatever runs on the fp32 matrix instruction: the dQ pass computes delta on its
way (tri_attn_bwd_dq_delta)."""
import ctypes
import math

import pytest
import torch

from trident_amd import _lib, operation

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("split", [False, True])
@pytest.mark.parametrize("kind", ["fp32", "same type", "length", "keys", "causal"])
@pytest.mark.parametrize("dtype,B,H,S,D,p", [(torch.bfloat16, 2, 2, 256, 64, 0.0), (torch.float16, 2, 2, 128, 64, 0.25), (torch.bfloat16, 1, 2, 1344, 64, 0.0),
                                             (torch.bfloat16, 2, 2, 130, 32, 0.0), (torch.float16, 1, 3, 777, 16, 0.25), (torch.float16, 1, 1, 1, 64, 0.0),
                                             (torch.bfloat16, 1, 2, 2049, 32, 0.25), (torch.float32, 2, 2, 1, 16, 0.0),
                                             (torch.float32, 2, 2, 257, 64, 0.25), (torch.float32, 1, 2, 640, 128, 0.0), (torch.float32, 1, 3, 130, 32, 0.0)])
def test_delta_on_the_way(dtype, B, H, S, D, p, kind, split, device):
    """The whole backward against delta, dK/dV and dQ one by one: delta is the same fp32 products summed in another order, and what
    follows differs by what that moves before the rounding to 16 bits."""
    lib = _lib.lib()
    g = torch.Generator().manual_seed(S + D)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype).to(device) for _ in range(4)]
    mask = 0.5 * torch.randn(B, 1, 1 if kind == "keys" else S, S, generator=g)
    if kind == "length":
        mask = torch.zeros(B, 1, S, S)
        mask[..., (2 * S + 2) // 3:] = -math.inf
    mask = mask.to(dtype if kind == "same type" else torch.float32).to(device) if kind != "causal" else None
    padded = operation._PreparedMask(mask, q) if S % 64 and mask is not None and dtype != torch.float32 else None
    view = None if padded or mask is None else operation._expand_mask(mask, (B, H, S, S))
    o, lse = torch.empty_like(q), torch.empty(B, H, S, device=device)
    results = []
    for whole in (False, True):
        delta = torch.full_like(lse, float("nan"))
        dq, dk, dv = [torch.full_like(q, float("nan")) for _ in range(3)]
        args = operation._make_args(q, k, v, o, lse, view, p, mask is None, 1.0 / math.sqrt(D), 7, 0, d_o, dq, dk, dv, None, delta)
        if padded:
            padded.describe(args)
        elif mask is not None:
            classes = operation._mask_classes(mask, args)  # noqa: F841
        if not whole:
            _lib.check(lib.tri_attn_fwd(ctypes.byref(args)))
        workspace = operation._take_workspace(args, 3, q.device) if split else None  # noqa: F841
        if whole:
            _lib.check(lib.tri_attn_bwd_dq_delta(ctypes.byref(args)))  # (not refused)
            assert not torch.isnan(delta).any()
            delta.fill_(float("nan"))
            _lib.check(lib.tri_attn_bwd(ctypes.byref(args)))
        else:
            for entry in (lib.tri_attn_bwd_delta, lib.tri_attn_bwd_dkdv, lib.tri_attn_bwd_dq):
                _lib.check(entry(ctypes.byref(args)))
        results.append((delta, dq, dk, dv))
    (d0, *g0), (d1, *g1) = results
    terms = (o.float() * d_o.float()).abs().sum(-1)
    assert ((d0 - d1).abs() <= D * 2.0 ** -24 * 2 * terms).all()
    limit = 2.0 ** -7 if dtype != torch.float32 else 2.0 ** -15
    for a, b in zip(g0, g1):
        a, b = a.float(), b.float()
        assert not torch.isnan(b).any()
        assert (a - b).abs().max().item() <= limit * max(1.0, a.abs().max().item())


def test_rows_off_the_16_byte_boundaries_and_mask_gradients_keep_the_pre_pass(device):
    B, H, S, D = 1, 2, 128, 64
    q, k, v, d_o = [torch.randn(B, H, S, D, device=device, dtype=torch.bfloat16) for _ in range(4)]
    mask = torch.randn(B, H, S, S, device=device)
    lse, delta = torch.zeros(B, H, S, device=device), torch.zeros(B, H, S, device=device)
    dq, dk, dv = [torch.empty_like(q) for _ in range(3)]
    odd = torch.zeros(B, H, S, D + 4, device=device, dtype=torch.bfloat16)[..., :D]
    for o, dmask in ((odd, None), (torch.zeros_like(q), torch.empty_like(mask))):
        args = operation._make_args(q, k, v, o, lse, mask, 0.0, False, 0.125, 0, 0, d_o, dq, dk, dv, dmask, delta)
        assert _lib.lib().tri_attn_bwd_dq_delta(ctypes.byref(args)) == _lib.ENOFUSE
    q, k, v, d_o, dq, dk, dv = [x.float() for x in (q, k, v, d_o, dq, dk, dv)]
    odd = torch.zeros(B, H, S, D + 1, device=device)[..., :D]
    args = operation._make_args(q, k, v, odd, lse, None, 0.0, True, 0.125, 0, 0, d_o, dq, dk, dv, None, delta)
    assert _lib.lib().tri_attn_bwd_dq_delta(ctypes.byref(args)) == _lib.ENOFUSE
