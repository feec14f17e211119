"""Head size 64 in workgroups of four waves: fp32 masks with a ring of three (forward, dQ) or two tiles (dK/dV), two workgroups on a CU,
and the numbers of items from which launches without a mask take eight waves. Head size 128 in such workgroups."""
import math

import pytest
import torch

from tests import parity
from trident_amd.operation import Attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("p", [0.0, 0.2])
@pytest.mark.parametrize("kind", ["length", "dense"])
@pytest.mark.parametrize("S", [64, 65, 128, 129, 192, 256, 321, 512, 777])
def test_fp32_masks_do_not_depend_on_the_company(S, kind, p, device):
    """One to thirteen tiles, with and without tiles left out or of zeros only: every batch of a launch with several workgroups per CU gets
    what it gets alone (without dropout, whose decisions depend on the head's number), and two heads match the oracle."""
    B, H, D, dtype, seed = 24, 8, 64, torch.bfloat16, 77
    g = torch.Generator().manual_seed(S)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4)]
    if kind == "length":
        lengths = torch.randint((S + 1) // 2, S + 1, (B,), generator=g)
        hidden = torch.arange(S)[None, None, None, :] >= lengths[:, None, None, None]
        mask = torch.zeros(B, 1, S, S).masked_fill(hidden, -math.inf)
    else:
        mask = 0.5 * torch.randn(B, 1, S, S, generator=g)
    tq, tk, tv, tdo, tm = [x.to(device) for x in (q, k, v, d_o, mask)]
    scale = 1.0 / math.sqrt(D)

    def step(s):
        o, lse = Attention._forward(tq[s], tk[s], tv[s], tm[s], p, False, scale, seed, 0)
        return (o, *Attention._backward(tdo[s], tq[s], tk[s], tv[s], o, lse, tm[s], scale, p, False, seed, 0, False)[:3])

    whole = step(slice(None))
    if p == 0.0:
        for b in range(B):
            for a, c in zip(whole, step(slice(b, b + 1))):
                assert torch.equal(a[b:b + 1], c)
    at = slice(0, 1)  # (the first batch: its heads have the numbers they have alone)
    kw = dict(mask=mask[at], dropout_p=p, is_causal=False, scale=scale, seed=seed, offset=0)
    o = whole[0][at]
    o_ref, _ = parity.oracle_forward(q[at], k[at], v[at], **kw)
    dq, dk, dv, _, _ = parity.oracle_backward(q[at], k[at], v[at], d_o[at], o=o, **kw)
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q[at], k[at], v[at], d_o[at], o=o, **kw)
    parity.close(o, o_ref, dtype, "O")
    for name, got, want, total in zip(("dQ", "dK", "dV"), whole[1:], (dq, dk, dv), (a_dq, a_dk, a_dv)):
        parity.close(got[at], want, dtype, name, total)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads", [64, 65, 128, 129, 256, 257])
def test_four_and_eight_waves_agree(heads, causal, device):
    """512 rows, two items of 256 each: one workgroup of eight waves or two of four, by the number of heads."""
    S, D, dtype = 512, 64, torch.float16
    g = torch.Generator().manual_seed(heads)
    q, k, v, d_o = [torch.randn(1, heads, S, D, generator=g).to(dtype) for _ in range(4)]
    tq, tk, tv, tdo = [x.to(device) for x in (q, k, v, d_o)]
    scale = 1.0 / math.sqrt(D)
    o, lse = Attention._forward(tq, tk, tv, None, 0.0, causal, scale, 0, 0)
    grads = Attention._backward(tdo, tq, tk, tv, o, lse, None, scale, 0.0, causal, 0, 0, False)[:3]
    for h in (0, heads - 1):
        at = (slice(0, 1), slice(h, h + 1))
        kw = dict(mask=None, dropout_p=0.0, is_causal=causal, scale=scale, seed=0, offset=0)
        parity.close(o[at], parity.oracle_forward(q[at], k[at], v[at], **kw)[0], dtype, "O")
        ref = parity.oracle_backward(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[:3]
        sums = parity.oracle_abs_sums(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[1:]
        for name, got, want, total in zip(("dQ", "dK", "dV"), grads, ref, sums):
            parity.close(got[at], want, dtype, name, total)


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("causal,heads,S", [(False, 1025, 64), (False, 513, 130), (False, 1025, 128), (False, 257, 512), (True, 513, 65), (True, 513, 128),
                                            (True, 171, 321), (True, 129, 512), (True, 171, 384)])
def test_launches_of_several_rounds(causal, heads, S, p, device):
    """Just beyond the number of workgroups from which three of them share a CU, with a ring of three tiles: one to eight tiles, ragged ends,
    first and last heads against the oracle."""
    D, dtype, seed = 64, torch.bfloat16, 99
    g = torch.Generator().manual_seed(heads + S)
    q, k, v, d_o = [torch.randn(1, heads, S, D, generator=g).to(dtype) for _ in range(4)]
    tq, tk, tv, tdo = [x.to(device) for x in (q, k, v, d_o)]
    scale = 1.0 / math.sqrt(D)
    o, lse = Attention._forward(tq, tk, tv, None, p, causal, scale, seed, 0)
    grads = Attention._backward(tdo, tq, tk, tv, o, lse, None, scale, p, causal, seed, 0, False)[:3]
    assert all(x.isfinite().all() for x in (o, *grads))
    for h in [0] + ([heads - 1] if p == 0.0 else []):  # (decisions depend on the head's number: the oracle counts from 0)
        at = (slice(0, 1), slice(h, h + 1))
        kw = dict(mask=None, dropout_p=p, is_causal=causal, scale=scale, seed=seed, offset=0)
        parity.close(o[at], parity.oracle_forward(q[at], k[at], v[at], **kw)[0], dtype, "O")
        ref = parity.oracle_backward(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[:3]
        sums = parity.oracle_abs_sums(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[1:]
        for name, got, want, total in zip(("dQ", "dK", "dV"), grads, ref, sums):
            parity.close(got[at], want, dtype, name, total)


@pytest.mark.parametrize("p", [0.0, 0.1])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("heads,S", [(2, 16), (3, 64), (9, 65), (5, 128), (4, 129), (128, 256), (129, 256), (64, 257), (171, 384), (65, 511), (64, 512),
                                     (228, 320), (129, 512), (9, 1000), (84, 1016), (33, 1025), (103, 640), (23, 2048), (40, 1281), (129, 777),
                                     (52, 2049), (257, 512)])
def test_head_size_128_in_four_waves(heads, S, causal, p, device):
    """Around the numbers of heads and rows at which workgroups of four waves (two to a CU, a ring of two tiles) take over from eight: the first
    and last heads match the oracle."""
    D, dtype, seed = 128, torch.bfloat16, 31
    g = torch.Generator().manual_seed(heads + S)
    q, k, v, d_o = [torch.randn(1, heads, S, D, generator=g).to(dtype) for _ in range(4)]
    tq, tk, tv, tdo = [x.to(device) for x in (q, k, v, d_o)]
    scale = 1.0 / math.sqrt(D)
    o, lse = Attention._forward(tq, tk, tv, None, p, causal, scale, seed, 0)
    grads = Attention._backward(tdo, tq, tk, tv, o, lse, None, scale, p, causal, seed, 0, False)[:3]
    for h in [0] + ([heads - 1] if p == 0.0 else []):  # (decisions depend on the head's number: the oracle counts from 0)
        at = (slice(0, 1), slice(h, h + 1))
        kw = dict(mask=None, dropout_p=p, is_causal=causal, scale=scale, seed=seed, offset=0)
        parity.close(o[at], parity.oracle_forward(q[at], k[at], v[at], **kw)[0], dtype, "O")
        ref = parity.oracle_backward(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[:3]
        sums = parity.oracle_abs_sums(q[at], k[at], v[at], d_o[at], o=o[at], **kw)[1:]
        for name, got, want, total in zip(("dQ", "dK", "dV"), grads, ref, sums):
            parity.close(got[at], want, dtype, name, total)
