"""dK and dV of 16-bit masks at head size 64: 128 keys a workgroup, two of them on a CU, a ring of three row tiles."""
import math

import pytest
import torch

from tests import parity
from trident_amd.operation import Attention

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("kind", ["keys", "length", "dense"])
@pytest.mark.parametrize("S", [128, 129, 191, 256, 257, 512, 777])
def test_a_batch_does_not_depend_on_its_company(S, kind, dtype, device):
    """Two to thirteen row tiles, with and without tiles left out or of zeros only: every batch of a launch with several workgroups per
    CU gets bit for bit what it gets alone, and two heads match the oracle."""
    B, H, D = 32, 8, 64
    g = torch.Generator().manual_seed(S)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4)]
    # (from S / 2 on: with a handful of keys their probabilities and terms of dS are of order 1 in every row, and the sum of S such terms
    # carries S times half an ulp of the operand type each, which is within the bound by sum |terms| but not within the plain atol)
    lengths = torch.randint((S + 1) // 2, S + 1, (B,), generator=g)
    hidden = torch.arange(S)[None, None, None, :] >= lengths[:, None, None, None]
    mask = {"keys": hidden, "length": hidden.expand(B, 1, S, S), "dense": hidden}[kind]
    mask = torch.zeros(mask.shape).masked_fill(mask, -math.inf) if kind != "dense" else 0.5 * torch.randn(B, 1, S, S, generator=g)
    mask = mask.to(dtype)
    tq, tk, tv, tdo, tm = [x.to(device) for x in (q, k, v, d_o, mask)]
    scale = 1.0 / math.sqrt(D)

    def gradients(s):
        o, lse = Attention._forward(tq[s], tk[s], tv[s], tm[s], 0.0, False, scale, 0, 0)
        return (o, *Attention._backward(tdo[s], tq[s], tk[s], tv[s], o, lse, tm[s], scale, 0.0, False, 0, 0, False)[:3])

    whole = gradients(slice(None))
    for b in range(B):
        for a, c in zip(whole, gradients(slice(b, b + 1))):
            assert torch.equal(a[b:b + 1], c)
    for b in (0, B - 1):
        at = (slice(b, b + 1), slice(1, 2))
        kw = dict(mask=mask[b:b + 1].float(), dropout_p=0.0, is_causal=False, scale=scale, seed=0, offset=0)
        o = whole[0][at]
        _, dk, dv, _, _ = parity.oracle_backward(q[at], k[at], v[at], d_o[at], o=o, **kw)
        _, _, a_dk, a_dv = parity.oracle_abs_sums(q[at], k[at], v[at], d_o[at], o=o, **kw)
        parity.close(whole[2][at], dk, dtype, f"{kind} dK", a_dk)
        parity.close(whole[3][at], dv, dtype, f"{kind} dV", a_dv)
