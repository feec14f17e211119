"""Dropout decisions where every word of the generator's counter and key is in use: the kernels fold the head, the offset, the seed and
the row or key of a lane into constants of the first rounds, and share a block's sixteen decisions inside a quad of lanes."""
import pytest
import torch

import trident_amd as trident
from tests import parity

pytestmark = pytest.mark.gpu

SEED, OFFSET = 0x71E2D3C4B5A69788, 0x79ABCDEF


@pytest.mark.parametrize("dtype,S,D,causal,masked", [
    (torch.bfloat16, 256, 128, True, False),   # the phased kernels
    (torch.float16, 331, 128, True, False),    # ... and those beside a ragged end
    (torch.bfloat16, 256, 128, False, True),   # pairs of waves beside a dense mask
    (torch.float16, 256, 64, True, False),     # forward with its rounds between the MFMAs
    (torch.bfloat16, 203, 64, False, True),
    (torch.float16, 130, 32, False, False),
    (torch.bfloat16, 65, 16, True, False),
    (torch.float32, 97, 64, True, False),      # the fp32 matrix kernels
    (torch.float32, 64, 32, False, True),
    (torch.float32, 33, 128, False, False),
])
def test_dropout_with_every_counter_word(dtype, S, D, causal, masked, device):
    g = torch.Generator().manual_seed(S * 131 + D)
    B, H = 2, 5  # heads 0 .. 9
    q, k, v, d_o = (torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4))
    mask = torch.randn(B, 1, S, S, generator=g) if masked else None
    reference_limits = trident.config.reference_limits
    trident.config.reference_limits = False
    trident.config.dropout_seed = (SEED, OFFSET)
    try:
        tq, tk, tv = (t.to(device).requires_grad_() for t in (q, k, v))
        out = trident.function.scaled_dot_product_attention(tq, tk, tv, None if mask is None else mask.to(device), 0.3, causal)
        grads = torch.autograd.grad(out, (tq, tk, tv), d_o.to(device))
    finally:
        trident.config.dropout_seed = None
        trident.config.reference_limits = reference_limits
    kw = dict(mask=mask, dropout_p=0.3, is_causal=causal, seed=SEED, offset=OFFSET)
    parity.close(out, parity.oracle_forward(q, k, v, **kw)[0], dtype, "O")
    out = out.detach()
    dq, dk, dv, _, _ = parity.oracle_backward(q, k, v, d_o, o=out, **kw)
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q, k, v, d_o, o=out, **kw)
    for name, got, want, total in zip(("dQ", "dK", "dV"), grads, (dq, dk, dv), (a_dq, a_dk, a_dv)):
        parity.close(got, want, dtype, name, total)
