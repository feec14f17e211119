"""Boolean masks of keys, kept as bits in registers: tiles of visible keys only, of hidden ones only and mixed ones, against the oracle and
against the same mask as an additive matrix of zeros and -inf, which takes the kernels that read a mask's values."""
import math

import pytest
import torch

import trident_amd as trident
from tests import parity

pytestmark = pytest.mark.gpu


def _masks(B, S, g):
    """Batch 0: a length; 1: holes all over; 2: nothing in the first tile, then a length; others: every key, one key."""
    keys = torch.arange(S)
    visible = torch.ones(B, S, dtype=torch.bool)
    visible[0] = keys < max(1, (5 * S) // 8)
    visible[1] = torch.rand(S, generator=g) < 0.7
    visible[1, S // 2] = True
    visible[2] = (keys >= min(64, S - 1)) & (keys <= max(S - 3, min(64, S - 1)))
    visible[4] = keys == S - 1
    return visible


def _step(q, k, v, d_o, mask, p, device):
    tq, tk, tv = (x.to(device).requires_grad_() for x in (q, k, v))
    trident.config.dropout_seed = (5, 9) if p else None
    out = trident.function.scaled_dot_product_attention(tq, tk, tv, mask.to(device), p, False)
    return (out.detach(), *torch.autograd.grad(out, (tq, tk, tv), d_o.to(device)))


@pytest.fixture(autouse=True)
def _any_length():
    limits, trident.config.reference_limits = trident.config.reference_limits, False
    yield
    trident.config.reference_limits, trident.config.dropout_seed = limits, None


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("D", [16, 32, 64, 128])
@pytest.mark.parametrize("p", [0.0, 0.2])
@pytest.mark.parametrize("S", [1, 63, 64, 65, 128, 191, 256, 333, 512, 777])
def test_bits_against_the_oracle(S, p, D, dtype, device):
    B, H = 5, 2
    g = torch.Generator().manual_seed(S * 7 + D)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4)]
    visible = _masks(B, S, g) if S > 1 else torch.ones(B, S, dtype=torch.bool)
    got = _step(q, k, v, d_o, visible[:, None, None, :], p, device)
    additive = torch.zeros(B, 1, 1, S).masked_fill(~visible[:, None, None, :], -math.inf)
    kw = dict(mask=additive.expand(B, 1, S, S), dropout_p=p, is_causal=False, scale=1.0 / math.sqrt(D), seed=5 if p else 0, offset=9 if p else 0)
    parity.close(got[0], parity.oracle_forward(q, k, v, **kw)[0], dtype, "O")
    dq, dk, dv, _, _ = parity.oracle_backward(q, k, v, d_o, o=got[0], **kw)
    _, a_dq, a_dk, a_dv = parity.oracle_abs_sums(q, k, v, d_o, o=got[0], **kw)
    for name, a, want, total in zip(("dQ", "dK", "dV"), got[1:], (dq, dk, dv), (a_dq, a_dk, a_dv)):
        parity.close(a, want, dtype, name, total)
    hidden = ~visible[:, None, :, None].expand(B, H, S, D)
    assert (got[2].cpu()[hidden] == 0).all() and (got[3].cpu()[hidden] == 0).all()


@pytest.mark.parametrize("form", ["batch", "head", "one", "strided"])
@pytest.mark.parametrize("heads,S,D,p", [(2, 4096, 64, 0.0), (2, 4097, 64, 0.0), (40, 640, 64, 0.0), (40, 333, 128, 0.0), (3, 2048, 128, 0.0),
                                         (64, 200, 32, 0.0), (24, 512, 128, 0.0), (1, 40, 128, 0.2), (40, 333, 128, 0.2), (24, 512, 128, 0.2),
                                         (3, 2048, 128, 0.2), (30, 130, 128, 0.2)])
def test_bits_against_the_additive_mask(heads, S, D, p, form, device):
    """Forms of a mask of keys: per batch, per head, one for all, every other entry of a wider tensor; the last length of the bits and the
    first behind it; launches of many heads, three workgroups to a CU, and of few, split."""
    B, dtype = 5, torch.bfloat16
    g = torch.Generator().manual_seed(S + D)
    q, k, v, d_o = [torch.randn(B, heads, S, D, generator=g).to(dtype) for _ in range(4)]
    visible = _masks(B, S, g)[:4].repeat(2, 1)[:B]
    mask = {"batch": visible[:, None, None, :], "one": visible[0][None, None, None, :],
            "head": torch.stack([visible.roll(h, 0) for h in range(heads)], 1)[:, :, None, :],
            "strided": torch.stack([visible, ~visible], -1).flatten(1)[:, None, None, ::2]}[form]
    got = _step(q, k, v, d_o, mask, p, device)
    additive = torch.zeros(mask.shape).masked_fill(~mask, -math.inf).to(dtype).expand(mask.shape[0], mask.shape[1], S, S)
    want = _step(q, k, v, d_o, additive, p, device)
    for name, a, b in zip(("O", "dQ", "dK", "dV"), got, want):
        # both round P, dS and the result to bf16: the difference of two roundings of terms whose sum is of order 1
        error = (a.float() - b.float()).norm() / b.float().norm()
        assert error < 6e-3, (name, float(error))


@pytest.mark.parametrize("S", [128, 200])
@pytest.mark.parametrize("D", [64, 128])
def test_a_batch_without_a_visible_key(S, D, device):
    """Softmax over nothing is NaN: for that batch's output and query gradients; the others are as they are without it."""
    B, H, dtype = 3, 4, torch.float16
    g = torch.Generator().manual_seed(S)
    q, k, v, d_o = [torch.randn(B, H, S, D, generator=g).to(dtype) for _ in range(4)]
    visible = torch.rand(B, S, generator=g) < 0.8
    visible[:, 0] = True
    visible[1] = False
    got = _step(q, k, v, d_o, visible[:, None, None, :], 0.0, device)
    alone = _step(q[::2], k[::2], v[::2], d_o[::2], visible[::2, None, None, :], 0.0, device)
    assert got[0][1].isnan().all() and got[1][1].isnan().all()
    for a, b in zip(got, alone):
        assert torch.equal(a[::2], b)
