"""Launches split along the sequence (few heads, at least 20 tiles of 64, 4 in fp32) against whole ones and 64-bit results: the operator gives
its calls a workspace and so splits them, the same call without one does not."""
import ctypes
import math

import pytest
import torch

from trident_amd import _lib, operation

pytestmark = pytest.mark.gpu


def _exact(q, k, v, d_o, mask, keep, zscale, causal, scale):
    """O, dQ, dK, dV in 64 bits, head by head."""
    B, H, S, D = q.shape
    out = [torch.empty(B, H, S, D, dtype=torch.float64, device=q.device) for _ in range(4)]
    hidden = torch.ones(S, S, dtype=torch.bool, device=q.device).triu_(1) if causal else None
    for b in range(B):
        for h in range(H):
            qq, kk, vv, g = [x[b, h].double() for x in (q, k, v, d_o)]
            s = qq @ kk.t() * scale
            if mask is not None:
                s += mask.expand(B, H, S, S)[b, h].double()
            if causal:
                s.masked_fill_(hidden, -math.inf)
            p = s.softmax(1)
            z = keep[b * H + h] * zscale if keep is not None else None
            pz = p if z is None else p * z
            dp = g @ vv.t()
            dp = dp if z is None else dp * z
            out[0][b, h] = pz @ vv
            ds = p * (dp - (dp * p).sum(1, keepdim=True))
            out[1][b, h] = ds @ kk * scale
            out[2][b, h] = ds.t() @ qq * scale
            out[3][b, h] = pz.t() @ g
    return out


def _mask(kind, B, H, S, dtype, device):
    g = torch.Generator(device=device).manual_seed(S)
    lengths = torch.tensor([S - 70 * i - S // 3 * (i % 2) for i in range(B)], device=device)
    exists = torch.arange(S, device=device)[None, :] < lengths[:, None]
    if kind == "bool keys":
        return exists[:, None, None, :].contiguous()
    if kind == "length":
        return torch.zeros(B, 1, S, S, device=device).masked_fill_(~exists[:, None, None, :], -math.inf)
    if kind == "dense":
        return torch.randn(B, 1, S, S, generator=g, device=device)
    if kind == "16 bit":
        return torch.randn(1, H, S, S, generator=g, device=device).to(dtype)
    return None


def _run(q, k, v, d_o, mask, p, causal, scale, rng, split, monkeypatch):
    """O, lse, dQ, dK, dV and whether any launch was split."""
    used = []
    take = operation._take_workspace

    def spy(args, which, device):
        workspace = take(args, which, device) if split else None
        used.append(workspace is not None)
        return workspace

    with monkeypatch.context() as m:
        m.setattr(operation, "_take_workspace", spy)
        m.setattr(operation, "_PADS_FROM", 0)
        given = operation._BooleanMask(mask) if mask is not None and mask.dtype == torch.bool else mask
        o, lse = operation.Attention._forward(q, k, v, given, p, causal, scale, *rng)
        dq, dk, dv, _ = operation.Attention._backward(d_o, q, k, v, o, lse, given, scale, p, causal, *rng, False)
    return (o, lse, dq, dk, dv), used


VARIANTS = ["plain", "causal", "dropout", "causal+dropout", "bool keys", "length", "dense", "16 bit", "bool keys+dropout", "dense+dropout"]


@pytest.mark.parametrize("variant", VARIANTS)
@pytest.mark.parametrize("dtype,B,H,S,D", [
    (torch.bfloat16, 1, 2, 2048, 128), (torch.float16, 1, 3, 1281, 128), (torch.bfloat16, 2, 1, 2047, 128), (torch.float16, 1, 1, 4160, 128),
    (torch.bfloat16, 1, 3, 1345, 64), (torch.float16, 2, 1, 2176, 64), (torch.bfloat16, 1, 1, 5000, 64),
    (torch.float16, 1, 4, 1343, 32), (torch.bfloat16, 2, 1, 2304, 32), (torch.bfloat16, 1, 2, 1409, 16), (torch.float16, 1, 5, 1920, 16),
    (torch.float32, 1, 3, 1281, 128), (torch.float32, 2, 1, 513, 128), (torch.float32, 1, 4, 640, 64), (torch.float32, 1, 2, 420, 32),
    (torch.float32, 1, 4, 1000, 16)])
def test_split_launches(dtype, B, H, S, D, variant, device, monkeypatch):
    """As close to the 64-bit result as the whole launch: the parts' sums are fp32, what differs is which rounding of P to 16 bits
    goes with which row maximum (a few per cent of the error; 10 % allowed, and fp32 rounding on top of it)."""
    p, causal = (0.2 if "dropout" in variant else 0.0), "causal" in variant
    rng = (77, 3) if p else (0, 0)
    scale = 1.0 / math.sqrt(D)
    g = torch.Generator(device=device).manual_seed(S + D)
    q, k, v, d_o = [torch.randn(B, S, H, D, generator=g, device=device).to(dtype).transpose(1, 2) for _ in range(4)]
    mask = _mask(variant.split("+")[0], B, H, S, dtype, device)
    keep = None
    if p:
        keep = torch.empty(B * H, S, S, dtype=torch.uint8, device=device)
        for bh in range(B * H):
            _lib.check(_lib.lib().tri_attn_dropout_mask(*rng, p, bh, 0, S, 0, S, keep[bh].data_ptr(), torch.cuda.current_stream().cuda_stream))
    thr = round(p * 256)
    additive = mask if mask is None or mask.dtype != torch.bool else torch.zeros(mask.shape, device=device).masked_fill(~mask, -math.inf)
    exact = _exact(q, k, v, d_o, additive, keep, 256 / (256 - thr), causal, scale)
    whole, used = _run(q, k, v, d_o, mask, p, causal, scale, rng, False, monkeypatch)
    assert not any(used)
    split, used = _run(q, k, v, d_o, mask, p, causal, scale, rng, True, monkeypatch)
    assert all(used), "the call was not split"
    again, _ = _run(q, k, v, d_o, mask, p, causal, scale, rng, True, monkeypatch)
    for name, a, b, c in zip(("O", "lse", "dQ", "dK", "dV"), split, whole, again):
        assert torch.equal(a, c), f"{name} differs between two runs"
        if name == "lse":
            assert (a - b).abs().max() <= (1e-5 if dtype == torch.float32 else 2.0 ** -8 * 1.5), name  # (whole launches sum P as rounded, padded masks as it is)
    for name, a, b, e in zip(("O", "dQ", "dK", "dV"), (split[0], *split[2:]), (whole[0], *whole[2:]), exact):
        off, off_whole = [((x.double() - e).norm() / e.norm()).item() for x in (a, b)]
        assert off <= 1.1 * off_whole + (1e-8 if dtype == torch.float32 else 1e-6), (name, off, off_whole)
        half_ulp = e.abs().max() * {torch.bfloat16: 2.0 ** -9, torch.float16: 2.0 ** -12, torch.float32: 2.0 ** -25}[dtype]  # (the result's own rounding)
        assert (a.double() - e).abs().max() <= 2 * (b.double() - e).abs().max() + half_ulp + 1e-6, name


@pytest.mark.parametrize("S,D", [(2048, 64), (1300, 128), (1300, 32), (2176, 128)])
@pytest.mark.parametrize("where", ["first rows", "last rows", "middle", "one row"])
def test_rows_without_a_visible_key(S, D, where, device, monkeypatch):
    """NaN where the whole launch gives NaN, and only there."""
    dtype = torch.bfloat16
    g = torch.Generator(device=device).manual_seed(S)
    q, k, v, d_o = [torch.randn(2, 1, S, D, generator=g, device=device).to(dtype) for _ in range(4)]
    lost = {"first rows": slice(0, 448), "last rows": slice(S - 400, S), "middle": slice(512, 960), "one row": slice(700, 701)}[where]
    mask = torch.zeros(2, 1, S, S, device=device)
    mask[1, :, lost] = -math.inf
    mask[1, ..., S // 2:] = -math.inf
    whole, _ = _run(q, k, v, d_o, mask, 0.0, False, 0.125, (0, 0), False, monkeypatch)
    split, used = _run(q, k, v, d_o, mask, 0.0, False, 0.125, (0, 0), True, monkeypatch)
    assert all(used)
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), split, whole):
        assert torch.equal(a.isnan(), b.isnan()), name
        a, b = a.float().nan_to_num(0.0, neginf=-1e4), b.float().nan_to_num(0.0, neginf=-1e4)
        assert (a - b).norm() <= 2.0 ** -6 * b.norm(), name


def test_workspaces_that_do_not_do(device):
    """Too small, misaligned or absent (also by the size of the structure): the whole launch, bit for bit."""
    B, H, S, D = 1, 2, 1400, 64
    q, k, v = [torch.randn(B, H, S, D, device=device).half() for _ in range(3)]
    results = []
    for case in ("none", "small", "misaligned", "old structure"):
        o, lse = torch.empty_like(q), torch.empty(B, H, S, device=device)
        args = operation._make_args(q, k, v, o, lse, None, 0.0, True, 0.125, 0, 0)
        size = _lib.lib().tri_attn_workspace_size(ctypes.byref(args), 0)
        assert size > 0
        workspace = torch.empty(size + 16, dtype=torch.uint8, device=device)
        if case != "none":
            args.workspace, args.workspace_size = workspace.data_ptr() + (8 if case == "misaligned" else 0), size - (case == "small")
        if case == "old structure":
            args.struct_size = _lib.TriAttnArgs.workspace.offset
        _lib.check(_lib.lib().tri_attn_fwd(ctypes.byref(args)))
        results.append((o, lse))
    for o, lse in results[1:]:
        assert torch.equal(o, results[0][0]) and torch.equal(lse, results[0][1])
    many = torch.empty(64, 16, 1024, 64, dtype=torch.float16, device=device)
    args = operation._make_args(many, many, many, many, torch.empty(64, 16, 1024, device=device), None, 0.0, True, 0.125, 0, 0)
    assert _lib.lib().tri_attn_workspace_size(ctypes.byref(args), 0) == 0


def test_infinities_in_keys_without_weight_reach_the_output(device, monkeypatch):
    """Probability 0 times an infinite value is NaN, also where the key's whole part of the sequence weighs nothing."""
    S, D = 2048, 128
    q = torch.ones(1, 2, S, D, dtype=torch.bfloat16, device=device)
    k, v = q.clone(), q.clone()
    k[:, :, S // 2:] = -20.0
    v[:, 0, 3 * S // 4, 5] = math.inf
    for split in (True, False):
        (o, *_), used = _run(q, k, v, q, None, 0.0, False, 1.0, (0, 0), split, monkeypatch)
        assert used[0] == split
        assert o[0, 0, :, 5].isnan().all() and torch.equal(o[0, 0, :, :5], v[0, 0, :, :5]) and torch.equal(o[0, 1], v[0, 1])


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype,S,D", [(torch.float32, 640, 64), (torch.float32, 513, 128), (torch.bfloat16, 2048, 128), (torch.float16, 1300, 64)])
def test_keys_of_nan_over_whole_parts_reach_the_output(dtype, S, D, causal, device, monkeypatch):
    """NaN wherever the whole launch gives NaN, whichever part the first or the last key of NaN begins or ends (parts begin at multiples
    of 64): a part with nothing but NaN scores has no maximum, and a sum that is NaN."""
    g = torch.Generator(device=device).manual_seed(S)
    q, k, v, d_o = [torch.randn(1, 2, S, D, generator=g, device=device).to(dtype) for _ in range(4)]
    for first, last in [(n, S) for n in range(64, S, 64)] + [(0, n) for n in range(64, S, 64)]:
        kk = k.clone()
        kk[:, 0, first:last] = math.nan
        whole, _ = _run(q, kk, v, d_o, None, 0.0, causal, 0.125, (0, 0), False, monkeypatch)
        split, used = _run(q, kk, v, d_o, None, 0.0, causal, 0.125, (0, 0), True, monkeypatch)
        assert all(used)
        assert split[0][0, 0, first if causal else 0:].isnan().all(), ("O", first, last)
        for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), split, whole):
            assert torch.equal(a.isnan(), b.isnan()), (name, first, last)


@pytest.mark.parametrize("kind", ["keys", "matrix"])
@pytest.mark.parametrize("S,D", [(2048, 64), (1344, 64), (1300, 32), (2048, 128), (1300, 128), (5120, 64)])
@pytest.mark.parametrize("hidden", [(0, 576), (512, 1152), (640, None)])
@pytest.mark.parametrize("what", ["key", "value", "grad"])
def test_what_a_mask_hides_over_whole_parts_is_not_left_out(what, hidden, S, D, kind, device, monkeypatch):
    """NaN wherever the whole launch gives NaN: probability 0 times a NaN key, an infinite value or an infinite dO row. Whole items leave
    out only tiles before the first or behind the last one that is not masked out altogether."""
    g = torch.Generator(device=device).manual_seed(S)
    q, k, v, d_o = [torch.randn(1, 1, S, D, generator=g, device=device).bfloat16() for _ in range(4)]
    first, last = hidden[0], hidden[1] or S
    mask = torch.zeros(1, 1, 1 if kind == "keys" else S, S, device=device)
    if what == "grad":  # rows that see the first keys only
        if kind == "keys":
            pytest.skip("a mask of keys hides no rows")
        mask[:, :, first:last, 128:] = -math.inf
    else:
        mask[..., first:last] = -math.inf
    spot = (first + last) // 2 // 64 * 64
    {"key": k, "value": v, "grad": d_o}[what][0, 0, spot:spot + 3] = math.nan if what == "key" else math.inf
    whole, _ = _run(q, k, v, d_o, mask, 0.0, False, 0.125, (0, 0), False, monkeypatch)
    split, used = _run(q, k, v, d_o, mask, 0.0, False, 0.125, (0, 0), True, monkeypatch)
    assert all(used)
    for name, a, b in zip(("O", "lse", "dQ", "dK", "dV"), split, whole):
        # (beyond 64 tiles, and in dK/dV at D = 128, whole items leave out nothing, parts what whole ones leave out elsewhere)
        ends = name in ("dK", "dV") and (S > 4096 or S % 128 == 0 and D == 128) or S > 4096 and (hidden[0] == 0 or hidden[1] is None)
        assert not (a.isnan() & ~b.isnan()).any() if ends else torch.equal(a.isnan(), b.isnan()), name


@pytest.mark.parametrize("dtype,heads,S,D,causal,which,split", [
    # whole launch -> split one as it was planned before (us): the plan took a CU for one that holds more workgroups than it does, and a
    # tile for as long beside three other workgroups as alone
    (torch.bfloat16, 25, 1280, 32, False, 0, False),   # forward 16.1 -> 23.7
    (torch.bfloat16, 20, 1237, 32, False, 0, False),   # forward 17.1 -> 23.7
    (torch.float16, 22, 1408, 32, True, 0, False),     # forward 17.6 -> 22.2
    (torch.float16, 21, 4096, 16, True, 1, False),     # dK/dV 70.3 -> 112.3
    (torch.bfloat16, 18, 4224, 32, True, 1, False),    # dK/dV 79.6 -> 115.7
    (torch.float16, 12, 4992, 32, False, 1, False),    # dK/dV 102.3 -> 133.1
    # launches that take half as long split
    (torch.float32, 5, 193, 128, False, 1, True),      # dK/dV 43.3 -> 21.3
    (torch.float32, 9, 768, 128, True, 0, True),       # forward 116.5 -> 38.8
    (torch.bfloat16, 6, 1984, 64, True, 1, True),      # dK/dV 57.9 -> 28.9
    (torch.bfloat16, 6, 3392, 32, True, 1, True)])     # dK/dV 79.4 -> 36.7
def test_launches_that_split(dtype, heads, S, D, causal, which, split, device):
    q = torch.empty(1, heads, S, D, dtype=dtype, device=device)
    lse = torch.empty(1, heads, S, device=device)
    args = operation._make_args(q, q, q, q, lse, None, 0.0, causal, 0.125, 0, 0, q, q, q, q, None, lse)
    assert (_lib.lib().tri_attn_workspace_size(ctypes.byref(args), which) > 0) == split


@pytest.mark.parametrize("dtype,heads,S,D,p,which", [
    # whole launch -> parts (us)
    (torch.bfloat16, 4, 11776, 16, 0.0, 3),   # dQ 255 -> 123
    (torch.bfloat16, 16, 9108, 32, 0.1, 0),   # forward 827 -> 409
    (torch.bfloat16, 16, 9108, 32, 0.1, 1),   # dK/dV 1275 -> 632
    (torch.float16, 24, 6995, 32, 0.0, 0),    # forward 418 -> 189
    (torch.bfloat16, 6, 5694, 128, 0.1, 3)])  # dQ 530 -> 281
def test_key_masks_beyond_64_tiles_split(dtype, heads, S, D, p, which, device):
    """Workgroups of more than 64 tiles do without the mask's classes, which costs them more than many heads make up for. (One part of
    up to 64 tiles has them.)"""
    q = torch.empty(1, heads, S, D, dtype=dtype, device=device)
    lse = torch.empty(1, heads, S, device=device)
    mask = operation._PreparedMask(torch.ones(1, 1, 1, S, dtype=torch.bool, device=device), q)
    args = operation._make_args(q, q, q, q, lse, None, p, False, 0.125, 0, 0, q, q, q, q, None, lse)
    mask.describe(args)
    assert _lib.lib().tri_attn_workspace_size(ctypes.byref(args), which) > 0
    if which != 1 and D < 128:
        args.mask_classes = None  # (nothing to make use of: as a launch that fills the GPU)
        assert _lib.lib().tri_attn_workspace_size(ctypes.byref(args), which) == 0 or heads < 16


@pytest.mark.parametrize("S", [16384, 65536, 262144])
@pytest.mark.parametrize("D,masked", [(16, True), (32, True), (128, False)])
def test_workspaces_are_bounded(S, D, masked, device):
    q = torch.empty(1, 2, S, D, dtype=torch.bfloat16, device=device)
    lse = torch.empty(1, 2, S, device=device)
    args = operation._make_args(q, q, q, q, lse, None, 0.0, False, 0.125, 0, 0, q, q, q, q, None, lse)
    if masked:
        mask = operation._PreparedMask(torch.ones(1, 1, 1, S, dtype=torch.bool, device=device), q)
        mask.describe(args)
    for which in (0, 1, 2, 3):
        assert 0 <= _lib.lib().tri_attn_workspace_size(ctypes.byref(args), which) <= 1 << 28


def test_whole_launches_of_eight_waves_beside_masks_do_not_split(device):
    q = torch.empty(1, 10, 4096, 128, dtype=torch.bfloat16, device=device)
    lse = torch.empty(1, 10, 4096, device=device)
    mask = torch.zeros(1, 10, 4096, 4096, device=device)
    args = operation._make_args(q, q, q, q, lse, mask, 0.1, False, 0.125, 0, 0)
    assert _lib.lib().tri_attn_workspace_size(ctypes.byref(args), 0) == 0  # (forward 90 us, split 213)
    q = torch.empty(1, 8, 6400, 128, dtype=torch.bfloat16, device=device)
    lse = torch.empty(1, 8, 6400, device=device)
    mask = operation._PreparedMask(torch.ones(1, 1, 1, 6400, dtype=torch.bool, device=device), q)
    args = operation._make_args(q, q, q, q, lse, None, 0.0, False, 0.125, 0, 0, q, q, q, q, None, lse)
    mask.describe(args)
    assert _lib.lib().tri_attn_workspace_size(ctypes.byref(args), 2) == 0  # (dQ 287 us, split 400)
