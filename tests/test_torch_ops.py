"""The C++ host path (csrc_torch/torch_ops.cpp) against the Python autograd Functions it stands in for: the same launches, so the
same bits; and the calls it hands back to them."""
import pytest
import torch

import trident_amd as trident
from trident_amd import _lib, operation


def test_calls_that_are_not_plain_are_handed_back():
    """CPU tensors, subclasses, other argument types: None and no exception (the Python Functions raise what there is to raise)."""
    ops = _lib.torch_ops()
    x = torch.zeros(1, 1, 8, 16)
    for args in ((x, x, x, None, 0.0, False, 0.25), (x, x, None, None, 0.0, False, 0.25), (x, x, x, "mask", 0.0, False, 0.25)):
        assert ops.attention(*args) is None
    assert ops.softmax(x[0, 0], None, 1) is None
    assert ops.dropout(x[0, 0], 0.5) is None


class _Subclass(torch.Tensor):
    pass


@pytest.mark.gpu
def test_watched_calls_are_handed_back(device):
    ops = _lib.torch_ops()
    x = torch.zeros(1, 1, 64, 16, dtype=torch.float16, device=device)

    def native(t=x):
        return ops.attention(t, t, t, None, 0.0, False, 0.25) is not None

    assert native()
    assert not native(x.as_subclass(_Subclass))
    with torch.device("cpu"):  # (a torch function mode)
        assert not native()
    with torch.autograd.forward_ad.dual_level():
        assert not native()
    seen = []
    torch.func.vmap(lambda t: seen.append(native()) or t)(torch.zeros(2))
    assert seen == [False]
    trident.config.use_trace = True
    try:
        assert not native()
    finally:
        trident.config.use_trace = False


def _mask(kind, B, H, S, dtype, device):
    g = torch.Generator(device=device).manual_seed(S)
    if kind == "none":
        return None
    if kind == "bool":
        keep = torch.rand(B, 1, 1, S, generator=g, device=device) > 0.3
        keep[..., 0] = True
        return keep
    shape = {"full grad": (B, H, S, S), "shared grad": (1, H, S, S), "keys grad": (B, 1, 1, S), "matrix": (S, S), "length": (B, 1, S, S)}[kind]
    mask = torch.randn(shape, generator=g, device=device)
    if kind == "length":
        mask = torch.zeros(shape, device=device)
        mask[..., S // 2:] = float("-inf")
    return (mask.to(dtype) if "grad" in kind else mask).requires_grad_("grad" in kind)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["none", "bool", "full grad", "shared grad", "keys grad", "matrix", "length"])
@pytest.mark.parametrize("dtype,S,D,p,layout", [(torch.bfloat16, 128, 64, 0.0, "bhsd"), (torch.float16, 100, 32, 0.2, "bshd"),
                                                (torch.float32, 65, 16, 0.2, "bhsd"), (torch.bfloat16, 777, 128, 0.0, "bshd")])
def test_attention_is_the_function_it_stands_in_for(kind, dtype, S, D, p, layout, device, monkeypatch):
    monkeypatch.setattr(trident.config, "reference_limits", False)
    B, H = 2, 3
    g = torch.Generator(device=device).manual_seed(S + D)
    make = (lambda: torch.randn(B, S, H, D, generator=g, device=device).to(dtype).transpose(1, 2)) if layout == "bshd" else \
        (lambda: torch.randn(B, H, S, D, generator=g, device=device).to(dtype))
    q, k, v, grad = make().requires_grad_(), make(), make().requires_grad_(), make()
    mask = _mask(kind, B, H, S, dtype, device)
    inputs = [q, v] + ([mask] if "grad" in kind else [])
    results = []
    for f in (operation.Attention.call, operation.Attention.apply):
        monkeypatch.setattr(trident.config, "dropout_seed", (5, 1))
        packed = []
        with torch.autograd.graph.saved_tensors_hooks(lambda t: packed.append(tuple(t.shape)) or t, lambda t: t):
            out = f(q, k, v, mask, p, False, 0.125, False)
        first = torch.autograd.grad(out, inputs, grad, retain_graph=True)
        results.append(([out.detach(), *first], packed))
        for a, b in zip(first, torch.autograd.grad(out, inputs, grad)):
            if a is not first[-1] or kind != "keys grad":  # (that gradient is added up atomically)
                assert torch.equal(a, b)
        with torch.no_grad():
            monkeypatch.setattr(trident.config, "dropout_seed", (5, 1))
            assert torch.equal(f(q, k, v, mask, p, False, 0.125, False), out)
    assert results[0][1] == results[1][1]
    for n, (a, b) in enumerate(zip(results[0][0], results[1][0])):
        assert a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
        if kind == "keys grad" and n == 3:
            assert (a - b).abs().max() <= 1e-2 * b.abs().max()  # (fp32 atomic adds in another order, rounded to the mask's type)
        else:
            assert torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,B,H,S,D,kind,causal,p", [
    (torch.bfloat16, 1, 2, 2048, 128, "none", True, 0.0), (torch.float16, 1, 3, 1300, 64, "bool", False, 0.0),
    (torch.bfloat16, 2, 1, 1408, 32, "length", False, 0.2), (torch.bfloat16, 1, 2, 1300, 64, "shared grad", False, 0.0),
    (torch.float32, 1, 3, 513, 64, "none", True, 0.0), (torch.float32, 2, 1, 640, 128, "matrix", False, 0.2)])
def test_split_attention_is_the_function_it_stands_in_for(dtype, B, H, S, D, kind, causal, p, device, monkeypatch):
    """Both host paths give a call of few heads the workspace with which it runs split, in both directions: the same bits, and other
    ones than without a workspace (parts add their sums up in another order)."""
    monkeypatch.setattr(trident.config, "reference_limits", False)
    g = torch.Generator(device=device).manual_seed(S + D)
    q, k, v, grad = [torch.randn(B, H, S, D, generator=g, device=device).to(dtype) for _ in range(4)]
    q, k, v = [t.requires_grad_() for t in (q, k, v)]
    mask = _mask(kind, B, H, S, dtype, device)
    inputs = [q, k, v] + ([mask] if "grad" in kind else [])
    take, used = operation._take_workspace, []

    def spy(args, which, gpu):
        workspace = take(args, which, gpu)
        used.append(workspace is not None)
        return workspace

    def run(f):
        monkeypatch.setattr(trident.config, "dropout_seed", (5, 1))
        out = f(q, k, v, mask, p, causal, 0.125, False)
        return [out.detach(), *torch.autograd.grad(out, inputs, grad)]

    got = run(operation.Attention.call)
    monkeypatch.setattr(operation, "_take_workspace", spy)
    want = run(operation.Attention.apply)
    assert len(used) >= 2 and all(used[:2])
    monkeypatch.setattr(operation, "_take_workspace", lambda *_: None)
    whole = run(operation.Attention.apply)
    for a, b in zip(got, want):
        assert torch.equal(a, b)
    for a, b in zip(got[:4], whole):
        assert not torch.equal(a, b)


@pytest.mark.gpu
@pytest.mark.parametrize("shape,dim", [((40, 33), 0), ((40, 33), 1), ((40, 33), None), ((3, 5, 16), -1)])
@pytest.mark.parametrize("masked", [False, True])
def test_row_operations_are_the_functions_they_stand_in_for(shape, dim, masked, device, monkeypatch):
    g = torch.Generator(device=device).manual_seed(7)
    x = torch.randn(shape, generator=g, device=device).requires_grad_()
    grad = torch.randn(shape[::-1], generator=g, device=device).permute(*reversed(range(len(shape))))
    mask = torch.rand(shape[-1:], generator=g, device=device) > 0.7  # (broadcast over the rows)
    mask[0] = False

    def run(softmax, dropout):
        monkeypatch.setattr(trident.config, "dropout_seed", (9, 4))
        y = softmax()
        z = dropout(y) if len(shape) == 2 else y
        return [y.detach(), z.detach(), *torch.autograd.grad(z, x, grad)]

    got = run(lambda: trident.function.masked_softmax(x, mask, dim) if masked else trident.function.softmax(x, dim),
              lambda y: trident.function.dropout(y, 0.25))
    want = run(lambda: operation.MaskedSoftmax.apply(x, mask, dim) if masked else operation.Softmax.apply(x, dim),
               lambda y: operation.Dropout.apply(y, 0.25))
    for a, b in zip(got, want):
        assert torch.equal(a.nan_to_num(7.0), b.nan_to_num(7.0)) and a.stride() == b.stride()  # (masked out columns: NaN)


@pytest.mark.gpu
def test_a_call_that_fails_raises_as_before(device):
    x = torch.zeros(1, 1, 64, 16, dtype=torch.float16, device=device)
    with pytest.raises(RuntimeError, match="dropout_p must lie in"):
        trident.function.scaled_dot_product_attention(x, x, x, None, 1.5)
    with pytest.raises(RuntimeError, match="expanded size"):
        trident.function.scaled_dot_product_attention(x, x, x, torch.zeros(3, 64, device=device))
    with pytest.raises(RuntimeError, match="dropout_p must lie in"):
        trident.function.dropout(x[0, 0], 1.5)


@pytest.mark.gpu
@pytest.mark.parametrize("unpack", [lambda t: t.cpu(), lambda t: t.double(), lambda t: t[..., :8]])
def test_saved_tensors_that_come_back_changed_are_refused(unpack, device):
    """A hook's unpack may return anything: what the kernels could not read raises, and nothing is launched."""
    x = torch.zeros(1, 1, 64, 16, dtype=torch.float16, device=device, requires_grad=True)
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        outputs = [trident.function.scaled_dot_product_attention(x, x, x), trident.function.softmax(x[0, 0], 1)]
    for out in outputs:
        with pytest.raises(RuntimeError, match="trident_amd: .*(on the same GPU|another shape or dtype)"):
            out.sum().backward()


def _wider(t):
    """The same values in rows of a wider buffer."""
    return torch.zeros(t.shape[:-1] + (t.shape[-1] + 8,), dtype=t.dtype, device=t.device)[..., : t.shape[-1]].copy_(t)


def _turned(t):
    """The same values with the first and the last dimension exchanged in memory."""
    return t.transpose(0, -1).contiguous().transpose(0, -1)


@pytest.mark.gpu
@pytest.mark.parametrize("path", ["C++", "Python"])
@pytest.mark.parametrize("unpack", [_wider, _turned, lambda t: t.clone()])
@pytest.mark.parametrize("operation_of", ["rows", "columns", "3-d", "attention"])
def test_saved_tensors_that_come_back_in_another_layout(operation_of, unpack, path, device):
    """Equal values, other strides: the gradients of a call without the hook, bit for bit."""
    g = torch.Generator(device=device).manual_seed(3)
    shape, dim = {"rows": ((40, 60), 1), "columns": ((40, 60), 0), "3-d": ((3, 5, 60), -1), "attention": ((2, 3, 64, 32), None)}[operation_of]
    x = torch.randn(shape, generator=g, device=device).half().requires_grad_()
    grad = torch.randn(shape, generator=g, device=device).half()

    def call():
        if dim is None:
            return operation.Attention.apply(x, x, x, None, 0.0, False, 0.25, False) if path == "Python" else trident.function.attention(x, x, x, softmax_scale=0.25)
        return operation.Softmax.apply(x, dim) if path == "Python" else trident.function.softmax(x, dim)

    want = torch.autograd.grad(call(), x, grad)[0]
    if dim is None and unpack is _turned:
        # (lse only: rows of q, k, v and o of another stride are copied or refused)
        unpack = lambda t: _turned(t) if t.dim() == 3 else t
    with torch.autograd.graph.saved_tensors_hooks(lambda t: t, unpack):
        out = call()
    assert torch.equal(torch.autograd.grad(out, x, grad)[0], want)
