"""Long columns of narrow matrices: launches split along the columns (a workspace, two launches) against whole ones and 64 bits."""
import ctypes

import pytest
import torch

from trident_amd import _lib, rowops

pytestmark = pytest.mark.gpu


def _run(x, mask, grad, split, monkeypatch):
    """Output and gradient of softmax along dim 0, and whether both launches were split."""
    used = []
    take = rowops._take_workspace

    def spy(args, backward, device):
        workspace = take(args, backward, device) if split else None
        if workspace is not None:
            workspace.fill_(255)  # (NaN wherever nothing is written before it is read)
        used.append(workspace is not None)
        return workspace

    with monkeypatch.context() as m:
        m.setattr(rowops, "_take_workspace", spy)
        out = rowops._softmax_forward(x, mask, 0, "")
        return (out, rowops._softmax_backward(grad, out, 0, "")), used


@pytest.mark.parametrize("mask_dtype", [None, torch.uint8, torch.float32, torch.int64])
@pytest.mark.parametrize("dtype,rows,cols", [(torch.float32, 9000, 4), (torch.float32, 8193, 132), (torch.float32, 2049, 33), (torch.bfloat16, 8193, 8),
                                             (torch.bfloat16, 9485, 232), (torch.float16, 1025, 156), (torch.float16, 40000, 24), (torch.bfloat16, 200000, 1)])
def test_split_columns(dtype, rows, cols, mask_dtype, device, monkeypatch):
    g = torch.Generator(device=device).manual_seed(rows + cols)
    x = torch.randn(rows, cols, generator=g, device=device).mul_(3).to(dtype)
    x[rows // 2:, 0] = -1e4       # (parts that weigh nothing)
    grad = torch.randn(rows, cols, generator=g, device=device).to(dtype)
    mask = None if mask_dtype is None else (torch.rand(rows, cols, generator=g, device=device) < 0.25).to(mask_dtype)
    if cols > 3 and mask is not None:
        mask[:, 1] = 1            # (a column without an element: NaN)
        mask[: rows - 7, 2] = 1   # (parts without one)
    whole, used = _run(x, mask, grad, False, monkeypatch)
    split, used = _run(x, mask, grad, True, monkeypatch)
    assert all(used) or cols == 1  # (a single column is contiguous down its length: a row)
    again, _ = _run(x, mask, grad, True, monkeypatch)
    hidden = torch.zeros(x.shape, dtype=torch.bool, device=device) if mask is None else mask > 0
    exact = x.double().masked_fill(hidden, float("-inf")).softmax(0)
    want = exact * (grad.double() - (exact * grad.double()).sum(0))
    for a, b, c, e in zip(split, whole, again, (exact, want)):
        assert torch.equal(a.nan_to_num(7.0), c.nan_to_num(7.0)) and torch.equal(a.isnan(), e.isnan())
        a, b, e = a.double().nan_to_num(0.0), b.double().nan_to_num(0.0), e.nan_to_num(0.0)
        assert (a - e).norm() <= 1.05 * (b - e).norm() + 1e-7 * e.norm()
        assert (a - e).abs().max() <= 1.5 * (b - e).abs().max() + 1e-7 * e.abs().max()


@pytest.mark.parametrize("dtype,rows,cols", [(torch.float32, 2049, 512), (torch.float32, 4096, 500), (torch.bfloat16, 4000, 1024), (torch.float16, 2100, 1023),
                                             (torch.float32, 4096, 2052), (torch.float32, 2049, 3072), (torch.bfloat16, 2100, 8192), (torch.float32, 2049, 7672),
                                             (torch.float32, 2300, 4608)])
def test_panels_of_32_bytes(dtype, rows, cols, device, monkeypatch):
    """The backward's narrow panels, whose lines are dealt out in another order: numbers of them that are dealt, do not fill up the last
    XCD, or stay in order. A panel's sums do not depend on its place: equal to those of the same columns in another matrix."""
    g = torch.Generator(device=device).manual_seed(rows + cols)
    x, grad = [torch.randn(rows, cols, generator=g, device=device).to(dtype) for _ in range(2)]
    (out, dx), _ = _run(x, None, grad, False, monkeypatch)
    exact = x.double().softmax(0)
    want = exact * (grad.double() - (exact * grad.double()).sum(0))
    limit = {torch.float32: 1e-6, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}[dtype]  # (half an ulp of every element and of the output)
    for a, e in ((out, exact), (dx, want)):
        per_column = (a.double() - e).norm(dim=0) / e.norm(dim=0)
        assert per_column.max() <= 1.5 * limit
    if cols % 8 == 0:
        (_, again), _ = _run(x.roll(cols // 2, 1), None, grad.roll(cols // 2, 1), False, monkeypatch)
        assert torch.equal(again, dx.roll(cols // 2, 1))


def test_columns_far_from_zero(device, monkeypatch):
    x = torch.randn(9000, 12, device=device)
    x[:, 3] -= 1e10
    x[:, 5] = -1e30
    grad = torch.randn_like(x)
    split, used = _run(x, None, grad, True, monkeypatch)
    whole, _ = _run(x, None, grad, False, monkeypatch)
    assert all(used)
    assert torch.equal(split[0][:, 3], whole[0][:, 3]) and torch.equal(split[0][:, 5], whole[0][:, 5])
    assert (split[0] - whole[0]).abs().max() <= 1e-6 * whole[0].max()


def test_old_structures_run_whole(device):
    x, out = torch.randn(9000, 8, device=device), torch.empty(9000, 8, device=device)
    args = rowops._row_args(x, 0)
    args.input, args.output = x.data_ptr(), out.data_ptr()
    assert _lib.lib().tri_softmax_workspace_size(ctypes.byref(args), 0) > 0
    args.struct_size = _lib.TriRowArgs.workspace.offset
    _lib.check(_lib.lib().tri_softmax_fwd(ctypes.byref(args)))
    assert (out.double() - x.double().softmax(0)).abs().max() <= 1e-6
