"""Parity of the sibling operations (Softmax, MaskedSoftmax, Dropout) on the GPU, through the operator API and the
C ABI, against the CPU oracle. The first tests of each group are the reference's own (tests/test_softmax.py,
tests/test_masked_softmax.py, tests/test_dropout.py) with seeded inputs and the oracle in place of the run-time
PyTorch call. Tolerance: fp32 atol 1e-4 (the reference's rule is atol 1e-2), fp16/bf16 atol 1e-2 against fp64."""
import numpy as np
import pytest
import torch

import trident_amd as trident
from oracle import rowops
from tests import parity

pytestmark = pytest.mark.gpu


def _pair(shape, seed, dtype=torch.float32):
    g = torch.Generator().manual_seed(seed)
    return torch.randn(shape, generator=g).to(dtype), torch.randn(shape, generator=g).to(dtype)


def _build_mask(shape, seed):
    mask = torch.randint(0, 2, shape, generator=torch.Generator().manual_seed(seed))
    mask[0, :] = mask[:, 0] = 0
    return mask


def _softmax_case(device, x, g, dim, dtype, mask=None, tag=""):
    tx = x.to(device).requires_grad_(True)
    if mask is None:
        out = trident.function.softmax(tx, dim)
    else:
        out = trident.function.masked_softmax(tx, mask.to(device), dim)
    assert out.dtype == dtype and out.shape == x.shape
    out.backward(g.to(device))
    want = rowops.softmax_forward(parity.to64(x), dim, None if mask is None else mask.numpy())
    parity.close(out, want, dtype, tag + " out")
    # the gradient is defined on the stored (rounded) output, like delta in the attention backward
    parity.close(tx.grad, rowops.softmax_backward(parity.to64(out), parity.to64(g), dim), dtype, tag + " grad")
    return out


@pytest.mark.parametrize("y_size, x_size, dim", [(2, 512, 0), (3, 1000, 1), (3, 1000, 0), (2, 512, 1)])
def test_softmax_reference_shapes(y_size, x_size, dim, device):
    x, g = _pair((y_size, x_size), 1)
    _softmax_case(device, x, g, dim, torch.float32, tag="softmax")


@pytest.mark.parametrize("y_size, x_size, dim", [(2, 512, 0), (3, 1000, 1), (3, 1000, 0), (2, 512, 1)])
def test_masked_softmax_reference_shapes(y_size, x_size, dim, device):
    x, g = _pair((y_size, x_size), 2)
    mask = _build_mask((y_size, x_size), 3)
    out = _softmax_case(device, x, g, dim, torch.float32, mask=mask, tag="masked softmax")
    assert (out[mask.bool().to(device)] == 0).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
def test_modules_keep_dtype(dtype, device):
    """tests/test_softmax.py:47-61, tests/test_masked_softmax.py:58-73, tests/test_dropout.py:46-58."""
    x, g = _pair((1, 32), 4, dtype)
    tx = x.to(device).requires_grad_(True)
    out = trident.Softmax(1).forward(tx)
    assert out is not None and out.dtype == dtype
    out.backward(g.to(device))
    assert tx.grad is not None and tx.grad.dtype == dtype
    tx = x.to(device).requires_grad_(True)
    out = trident.MaskedSoftmax(1).forward(tx, _build_mask((1, 32), 5).to(device))
    assert out.dtype == dtype
    out.backward(g.to(device))
    assert tx.grad.dtype == dtype
    x1, g1 = _pair((16,), 6, dtype)
    tx = x1.to(device).requires_grad_(True)
    out = trident.Dropout(0.7).forward(tx)
    assert out is not None and out.dtype == dtype
    out.backward(g1.to(device))
    assert tx.grad is not None and tx.grad.dtype == dtype


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,dim", [((5, 7), 1), ((64, 2048), 1), ((9, 2056), 1), ((3, 5000), 1), ((17, 4097), 1), ((3, 20000), 1),
                                       ((300, 33), 0), ((4, 6, 128), 2)])
def test_softmax_shapes_and_dtypes(shape, dim, dtype, device):
    """16 lanes, a wave or a workgroup per row, rows that stay in registers and rows too long for that (two sweeps),
    16-byte and per-element accesses (odd lengths), the column kernel (dim 0), a contiguous 3-D input along
    its last dimension."""
    x, g = _pair(shape, 10 + shape[-1], dtype)
    _softmax_case(device, x * 3, g, dim, dtype, tag=f"softmax {shape} {dtype}")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("x_size", [1, 3, 9, 255, 505, 513, 1273, 2041, 2047, 2553, 5113, 5121, 10239, 10241])
@pytest.mark.parametrize("offset", [0, 1])
def test_softmax_of_rows_off_the_16_byte_boundaries(x_size, offset, dtype, device):
    """Odd row lengths: the last length that each thread group holds in registers and the first beyond it (a row shares up to
    two 16-byte pieces with its neighbours), with a mask; and the same rows in tensors that are not aligned themselves."""
    rows = 5
    storage, g = _pair((rows * x_size + offset,), 90 + x_size, dtype)
    mask = _build_mask((rows, x_size), 91).to(torch.uint8)
    tx = (storage * 3).to(device)[offset:].view(rows, x_size).requires_grad_(True)
    tg = g.to(device)[offset:].view(rows, x_size)
    out = trident.function.masked_softmax(tx, mask.to(device), 1)
    (grad,) = torch.autograd.grad(out, (tx,), tg)
    want = rowops.softmax_forward(parity.to64(tx.detach()), 1, mask.numpy())
    parity.close(out, want, dtype, f"rows {x_size} + {offset} {dtype}")
    parity.close(grad, rowops.softmax_backward(parity.to64(out), parity.to64(tg), 1), dtype, f"rows {x_size} + {offset} grad")


# Pieces of a row on the edges of what a thread holds: the last piece falls to thread 0 again (129, 513, 2049, 4097, 20481 + the shift), a row
# is two pieces or one more than the threads; the tensor ends inside a piece or on its boundary.
@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("rows", [5, 8])
@pytest.mark.parametrize("x_size", [65, 129, 130, 257, 259, 511, 513, 633, 1027, 2049, 2050, 2555, 4097, 4099, 20483])
def test_rows_keep_to_their_own_elements(x_size, rows, masked, dtype, device):
    """Rows that share 16-byte pieces with their neighbours: every other row is nothing but NaN and infinities (in the gradient, too), which
    the rows between them must neither read as theirs nor overwrite."""
    x, g = _pair((rows, x_size), 4000 + x_size + rows, dtype)
    mask = _build_mask((rows, x_size), x_size).to(torch.uint8) if masked else None
    if masked:
        mask[:, -1] = mask[:, 0] = 0
    clean = slice(0, rows, 2)
    x[1::2], g[1::2] = float("nan"), float("inf")
    tx = x.to(device).requires_grad_(True)
    out = trident.function.masked_softmax(tx, mask.to(device), 1) if masked else trident.function.softmax(tx, 1)
    (grad,) = torch.autograd.grad(out, tx, g.to(device))
    want = rowops.softmax_forward(parity.to64(x[clean]), 1, mask[clean].numpy() if masked else None)
    parity.close(out[clean], want, dtype, "out")
    parity.close(grad[clean], rowops.softmax_backward(parity.to64(out[clean]), parity.to64(g[clean]), 1), dtype, "grad")
    assert out[1::2].isnan().all() and grad[1::2].isnan().all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mask_dtype", [torch.uint8, torch.float16, torch.int64])
@pytest.mark.parametrize("x_size", [8, 63, 64, 65, 97, 256, 257, 512, 1000, 1001, 1024, 1025])
def test_softmax_with_a_mask_off_the_16_byte_boundaries(x_size, mask_dtype, dtype, device):
    """Aligned tensors under a mask that starts one element behind a boundary: rows on 16-byte boundaries and off them, the
    lengths around which short odd rows and long ones change kernels; and the same data one element behind a boundary."""
    rows = 7
    x, g = _pair((rows, x_size), 190 + x_size, dtype)
    mask = _build_mask((rows, x_size), 191)
    storage = torch.zeros(rows * x_size + 1, dtype=mask_dtype, device=device)
    storage[1:] = mask.flatten().to(device)
    for offset in (0, 1):
        base = torch.zeros(rows * x_size + offset, dtype=dtype, device=device)
        base[offset:] = (x * 3).flatten().to(device)
        tx = base[offset:].view(rows, x_size).requires_grad_(True)
        out = trident.function.masked_softmax(tx, storage[1:].view(rows, x_size), 1)
        (grad,) = torch.autograd.grad(out, (tx,), g.to(device))
        want = rowops.softmax_forward(parity.to64(tx.detach()), 1, mask.numpy())
        parity.close(out, want, dtype, f"rows {x_size} + {offset} {dtype} {mask_dtype}")
        parity.close(grad, rowops.softmax_backward(parity.to64(out), parity.to64(g), 1), dtype, f"rows {x_size} + {offset} grad")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("mask_dtype", [torch.uint8, torch.bool, torch.bfloat16, torch.int32, torch.int64])
@pytest.mark.parametrize("x_size", [1280, 4096, 4100, 8192, 8193, 8200, 16384, 24584])
def test_masked_softmax_of_long_rows(x_size, mask_dtype, dtype, device):
    """Rows that a workgroup just holds, and rows of two to six sweeps, whole vectors and shifted ones, masks that a thread keeps
    as they lie in memory and as bits; every byte but 0 of a uint8 mask counts."""
    x, g = _pair((3, x_size), 198, dtype)
    mask = _build_mask((3, x_size), 199)
    given = mask.to(mask_dtype)
    if mask_dtype == torch.uint8:
        given = given * torch.randint(1, 256, given.shape, generator=torch.Generator().manual_seed(1)).to(torch.uint8)
    tx = (x * 3).to(device).requires_grad_(True)
    out = trident.function.masked_softmax(tx, given.to(device), 1)
    out.backward(g.to(device))
    parity.close(out, rowops.softmax_forward(parity.to64((x * 3).to(dtype)), 1, mask.numpy()), dtype, f"{x_size} {mask_dtype} out")
    parity.close(tx.grad, rowops.softmax_backward(parity.to64(out), parity.to64(g), 1), dtype, f"{x_size} {mask_dtype} grad")


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("rows", [1, 2, 4, 5, 8, 9, 15, 16, 17])
@pytest.mark.parametrize("cols,mask_dtype", [(40, None), (1031, torch.uint8), (2056, torch.int64), (4104, torch.float32)])
def test_softmax_down_a_few_rows(rows, cols, mask_dtype, dtype, device):
    """Columns a thread holds whole (up to 16 elements, 4 or 8 in the backward) and the first lengths beyond, whole vectors and
    single elements across the columns, masks, a column that is masked out altogether."""
    x, g = _pair((rows, cols), 170 + rows, dtype)
    if mask_dtype is None:
        _softmax_case(device, x * 3, g, 0, dtype, tag=f"{rows} rows {dtype}")
        return
    mask = _build_mask((rows, cols), 171)
    mask[:, 5] = 1
    tx = (x * 3).to(device).requires_grad_(True)
    out = trident.function.masked_softmax(tx, mask.to(mask_dtype).to(device), 0)
    out.backward(g.to(device))
    want = rowops.softmax_forward(parity.to64((x * 3).to(dtype)), 0, mask.numpy())
    live = [c for c in range(cols) if c != 5]
    assert torch.isnan(out[:, 5]).all() and torch.isnan(tx.grad[:, 5]).all()
    parity.close(out[:, live], want[:, live], dtype, f"{rows} rows {dtype} {mask_dtype}")
    gradient = rowops.softmax_backward(parity.to64(out[:, live]), parity.to64(g[:, live]), 0)
    parity.close(tx.grad[:, live], gradient, dtype, f"{rows} rows grad")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("mask_dtype", [None, torch.uint8, torch.int64])
@pytest.mark.parametrize("rows,cols", [(18, 40), (31, 1031), (32, 2048), (33, 2048), (3, 524288), (16, 524296), (2, 524287), (17, 262144), (17, 262152)])
def test_softmax_down_a_few_rows_of_many_columns(rows, cols, mask_dtype, dtype, device):
    """The lengths and widths at which columns change between one per thread, whole vectors of them and panels."""
    x, g = _pair((rows, cols), 175 + rows, dtype)
    mask = None if mask_dtype is None else _build_mask((rows, cols), 176)
    tx = (x * 3).to(device).requires_grad_(True)
    out = trident.function.softmax(tx, 0) if mask is None else trident.function.masked_softmax(tx, mask.to(mask_dtype).to(device), 0)
    out.backward(g.to(device))
    parity.close(out, rowops.softmax_forward(parity.to64((x * 3).to(dtype)), 0, None if mask is None else mask.numpy()), dtype, f"{rows} x {cols} out")
    parity.close(tx.grad, rowops.softmax_backward(parity.to64(out), parity.to64(g), 0), dtype, f"{rows} x {cols} grad")


def _milliseconds(run):
    for _ in range(3):
        run()
    times = []
    for _ in range(5):
        start, end = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        start.record()
        for _ in range(10):
            run()
        end.record()
        end.synchronize()
        times.append(start.elapsed_time(end) / 10)
    return min(times)


@pytest.mark.parametrize("what", ["mask", "data"])
def test_unaligned_rows_take_a_streaming_kernels_time(what, device):
    """bf16 rows under a mask, and rows themselves, that start off a 16-byte boundary: no more than 3.3 times the time of the
    backward, which moves three tensors on boundaries (with a workgroup per row and element-wise loads throughout, more than
    four times; now 1.7 and 2.1-2.5)."""
    from trident_amd.rowops import _softmax_backward, _softmax_forward
    rows, cols = 32768, 512
    x = torch.randn(rows * cols + 1, device=device).bfloat16()
    mask = (torch.rand(rows * cols + 1, device=device) < 0.25).to(torch.uint8)[1:].view(rows, cols) if what == "mask" else None
    x = x[1:].view(rows, cols) if what == "data" else x[:-1].view(rows, cols)
    out = _softmax_forward(x, mask, 1, "forward")
    forward = _milliseconds(lambda: _softmax_forward(x, mask, 1, "forward"))
    backward = _milliseconds(lambda: _softmax_backward(out, out, 1, "backward"))
    assert forward <= 3.3 * backward, (forward, backward)


@pytest.mark.parametrize("cols", [17, 33, 49])
def test_short_odd_rows_take_a_streaming_kernels_time(cols, device):
    """bf16, 16.7 M elements: backward no longer than three times that of the even length beside it (cut along the tensor's pieces,
    which are then mostly shared ones, it took four times)."""
    from trident_amd.rowops import _softmax_backward, _softmax_forward
    times = []
    for n in (cols, cols // 8 * 8 + 8):
        x = torch.randn((1 << 24) // n, n, device=device).bfloat16()
        out = _softmax_forward(x, None, 1, "forward")
        times.append(_milliseconds(lambda: _softmax_backward(x, out, 1, "backward")))
    assert times[0] <= 3 * times[1], times


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_a_few_long_rows_take_a_streaming_kernels_time(dtype, device):
    """The forward moves two tensors where the backward moves three: it takes no more than twice the backward's time (in panels,
    bound by exponentials of elements that do not exist, it took three times)."""
    from trident_amd.rowops import _softmax_backward, _softmax_forward
    x = torch.randn(2, 1 << 22, device=device).to(dtype)
    out = _softmax_forward(x, None, 0, "forward")
    forward = _milliseconds(lambda: _softmax_forward(x, None, 0, "forward"))
    backward = _milliseconds(lambda: _softmax_backward(x, out, 0, "backward"))
    assert forward <= 2 * backward, (forward, backward)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,mask_dtype", [((2, 40), None), ((129, 2056), torch.uint8), ((4101, 24), torch.int64), ((300, 777), torch.bfloat16),
                                              ((20000, 8), None), ((35001, 3), torch.bool), ((1025, 4096), None)])
def test_softmax_down_the_columns(shape, mask_dtype, dtype, device):
    """The column kernels: columns that stay in registers and columns swept twice, whole vectors and single elements across
    the columns (odd widths), panels of every width, fewer panels than XCDs, masks of every element size."""
    x, g = _pair(shape, 70 + shape[1], dtype)
    mask = None if mask_dtype is None else _build_mask(shape, 71).to(mask_dtype)
    if mask_dtype is None:
        _softmax_case(device, x * 3, g, 0, dtype, tag=f"columns {shape} {dtype}")
        return
    tx = (x * 3).to(device).requires_grad_(True)
    out = trident.function.masked_softmax(tx, mask.to(device), 0)
    out.backward(g.to(device))
    want = rowops.softmax_forward(parity.to64((x * 3).to(dtype)), 0, mask.float().numpy())
    parity.close(out, want, dtype, f"columns {shape} {dtype} {mask_dtype}")
    parity.close(tx.grad, rowops.softmax_backward(parity.to64(out), parity.to64(g), 0), dtype, f"columns {shape} grad")


@pytest.mark.parametrize("mask_dtype", [torch.int64, torch.int32, torch.bool, torch.uint8, torch.float32, torch.bfloat16])
def test_masked_softmax_mask_dtypes_and_fully_masked_row(mask_dtype, device):
    x, g = _pair((6, 300), 20, torch.bfloat16)
    mask = _build_mask((6, 300), 21)
    mask[3, :] = 1  # a fully masked row is NaN, like softmax over -inf
    tx = x.to(device)
    out = trident.function.masked_softmax(tx, mask.to(mask_dtype).to(device), 1)
    want = rowops.softmax_forward(parity.to64(x), 1, mask.numpy())
    parity.close(out, want, torch.bfloat16, f"mask {mask_dtype}")
    assert torch.isnan(out[3]).all() and not torch.isnan(out[2]).any()


def test_softmax_of_a_transposed_view_and_large_values(device):
    x, g = _pair((40, 70), 30)
    xt = (x * 30).t()  # strides (1, 70): rows are columns of the storage
    _softmax_case(device, xt, g.t(), 1, torch.float32, tag="transposed")
    big = torch.tensor([[1e4, 1e4 - 1, -1e4, 0.0]])
    out = trident.function.softmax(big.to(device), 1)
    parity.close(out, rowops.softmax_forward(parity.to64(big), 1), torch.float32, "large values")


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("masked", [False, True])
@pytest.mark.parametrize("shape,dim", [((5, 100), 1), ((5, 128), 1), ((3, 4096), 1), ((3, 2047), 1), ((2, 20000), 1), ((9, 33), 0), ((40, 64), 0),
                                       ((300, 33), 0), ((3000, 64), 0)])
def test_softmax_of_elements_far_from_zero(shape, dim, masked, dtype, device):
    """Rows and columns around a large number, as masks that fill with one leave them: all alike, differences of a few units,
    sizes around that from which the maximum is subtracted before the product with log2 e, and such elements among ordinary ones."""
    x, g = _pair(shape, 193)
    g = g.to(dtype)
    mask = _build_mask(shape, 194) if masked else None
    for centre in (-1e9, 1e9, -1e10, 1e10, -1e30, -2e38, 2e38):
        _softmax_case(device, torch.full(shape, centre, dtype=dtype), g, dim, dtype, mask, f"{centre}")
    for centre in (3e6, -1.04e9, 1.04e9, -1e10, 1e38):
        _softmax_case(device, (x.double() + centre).to(dtype), g, dim, dtype, mask, f"around {centre}")
    place = torch.arange(shape[dim]).view((-1, 1) if dim == 0 else (1, -1))
    for fill in (-1e9, -1e10, -1e30):
        _softmax_case(device, torch.where(place >= 7, fill, x).to(dtype), g, dim, dtype, mask, f"{fill} from the eighth on")
    lines = torch.arange(shape[1 - dim]).view((1, -1) if dim == 0 else (-1, 1))
    _softmax_case(device, torch.where(lines % 2 == 0, -1e20, x).to(dtype), g, dim, dtype, mask, "every other one far")


# ------------------------------------------------------------------ dropout
@pytest.mark.parametrize("x_size, p", [(256, 0.0), (512, 1.0)])
def test_dropout_reference_cases(x_size, p, device):
    """tests/test_dropout.py:22-43: p = 0 is the identity, p = 1 gives zeros, for values and gradient."""
    x, g = _pair((x_size,), 40)
    tx = x.to(device).requires_grad_(True)
    out = trident.function.dropout(tx, p)
    out.backward(g.abs().to(device))
    want = torch.nn.functional.dropout(x, p)
    assert torch.equal(out.cpu(), want)
    assert torch.equal(tx.grad.cpu(), g.abs() if p == 0.0 else torch.zeros_like(g))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("shape,p", [((4096,), 0.1), ((33, 77), 0.5), ((1, 5), 0.9), ((8, 128, 64), 0.25)])
def test_dropout_is_bit_exact_against_the_documented_stream(shape, p, dtype, device):
    x, g = _pair(shape, 50, dtype)
    trident.config.dropout_seed = (0xD0C5EED, 11)
    try:
        tx = x.to(device).requires_grad_(True)
        out = trident.function.dropout(tx, p)
        out.backward(g.to(device))
    finally:
        trident.config.dropout_seed = None
    keep = rowops.dropout_keep(0xD0C5EED, 11, x.numel(), p).reshape(shape)
    assert np.array_equal((out != 0).cpu().numpy() | (x == 0).numpy(), keep | (x == 0).numpy())
    parity.close(out, rowops.dropout_apply(parity.to64(x), p, 0xD0C5EED, 11), dtype, "dropout out")
    parity.close(tx.grad, rowops.dropout_apply(parity.to64(g), p, 0xD0C5EED, 11), dtype, "dropout grad")


def test_dropout_seeding_and_eval_mode(device):
    x = torch.randn(1000, generator=torch.Generator().manual_seed(60)).to(device)
    torch.manual_seed(5)
    a = trident.function.dropout(x, 0.4)
    torch.manual_seed(5)
    b = trident.function.dropout(x, 0.4)
    c = trident.function.dropout(x, 0.4)
    assert torch.equal(a, b) and not torch.equal(a, c)
    layer = trident.Dropout(0.4).eval()
    assert torch.equal(layer(x), x)
