"""Rows that are no multiple of a 16-byte pack, or that start unaligned: the softmax and
cross-entropy kernels read them in unaligned packs whose last one overlaps the one before.

Widths: one pack and its neighbours, one past each workgroup width's whole packs, the
cross-entropy backward's change from rows to the flat matrix (8192 16-bit or 4096 fp32
columns), and rows past the register kernels. ``offset`` moves the tensors off 16-byte
alignment. References in fp64; a 16-bit result within two roundings (softmax's backward
reads a rounded y), an fp32 one within 1e-5 (the declarations' gate)."""

import pytest
import torch

from evograd_amd import _lib, pair_module

pytestmark = pytest.mark.gpu
EPS = {torch.float32: 1e-5, torch.float16: 2.0 ** -9, torch.bfloat16: 2.0 ** -6}
# fp16 entries below 2^-14 are subnormal, spaced by 2^-24: a rounding moves them by up to half
# of that whatever their size (bf16 and fp32 have fp32's exponent range)
FLOOR = {torch.float32: 0.0, torch.float16: 2.0 ** -25, torch.bfloat16: 0.0}


def _at(t, offset):
    """A contiguous copy of t that starts ``offset`` elements into its storage."""
    flat = torch.full((t.numel() + offset,), float("nan"), device="cuda", dtype=t.dtype)
    flat[offset:] = t.reshape(-1)
    return flat[offset:].view(t.shape)


def _close(got, want, dtype, scale=1.0):
    tol = EPS[dtype] * (want.abs() + scale) + FLOOR[dtype]
    assert ((got.double() - want).abs() <= tol).all(), (got.double() - want).abs().max()


CASES = [(5, 1, 0), (3, 3, 0), (7, 4, 1), (5, 7, 0), (5, 8, 1), (6, 9, 0), (9, 513, 0), (4, 1000, 3),
         (3, 1025, 0), (5, 4097, 0), (3, 8191, 0), (4, 8193, 0), (3, 8200, 1), (2, 32769, 0),
         (2, 65544, 3), (2, 65537, 0), (1, 131075, 0)]


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("rows,cols,offset", CASES)
def test_softmax_ragged_rows(rows, cols, offset, dtype):
    print(f"\n[gpu-ragged] softmax {rows}x{cols}+{offset} {dtype}", flush=True)
    mod = pair_module("softmax")
    g = torch.Generator(device="cuda").manual_seed(rows * 1000 + cols)
    x = _at((2 * torch.randn(rows, cols, device="cuda", generator=g)).to(dtype), offset)
    dy = _at(torch.randn(rows, cols, device="cuda", generator=g).to(dtype), offset)
    y, saved = mod.softmax_forward_with_saved(x)
    want = torch.softmax(x.double(), -1)
    _close(y, want, dtype, scale=0.0 if dtype == torch.bfloat16 else 1e-4)
    dx = mod.softmax_backward_from_saved(dy, saved)
    yd, gd = y.double(), dy.double()
    _close(dx, yd * (gd - (gd * yd).sum(-1, keepdim=True)), dtype, scale=1.0 / cols)


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("rows,cols,offset", CASES)
def test_cross_entropy_ragged_rows(rows, cols, offset, dtype):
    print(f"\n[gpu-ragged] cross_entropy {rows}x{cols}+{offset} {dtype}", flush=True)
    mod = pair_module("cross_entropy")
    g = torch.Generator(device="cuda").manual_seed(rows * 1000 + cols)
    x = _at((2 * torch.randn(rows, cols, device="cuda", generator=g)).to(dtype), offset)
    target = torch.randint(0, cols, (rows,), device="cuda", generator=g)
    target[0] = cols - 1  # in the overlapping pack
    if rows > 3:
        target[2] = -100
    loss, saved = mod.cross_entropy_forward_with_saved(x, target)
    ok = target != -100
    n = ok.sum()
    lse = torch.logsumexp(x.double(), -1)
    at = target.clamp(min=0)[:, None]
    _close(loss, ((lse - x.double().gather(1, at)[:, 0]) * ok).sum() / n, dtype)
    dl = mod.cross_entropy_backward_from_saved(torch.ones((), device="cuda", dtype=dtype), saved)
    want = torch.exp(x.double() - lse[:, None]).scatter_add(
        1, at, -torch.ones_like(at, dtype=torch.float64)) * (ok[:, None] / n)
    _close(dl, want, dtype, scale=1.0 / (rows * cols))


# Row counts on both sides of the lines between single elements and packs, per width.
LINES = [(16383, 65, 0), (16384, 67, 0), (32768, 127, 0), (2047, 129, 1), (2048, 200, 1),
         (4095, 511, 0), (4096, 257, 0), (1023, 513, 0), (1024, 1001, 3), (2048, 2047, 0),
         (511, 2049, 0), (512, 4095, 0), (1024, 2050, 1)]


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("rows,cols,offset", LINES)
def test_softmax_ragged_rows_many(rows, cols, offset, dtype):
    test_softmax_ragged_rows(rows, cols, offset, dtype)


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
@pytest.mark.parametrize("rows,cols", [(2048, 501), (4096, 501), (1024, 3739), (3, 33333),
                                       (2, 131075)])
def test_softmax_ragged_rows_in_place(rows, cols, dtype):
    """y over x, and dx over dy or over y, give the bits of separate buffers."""
    print(f"\n[gpu-ragged] softmax in place {rows}x{cols} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
    dy = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
    tail = (rows, cols, _lib.dtype_tag(dtype), _lib.stream_of(x))
    y, z, dx = torch.empty_like(x), x.clone(), torch.empty_like(x)
    for a, b in ((x, y), (z, z)):
        _lib.call("eg_softmax_fwd", a.data_ptr(), b.data_ptr(), *tail)
    assert torch.equal(y, z)
    _lib.call("eg_softmax_bwd", y.data_ptr(), dy.data_ptr(), dx.data_ptr(), *tail)
    over_dy, over_y = dy.clone(), y.clone()
    _lib.call("eg_softmax_bwd", y.data_ptr(), over_dy.data_ptr(), over_dy.data_ptr(), *tail)
    _lib.call("eg_softmax_bwd", over_y.data_ptr(), dy.data_ptr(), over_y.data_ptr(), *tail)
    assert torch.equal(dx, over_dy) and torch.equal(dx, over_y)


# Both sides of the lines between the backward's kernels (rows, flat with many rows or two per
# workgroup; packs or single elements) and of the forward's: whole packs, then ragged.
XENT_LINES = [(4095, 64, 0), (4096, 64, 0), (4096, 1280, 0), (4096, 1288, 0), (4097, 2048, 0),
              (300, 4088, 0), (300, 8184, 0), (200, 8192, 0),
              (6000, 9, 0), (6001, 9, 0), (6001, 255, 1), (6001, 897, 0), (6100, 1023, 3),
              (1100, 1025, 0), (1534, 1025, 0), (1535, 1025, 0), (193, 8193, 0), (33, 50257, 0),
              (70000, 5, 0)]


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("rows,cols,offset", XENT_LINES)
def test_cross_entropy_rows_many(rows, cols, offset, dtype):
    test_cross_entropy_ragged_rows(rows, cols, offset, dtype)


@pytest.mark.parametrize("dtype", (torch.float32, torch.bfloat16))
@pytest.mark.parametrize("rows,cols", [(6001, 33), (2000, 1277), (193, 8193), (5, 70), (4096, 64)])
def test_cross_entropy_backward_in_place(rows, cols, dtype):
    """dlogits over the logits gives the bits of separate buffers."""
    print(f"\n[gpu-ragged] cross_entropy in place {rows}x{cols} {dtype}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(cols)
    x = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
    t = torch.randint(0, cols, (rows,), device="cuda", generator=g)
    lse = torch.logsumexp(x.float(), -1)
    up, n = torch.ones((), device="cuda", dtype=dtype), torch.full((1,), float(rows), device="cuda")
    dx, z = torch.empty_like(x), x.clone()
    for a, b in ((x, dx), (z, z)):
        _lib.call("eg_cross_entropy_bwd", up.data_ptr(), a.data_ptr(), t.data_ptr(),
                  lse.data_ptr(), n.data_ptr(), b.data_ptr(), rows, cols, -100,
                  _lib.dtype_tag(dtype), _lib.stream_of(x))
    assert torch.equal(dx, z)
