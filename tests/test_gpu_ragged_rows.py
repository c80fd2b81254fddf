"""Rows that are no multiple of a 16-byte pack, or that start unaligned: the softmax and
cross-entropy kernels read them in unaligned packs whose last one overlaps the one before.

Widths: one pack and its neighbours, one past each workgroup width's whole packs, the
cross-entropy backward's change from rows to the flat matrix (8192 16-bit or 4096 fp32
columns), and rows past the register kernels. ``offset`` moves the tensors off 16-byte
alignment. References in fp64; a 16-bit result within two roundings (softmax's backward
reads a rounded y), an fp32 one within 1e-5 (the declarations' gate)."""

import pytest
import torch

from evograd_amd import pair_module

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
