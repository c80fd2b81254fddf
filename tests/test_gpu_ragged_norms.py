"""The norm kernels on rows that are no multiple of a 16-byte pack or start unaligned, and
both programs of the backward entry points: one launch up to 256 rows, the ring above.

Widths: one pack and its neighbours, and one past each workgroup width's whole packs.
References in fp64. A 16-bit result is one rounding of fp32 arithmetic on exact inputs; the
fp32 bound is the declarations' 1e-5, relative to the row's or column's scale."""

import pytest
import torch

from evograd_amd import pair_module

pytestmark = pytest.mark.gpu
ULP = {torch.float32: 0.0, torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8}


def _at(t, offset):
    flat = torch.full((t.numel() + offset,), float("nan"), device="cuda", dtype=t.dtype)
    flat[offset:] = t.reshape(-1)
    return flat[offset:].view(t.shape)


def _close(got, want, dtype, scale):
    tol = 1e-5 * scale + ULP[dtype] * want.abs() + 2.0 ** -25
    assert ((got.double() - want).abs() <= tol).all(), (got.double() - want).abs().max()


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("op", ("rmsnorm", "layernorm", "fused_add_rms_norm"))
@pytest.mark.parametrize("rows,cols,offset", [
    (3, 3, 0), (5, 4, 1), (4, 7, 0), (9, 8, 1), (6, 9, 0), (256, 257, 0), (257, 257, 0),
    (255, 512, 1), (300, 512, 3), (40, 1025, 0), (700, 1001, 0), (300, 2049, 0), (20, 4099, 0),
    (300, 4099, 0), (260, 8191, 0)])
def test_norms_ragged_rows(op, rows, cols, offset, dtype):
    print(f"\n[gpu-ragged] {op} {rows}x{cols}+{offset} {dtype}", flush=True)
    mod = pair_module(op)
    g = torch.Generator(device="cuda").manual_seed(rows * 1000 + cols)
    rnd = lambda *s: _at(torch.randn(*s, device="cuda", generator=g).to(dtype), offset)
    x, dy, w = rnd(rows, cols), rnd(rows, cols), rnd(cols)
    args, s = [x, w], x.double()
    if op == "layernorm":
        args.append(rnd(cols))
    if op == "fused_add_rms_norm":
        args.insert(1, rnd(rows, cols))
        s = s + args[1].double()
    eps = 1e-5
    y, saved = getattr(mod, op + "_forward_with_saved")(*args, eps)
    grads = getattr(mod, op + "_backward_from_saved")(dy, saved, eps)
    c = s - s.mean(-1, keepdim=True) if op == "layernorm" else s
    rstd = (c.square().mean(-1, keepdim=True) + eps).rsqrt()
    xhat, wd, gd = c * rstd, w.double(), dy.double()
    want = xhat * wd + (args[2].double() if op == "layernorm" else 0)
    _close(y, want, dtype, (xhat * wd).abs() + want.abs() + 1)
    gw = gd * wd
    t = (gw * xhat).mean(-1, keepdim=True)
    m = gw.mean(-1, keepdim=True) if op == "layernorm" else 0
    _close(grads[0], (gw - m - xhat * t) * rstd, dtype, (gw.abs() + xhat.abs() + 1) * rstd)
    n = 2 if op == "fused_add_rms_norm" else 1
    _close(grads[n], (gd * xhat).sum(0), dtype, (gd * xhat).abs().sum(0) + 1)
    if op == "layernorm":
        _close(grads[2], gd.sum(0), dtype, gd.abs().sum(0) + 1)
