"""The norm kernels on rows that are no multiple of a 16-byte pack or start unaligned, and
both programs of the backward entry points: one launch up to 256 rows, the ring above.

Widths: one pack and its neighbours, and one past each workgroup width's whole packs.
References in fp64. A 16-bit result is one rounding of fp32 arithmetic on exact inputs; the
fp32 bound is the declarations' 1e-5, relative to the row's or column's scale."""

import pytest
import torch

from evograd_amd import _lib, pair_module

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


@pytest.mark.parametrize("dtype", (torch.float32, torch.float16, torch.bfloat16))
@pytest.mark.parametrize("op", ("rmsnorm", "layernorm", "fused_add_rms_norm"))
@pytest.mark.parametrize("rows,cols", [(256, 3), (256, 257), (256, 512), (257, 512)])
def test_norm_column_sums_of_infinities(op, rows, cols, dtype):
    """An infinity or NaN in dy makes its own column's sums what a plain sum makes them,
    and no other column's, in both programs of the backward (the fp64 reference's sums)."""
    print(f"\n[gpu-ragged] infinities {op} {rows}x{cols} {dtype}", flush=True)
    mod = pair_module(op)
    g = torch.Generator(device="cuda").manual_seed(rows + cols)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).to(dtype)
    x, dy, w = rnd(rows, cols), rnd(rows, cols), rnd(cols)
    bad = [(3, 0, float("inf")), (70, cols - 1, float("-inf")), (200, 1, float("nan"))]
    if cols > 8:  # both signs in one column; an infinity in the last row and in every row
        bad += [(5, 4, float("inf")), (69, 4, float("inf")), (rows - 1, 6, float("-inf"))]
        bad += [(r, 7, float("inf")) for r in range(rows)]
    for r, c, v in bad:
        dy[r, c] = v
    if op == "layernorm" and dtype == torch.float32 and cols > 8:
        dy[1, 8] = dy[65, 8] = 3e38  # a sum that overflows
    args, s = [x, w], x.double()
    if op == "layernorm":
        args.append(rnd(cols))
    if op == "fused_add_rms_norm":
        args.insert(1, rnd(rows, cols))
        s = s + args[1].double()
    _, saved = getattr(mod, op + "_forward_with_saved")(*args, 1e-5)
    grads = getattr(mod, op + "_backward_from_saved")(dy, saved, 1e-5)
    c = s - s.mean(-1, keepdim=True) if op == "layernorm" else s
    xhat, gd = c * (c.square().mean(-1, keepdim=True) + 1e-5).rsqrt(), dy.double()
    sums = [(grads[2 if op == "fused_add_rms_norm" else 1], gd * xhat)]
    if op == "layernorm":
        sums.append((grads[2], gd))
    for got, terms in sums:
        want = terms.sum(0)
        if want.numel() > 8:  # the overflowing column of dweight depends on the order
            got, want, terms = (torch.cat((t[..., :8], t[..., 9:]), -1) for t in (got, want, terms))
        special = ~torch.isfinite(want)
        assert special.any()
        for kind in (torch.isnan, torch.isposinf, torch.isneginf):
            assert torch.equal(kind(got[special]), kind(want[special]))
        _close(got[~special], want[~special], dtype, terms.abs().sum(0)[~special] + 1)
    if op == "layernorm" and dtype == torch.float32 and cols > 8:
        assert torch.isposinf(grads[2][8])


@pytest.mark.parametrize("op", ("rmsnorm", "layernorm", "fused_add_rms_norm"))
@pytest.mark.parametrize("at", ("dx on dy", "dx on x", "dweight on weight"))
def test_norm_backward_in_place(op, at):
    """Outputs laid over inputs that the ring has read by then give what separate buffers
    give (two bf16 roundings of close fp32 sums) at a row count of the one launch, whose
    workgroups would read what others wrote."""
    print(f"\n[gpu-ragged] in place {op} {at}", flush=True)
    rows, cols = 200, 4096
    g = torch.Generator(device="cuda").manual_seed(9)
    rnd = lambda *s: torch.randn(*s, device="cuda", generator=g).bfloat16()
    entry = {"rmsnorm": "eg_rmsnorm_bwd", "layernorm": "eg_layernorm_bwd",
             "fused_add_rms_norm": "eg_fused_add_rmsnorm_bwd"}[op]
    dy, x, r, w = rnd(rows, cols), rnd(rows, cols), rnd(rows, cols), rnd(cols)
    stats = torch.rand(2, rows, device="cuda", generator=g) + 0.5
    ws = torch.empty(_lib.query("eg_layernorm_workspace_bytes", rows, cols), dtype=torch.uint8,
                     device="cuda")

    def run(alias):
        t = dict(dy=dy.clone(), x=x.clone(), w=w.clone())
        o = dict(dx=torch.empty_like(x), dw=torch.empty_like(w), db=torch.empty_like(w))
        if alias:
            o[{"dx": "dx", "dweight": "dw"}[at.split()[0]]] = t[at.split()[2].replace("weight", "w")]
        args = [t["dy"], t["x"]] + ([r] if op == "fused_add_rms_norm" else []) + [t["w"]]
        args += [stats[0], stats[1]] if op == "layernorm" else [stats[1]]
        args += [o["dx"], o["dw"]] + ([o["db"]] if op == "layernorm" else []) + [ws]
        _lib.call(entry, *(a.data_ptr() for a in args), rows, cols, _lib.EG_BF16,
                  _lib.stream_of(x))
        return [o["dx"], o["dw"]] + ([o["db"]] if op == "layernorm" else [])

    for got, want in zip(run(True), run(False)):
        torch.testing.assert_close(got, want, rtol=2.0 ** -7, atol=1e-4)


@pytest.mark.parametrize("op,rows,cols,dtype", [
    ("rmsnorm", 32, 12296, torch.bfloat16), ("rmsnorm", 33, 12296, torch.bfloat16),
    ("rmsnorm", 4, 16384, torch.float16), ("fused_add_rms_norm", 225, 6148, torch.float32),
    ("fused_add_rms_norm", 224, 8192, torch.float32), ("layernorm", 3, 16384, torch.bfloat16)])
def test_norms_wide_rows_on_either_program(op, rows, cols, dtype):
    """Both sides of the lines between the two backward programs at 1537-2048 packs."""
    test_norms_ragged_rows(op, rows, cols, 0, dtype)
