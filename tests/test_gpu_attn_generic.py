"""The generic attention kernels (fp32 MFMA): every dtype and head size off the 16-bit
MFMA path, against the declared gate at the edges of their 16-row tiles.

Row counts: below, at and past one 16-row tile, a ragged 32-key tile, and enough key
blocks for the cut dK/dV walk; head sizes: each register layout (16, 32, 64, 128) full,
partly filled in whole 4-column loads, and not a multiple of 4 (element loads).
"""

import pytest
import torch

from evograd_amd import decls, pair_module
from evograd_amd.inputs import make_case_inputs
from evograd_amd.opdecl import Workload
from oracle.verify import verify

pytestmark = pytest.mark.gpu
OP = decls.CAUSAL_ATTENTION_GQA


@pytest.mark.parametrize("dtype", ("float32", "bfloat16", "float16"))
@pytest.mark.parametrize("B,H,KVH,S,D", (
    (1, 1, 1, 1, 16), (1, 2, 1, 15, 32), (2, 2, 2, 16, 48), (1, 4, 2, 17, 10),
    (1, 4, 1, 33, 80), (2, 2, 1, 130, 70), (1, 8, 2, 257, 32), (1, 2, 2, 64, 126),
))
def test_generic_attention_edges(B, H, KVH, S, D, dtype):
    w = Workload(dims=dict(B=B, H=H, KVH=KVH, S=S, D=D), dtype=dtype)
    print("\n[gpu-attn-generic]", w.dims, dtype, flush=True)
    rep = verify(OP, pair_module("causal_attention_gqa"), device="cuda", workloads=(w,))
    assert rep.ok, "\n".join(rep.failures())


# 40 heads of 130 rows: a grid resident at once, whose second half runs shortest first.
@pytest.mark.parametrize("H,KVH,S", ((4, 2, 200), (40, 10, 130)))
@pytest.mark.parametrize("D", (64, 128))
def test_generic_attention_fp32_wide_heads(D, H, KVH, S):
    w = Workload(dims=dict(B=1, H=H, KVH=KVH, S=S, D=D), dtype="float32")
    print("\n[gpu-attn-generic]", w.dims, flush=True)
    rep = verify(OP, pair_module("causal_attention_gqa"), device="cuda", workloads=(w,))
    assert rep.ok, "\n".join(rep.failures())


@pytest.mark.parametrize("bad", (float("nan"), float("inf")))
@pytest.mark.parametrize("cut", (5, 16, 40))
@pytest.mark.parametrize("D", (16, 32, 64, 126))
def test_generic_attention_masked_rows_do_not_leak(D, cut, bad):
    """A non-finite row reaches only the outputs that causality lets it reach: bad keys and
    values leave earlier queries alone, bad queries and do leave later keys alone. One head
    size of each register layout."""
    mod = pair_module("causal_attention_gqa")
    w = Workload(dims=dict(B=1, H=2, KVH=1, S=50, D=D), dtype="float32")
    inp = make_case_inputs(OP, w, "cuda")
    print("\n[gpu-attn-generic] non-finite rows", D, cut, bad, flush=True)

    def step(q, k, v, do):
        o, saved = mod.causal_attention_gqa_forward_with_saved(q, k, v)
        return (o, *mod.causal_attention_gqa_backward_from_saved(do, saved))

    names = ("q", "k", "v", "do")
    clean = step(*(inp[n] for n in names))
    late = {n: inp[n].clone() for n in names}
    for n in names:
        late[n][:, :, cut:] = bad
    got = step(*(late[n] for n in names))
    for x, y in zip(got[:2], clean[:2]):  # o, dq of the rows before
        torch.testing.assert_close(x[:, :, :cut], y[:, :, :cut], atol=1e-5, rtol=1e-5)
    early = {n: inp[n].clone() for n in names}
    for n in ("q", "do"):
        early[n][:, :, :cut] = bad
    got = step(*(early[n] for n in names))
    for x, y in zip(got[2:], clean[2:]):  # dk, dv of the keys after: no query before sees them
        torch.testing.assert_close(x[:, :, cut:], y[:, :, cut:], atol=1e-5, rtol=1e-5)
    for x, y in zip(got[:2], clean[:2]):
        torch.testing.assert_close(x[:, :, cut:], y[:, :, cut:], atol=1e-5, rtol=1e-5)
