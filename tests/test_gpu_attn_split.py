"""Attention on grids too small for the chip: two key groups per workgroup (768 positions
and more on few heads) and the chosen cut of the dK/dV walk, under the declared gate.

Sizes: the first length that splits the keys and the last that does not, an odd number of
64-key tiles, a last tile of one key, a last row block whose second group has no tile for
some waves, grouped heads, the rotated pair, and walks cut into 1, 2, 3 and 8 parts."""

import pytest
import torch

from evograd_amd import decls, pair_module
from evograd_amd.opdecl import Workload
from oracle.verify import verify

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", ("bfloat16", "float16"))
@pytest.mark.parametrize("B,H,KVH,S,D", [
    (1, 2, 2, 767, 64), (1, 2, 1, 768, 128), (1, 3, 3, 833, 64), (2, 4, 2, 1000, 128),
    (1, 2, 2, 1025, 128), (4, 8, 8, 300, 64), (2, 12, 12, 260, 64), (1, 4, 1, 1300, 64)])
def test_attention_split(B, H, KVH, S, D, dtype):
    w = Workload(dims=dict(B=B, H=H, KVH=KVH, S=S, D=D), dtype=dtype)
    print("\n[gpu-attn-split]", w.dims, dtype, flush=True)
    for op in (decls.CAUSAL_ATTENTION_GQA, decls.LLAMA3_ATTENTION):
        rep = verify(op, pair_module(op.name), device="cuda", workloads=(w,))
        assert rep.ok, "\n".join(rep.failures())


def test_attention_split_is_bitwise_repeatable():
    g = torch.Generator(device="cuda").manual_seed(3)
    rnd = lambda h: torch.randn(1, h, 1100, 128, device="cuda", generator=g).bfloat16()
    q, k, v, do = rnd(4), rnd(2), rnd(2), rnd(4)
    mod = pair_module("causal_attention_gqa")
    runs = []
    for _ in range(2):
        o, saved = mod.causal_attention_gqa_forward_with_saved(q, k, v)
        runs.append((o, *mod.causal_attention_gqa_backward_from_saved(do, saved)))
    assert all(torch.equal(a, b) for a, b in zip(*runs))
