"""Attention on grids too small for the chip: two key groups per workgroup (768 positions
and more on few heads) and the chosen cut of the dK/dV walk, under the declared gate.

Sizes: the first length that splits the keys and the last that does not, an odd number of
64-key tiles, a last tile of one key, a last row block whose second group has no tile for
some waves, grouped heads, the rotated pair, and walks cut into 1 to 8 parts, as many as
the workspace query says."""

import pytest
import torch

from evograd_amd import _lib, decls, pair_module
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


# Few query tiles a part, with ranges that come out uneven; the last ones the longest walks.
PARTS = [(2, 32, 16, 200, 128, 3), (1, 12, 12, 300, 128, 4), (2, 8, 8, 333, 64, 4),
         (3, 2, 2, 333, 128, 5), (1, 24, 12, 200, 128, 6), (1, 8, 8, 300, 64, 6),
         (1, 6, 6, 333, 64, 7), (1, 4, 4, 300, 128, 7), (1, 4, 2, 129, 64, 8),
         (2, 12, 12, 1000, 64, 3), (1, 32, 32, 1300, 128, 2)]


@pytest.mark.parametrize("dtype", ("bfloat16", "float16"))
@pytest.mark.parametrize("B,H,KVH,S,D,parts", PARTS)
def test_attention_walk_cut_into_parts(B, H, KVH, S, D, parts, dtype):
    """Every number of parts, under the gate, and inside the workspace that is asked for."""
    print("\n[gpu-attn-split] parts", (B, H, KVH, S, D, parts), dtype, flush=True)
    need = _lib.query("eg_attn_gqa_workspace_bytes", B, H, KVH, S, D)
    delta = (B * H * S * 4 + 255) // 256 * 256
    assert need == delta + 2 * parts * B * KVH * S * D * 4
    w = Workload(dims=dict(B=B, H=H, KVH=KVH, S=S, D=D), dtype=dtype)
    for op in (decls.CAUSAL_ATTENTION_GQA, decls.LLAMA3_ATTENTION):
        rep = verify(op, pair_module(op.name), device="cuda", workloads=(w,))
        assert rep.ok, "\n".join(rep.failures())
    # the slabs again with a marked end: the first part's start and the last one's end are
    # written, nothing past them is
    T = getattr(torch, dtype)
    q, k, v, do = (torch.randn(B, h, S, D, device="cuda").to(T) for h in (H, KVH, KVH, H))
    o, saved = pair_module("causal_attention_gqa").causal_attention_gqa_forward_with_saved(q, k, v)
    lse = next(t for t in saved if t.dtype == torch.float32 and t.numel() == B * H * S)
    ws = torch.full((need + 4096,), 0xA5, dtype=torch.uint8, device="cuda")
    dq, dk, dv = torch.empty_like(q), torch.empty_like(k), torch.empty_like(v)
    _lib.call("eg_attn_gqa_bwd", *(t.data_ptr() for t in (do, q, k, v, o, lse, dq, dk, dv, ws)),
              B, H, KVH, S, D, D ** -0.5, _lib.dtype_tag(T), _lib.stream_of(q))
    assert (ws[need:] == 0xA5).all()
    assert (ws[need - 4 * D:need].view(torch.int32) != 0xA5A5A5A5 - (1 << 32)).any()


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


# On both sides of the lines for grids past 256 workgroups: dQ at 1152 positions (head size
# 64) and 2048 (128), the forward at 2048 (128).
@pytest.mark.parametrize("B,H,KVH,S,D", [(1, 40, 8, 1151, 64), (1, 40, 8, 1152, 64),
                                         (3, 16, 16, 900, 64), (1, 24, 8, 2047, 128),
                                         (1, 24, 8, 2048, 128)])
def test_attention_split_keys_lines(B, H, KVH, S, D):
    test_attention_split(B, H, KVH, S, D, "bfloat16")
