"""The fp32 products (eg_gemm on fp32 operands) at the edges of their three tilings, with
and without 16-byte loads, a residual, and k split over the caller's workspace.

Bound: each entry is K fp32 products summed in fp32 in some order (plus the residual and,
split, a sum of at most 8 partials), so its error is at most (K + 10) 2^-24 of the sum of
the absolute terms."""

import pytest
import torch

from evograd_amd import _lib

pytestmark = pytest.mark.gpu

# 32 x 32 tiles (a single one, ragged, k split), 64 x 64 (256 tiles), 128 x 128 (256 tiles)
SHAPES = [(1, 1, 1), (31, 33, 17), (32, 64, 32), (33, 70, 300), (64, 40, 1001), (1000, 1020, 33),
          (1030, 1000, 64), (2050, 2000, 20)]


@pytest.mark.parametrize("pad", (0, 1))  # pad 1: odd strides, element loads and stores
@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_gemm_f32(M, N, K, akc, bkc, pad):
    print(f"\n[gpu-gemm-f32] {M}x{N}x{K} akc={akc} bkc={bkc} pad={pad}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + 7 * N + 31 * K)
    up = lambda n: (n + 3) // 4 * 4 + pad
    def operand(rows, cols):  # what lies past a row's columns must not be read into the sums
        t = torch.full((rows, up(cols)), float("nan"), device="cuda")
        t[:, :cols] = torch.randn(rows, cols, device="cuda", generator=g)
        return t
    a = operand(M, K) if akc else operand(K, M)
    b = operand(N, K) if bkc else operand(K, N)
    r = operand(M, N)
    A = (a[:, :K] if akc else a[:, :M].t()).double()
    B = (b[:, :K].t() if bkc else b[:, :N]).double()
    want = A @ B + r[:, :N].double()
    bound = (A.abs() @ B.abs() + r[:, :N].double().abs()) * (K + 10) * 2.0 ** -24
    nbytes = _lib.query("eg_gemm_workspace_bytes", M, N, K, _lib.EG_F32)
    for ws_bytes in {0, nbytes}:
        c = torch.full((M, up(N)), float("nan"), device="cuda")
        ws = torch.full((max(ws_bytes, 16),), 255, dtype=torch.uint8, device="cuda")
        _lib.call("eg_gemm", a.data_ptr(), b.data_ptr(), c.data_ptr(), r.data_ptr(), M, N, K,
                  a.shape[1], b.shape[1], c.shape[1], r.shape[1], int(akc), int(bkc), _lib.EG_F32,
                  _lib.EG_F32, ws.data_ptr(), ws_bytes, torch.cuda.current_stream().cuda_stream)
        assert ((c[:, :N].double() - want).abs() <= bound).all()
        assert torch.isnan(c[:, N:]).all()


def test_gemm_f32_splits_small_outputs_only():
    q = lambda m, n, k: _lib.query("eg_gemm_workspace_bytes", m, n, k, _lib.EG_F32)
    assert q(64, 40, 1001) == 4 * 64 * 40 * 4      # 4 tiles, 32 k steps: 4 splits
    assert q(33, 70, 100) == 0                     # 4 k steps
    assert q(512, 512, 4096) == 0                  # 256 tiles of 32


# Each tiling where neither operand comes in whole aligned pieces: the last block of k alone,
# after others, one element past them; outputs narrower than a load.
@pytest.mark.parametrize("pad", (0, 1))
@pytest.mark.parametrize("akc,bkc", [(True, True), (True, False), (False, True), (False, False)])
@pytest.mark.parametrize("M,N,K", [(70, 35, 31), (70, 35, 65), (3, 2, 1025), (2, 3000, 50),
                                   (1001, 1026, 31), (1001, 1026, 97), (2050, 2003, 15),
                                   (2050, 2003, 49), (9000, 511, 33)])
def test_gemm_f32_ragged(M, N, K, akc, bkc, pad):
    test_gemm_f32(M, N, K, akc, bkc, pad)
