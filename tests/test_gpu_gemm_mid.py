"""The 128 x 128 product kernel (small outputs of eg_gemm): tile edges, ragged and padded
operands, residuals and split k against fp64, and its bits against the 256 x 256 kernel's.

Bound: fp32 accumulation of K exact products of 16-bit values (and the residual), so at
most (K + 20) 2^-24 of the sum of the absolute terms, then one rounding of the output."""

import pytest
import torch

from evograd_amd import _lib
from evograd_amd.timing import KernelTimer

pytestmark = pytest.mark.gpu
ULP = {torch.float16: 2.0 ** -11, torch.bfloat16: 2.0 ** -8, torch.float32: 2.0 ** -24}
LAYOUTS = [(True, True), (True, False), (False, True), (False, False)]


def _up(n, m=8):
    return (n + m - 1) // m * m


def _product(a, b, c, r, M, N, K, akc, bkc, dtype, ws_bytes):
    ws = torch.full((max(ws_bytes, 16),), 255, dtype=torch.uint8, device="cuda")
    _lib.call("eg_gemm", a.data_ptr(), b.data_ptr(), c.data_ptr(), _lib.ptr(r), M, N, K,
              a.shape[1], b.shape[1], c.shape[1], r.shape[1] if r is not None else 0, int(akc),
              int(bkc), _lib.dtype_tag(dtype), _lib.dtype_tag(c.dtype), ws.data_ptr(), ws_bytes,
              torch.cuda.current_stream().cuda_stream)


# one tile and less, past a tile in each direction, several k slices with a ragged last
# one (k-major operands), and an output whose depth is split
SHAPES = [(1, 8, 64), (127, 128, 128), (129, 130, 192), (77, 300, 448), (256, 136, 100),
          (64, 72, 4096)]


@pytest.mark.parametrize("M,N,K,akc,bkc", [
    (*shape, *layout) for shape in SHAPES for layout in LAYOUTS
    if shape[2] % 64 == 0 or layout != (True, True)])  # two k-contiguous: K % 64 == 0
@pytest.mark.parametrize("dtype,cdt", [(torch.bfloat16, torch.bfloat16),
                                       (torch.float16, torch.float16),
                                       (torch.bfloat16, torch.float32)])
def test_gemm_mid(M, N, K, akc, bkc, dtype, cdt):
    print(f"\n[gpu-gemm-mid] {M}x{N}x{K} akc={akc} bkc={bkc} {dtype} -> {cdt}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + 7 * N + 31 * K)
    def operand(rows, cols, ld):
        t = torch.zeros(rows, ld, device="cuda", dtype=dtype)
        t[:, :cols] = torch.randn(rows, cols, device="cuda", generator=g).to(dtype)
        return t
    a = operand(M, K, _up(K, 64)) if akc else operand(K, M, _up(M))
    b = operand(N, K, _up(K, 64)) if bkc else operand(K, N, _up(N))
    A = (a[:, :K] if akc else a[:, :M].t()).double()
    B = (b[:, :K].t() if bkc else b[:, :N]).double()
    nbytes = _lib.query("eg_gemm_workspace_bytes", M, N, K, _lib.dtype_tag(dtype))
    for ldc in (_up(N), _up(N) + 3):  # 16-byte and element stores
        for res in (None, torch.randn(M, ldc, device="cuda", generator=g).to(cdt)):
            want, terms = A @ B, A.abs() @ B.abs()
            if res is not None:
                want, terms = want + res[:, :N].double(), terms + res[:, :N].double().abs()
            for ws_bytes in {0, nbytes}:
                c = torch.full((M, ldc), float("nan"), device="cuda", dtype=cdt)
                _product(a, b, c, res, M, N, K, akc, bkc, dtype, ws_bytes)
                bound = terms * (K + 20) * 2.0 ** -24 + want.abs() * ULP[cdt] + 2.0 ** -25
                assert ((c[:, :N].double() - want).abs() <= bound).all()
                assert torch.isnan(c[:, N:]).all()


@pytest.mark.parametrize("akc,bkc", LAYOUTS)
def test_gemm_mid_bits_equal_the_large_tiles(akc, bkc):
    """Rows of an unsplit product do not depend on the kernel that formed them: 33 x 4 tiles
    of 256 x 256 against the same first rows alone, on 128 x 128 tiles."""
    M, N, K, m = 33 * 256, 1024, 192, 200
    print(f"\n[gpu-gemm-mid] bits akc={akc} bkc={bkc}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(5)
    a = torch.randn(*((M, K) if akc else (K, M)), device="cuda", generator=g).bfloat16()
    b = torch.randn(*((N, K) if bkc else (K, N)), device="cuda", generator=g).bfloat16()
    few = a[:m] if akc else a  # a k-major A keeps its row stride
    whole = torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
    part = torch.empty(m, N, device="cuda", dtype=torch.bfloat16)
    _product(a, b, whole, None, M, N, K, akc, bkc, torch.bfloat16, 0)
    _product(few, b, part, None, m, N, K, akc, bkc, torch.bfloat16, 0)
    assert torch.equal(whole[:m], part)


@pytest.mark.parametrize("M,N,K,kernel", [
    (1024, 4096, 4096, "gemm_mid_kernel"), (1024, 4096, 6144, "gemm_kernel"),
    (1280, 640, 22144, "gemm_kernel"),      # 50 small tiles in 5 ranges: 35 on one XCD
    (700, 3001, 9024, "gemm_mid_kernel"),   # 36 large tiles in 7 ranges: likewise
    (640, 1152, 4096, "gemm_mid_kernel")])  # 45 small tiles, split
def test_product_kernel_by_size(M, N, K, kernel):
    """The lines of the choice between the two kernels, and its products against fp64."""
    print(f"\n[gpu-gemm-mid] {M}x{N}x{K} on {kernel}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    a = torch.randn(M, K, device="cuda", generator=g).bfloat16()
    b = torch.randn(N, K, device="cuda", generator=g).bfloat16()
    c = torch.empty(M, N, device="cuda", dtype=torch.float32)
    need = _lib.query("eg_gemm_workspace_bytes", M, N, K, _lib.EG_BF16)
    timer = KernelTimer()
    timer.arm(0)
    _product(a, b, c, None, M, N, K, True, True, torch.bfloat16, need)
    assert timer.label() == kernel
    timer.close()
    A, B = a.double(), b.double().t()
    assert ((c.double() - A @ B).abs() <= (K + 20) * 2.0 ** -24 * (A.abs() @ B.abs())).all()
