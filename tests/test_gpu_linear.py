"""oasis_linear on [K, N] weights: every tile at its edges against fp64."""
import pytest
import torch

from helpers import L, cuda, stream, sync

pytestmark = pytest.mark.gpu


def _linear(x, w, dtype):
    M, N = x.shape[0], w.shape[1]
    out = torch.full((M, N), float("nan"), device="cuda", dtype=dtype)
    L.call("oasis_linear", L.ptr(x), L.ptr(w), L.ptr(out), M, x.shape[1], N, 0,
           L.F32 if dtype == torch.float32 else L.BF16, stream())
    sync()
    return out


# every kernel of the table (the shapes' kernels are checked without a GPU beside the other tile choices); partial
# last tiles on both sides, N below a tile and below a 16-column group, K of one ring stage, of fewer K tiles than
# the ring and of odd counts
SHAPES = [(1, 256, 8), (17, 1024, 1000), (64, 4096, 72), (300, 1024, 1000), (150, 512, 3048), (250, 1024, 3064),
          (243, 4096, 3048), (630, 1024, 1016), (321, 1024, 3064), (1, 64, 8), (5, 64, 64), (500, 320, 3064),
          (70, 128, 200), (640, 1024, 4088), (1030, 1024, 3064), (1057, 960, 3048), (1290, 1024, 3064),
          (1281, 192, 3064), (2561, 1024, 4088), (2500, 64, 4072), (577, 832, 1208), (643, 1024, 3064)]


@pytest.mark.parametrize("M,K,N", SHAPES)
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_linear_kn_tiles(M, K, N, dtype):
    g = torch.Generator().manual_seed(M + N)
    x = cuda(torch.randn(M, K, generator=g), torch.bfloat16)
    w = cuda(torch.randn(K, N, generator=g) * 0.05, torch.bfloat16)
    out = _linear(x, w, dtype).double()
    ref = x.double() @ w.double()
    # fp32 sums of exact bf16 products: K * 2^-24 of sum |x w| at most; a bf16 output adds 2^-9 of itself
    bound = K * 2.0 ** -24 * (x.double().abs() @ w.double().abs())
    if dtype == torch.bfloat16:
        bound = bound + 2.0 ** -8 * ref.abs()
    assert torch.isfinite(out).all() and ((out - ref).abs() <= bound).all()


def test_linear_kn_rows_past_32_bit_offsets():
    """A weight row of 2^24 + 8 columns (64 rows: 2.1 GB) runs on 64-bit addresses."""
    M, K, N = 3, 64, (1 << 24) + 8
    x = torch.randn(M, K, device="cuda").to(torch.bfloat16)
    w = torch.empty(K, N, device="cuda", dtype=torch.bfloat16).normal_()
    out = _linear(x, w, torch.float32)
    for cols in (slice(0, 128), slice(N // 2, N // 2 + 128), slice(N - 128, N)):
        ref = x.double() @ w[:, cols].double()
        assert (out[:, cols].double() - ref).abs().max() <= 1e-4
