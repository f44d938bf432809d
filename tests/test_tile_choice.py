"""The default GEMM tiles, by the library's own query (no kernel runs here): at shapes inside and outside the ones
that the DiT runs, the tile picked is among those measured within 12 % of the fastest of all."""
import pytest

from helpers import L
from test_gpu_linear import SHAPES as LINEAR_SHAPES

# (epilogue, M, N, K, tiles within 12 % of the fastest), MI355X, weights not in cache
BF16 = [
    ("store", 1000, 64, 64, {0, 1}), ("store", 321, 64, 64, {0, 1}), ("store", 321, 1024, 256, {0, 9}),
    ("store", 576, 3072, 256, {1, 3}), ("store", 1440, 2048, 768, {2, 23}), ("store", 9216, 512, 128, {18, 24}),
    ("gelu", 576, 4096, 256, {2, 4, 23, 24, 25}), ("gelu", 1440, 4096, 1024, {20, 24, 28}),
    ("gelu", 9216, 4096, 1024, {5, 19, 27}), ("res", 864, 2048, 128, {1, 3, 4}), ("res", 1152, 1024, 768, {1, 2, 3}),
    ("res", 1440, 1024, 1024, {1, 2, 3}), ("qkv", 432, 1536, 512, {0, 1, 9, 10}), ("qkv", 1440, 3072, 1024, {18, 24}),
    ("qkv", 4608, 3072, 1024, {26}), ("res", 9216, 3072, 1024, {5, 6, 7, 21, 22, 24, 27}),
    ("res", 4608, 3072, 1024, {5, 6, 27, 28}), ("res", 2000, 1024, 4096, {3, 4}), ("qkv", 720, 1536, 512, {1, 2, 3, 9}),
]
FP8 = [
    ("store", 1, 64, 128, {4, 12}), ("store", 144, 4096, 256, {4, 12}), ("store", 288, 1024, 128, {4}),
    ("store", 1000, 3072, 4096, {0, 2, 3, 10, 17}), ("store", 2304, 512, 128, {3, 4, 13, 19}),
    ("store", 9216, 3072, 128, {7, 18, 20, 21, 22}), ("gelu8", 576, 4096, 256, {3, 4, 13, 14, 16, 19}),
    ("gelu8", 1440, 4096, 1024, {17}), ("gelu8", 9216, 4096, 1024, {5, 21}), ("qkv", 144, 768, 256, {4}),
    ("qkv", 1440, 768, 256, {4, 19}), ("qkv", 432, 3072, 1024, {3, 4, 12, 13, 16, 19}),
    ("qkv", 9216, 3072, 1024, {18, 22}), ("res", 1440, 1024, 1024, {3, 4, 12, 13, 16, 19}),
    # the tiles whose gated residual spills registers (21, 22) take 1.4 to 1.6 times as long
    ("res", 9216, 3072, 1024, {5, 6, 7, 18, 20, 23}), ("res", 4608, 3072, 1024, {5, 6, 23}),
    ("res", 9216, 1536, 512, {5, 6, 7, 18, 20, 23}), ("res", 2000, 1024, 4096, {2, 3}), ("store", 720, 1024, 4096, {3}),
]
KIND = {"store": L.EPI_STORE_BF16, "gelu": L.EPI_GELU_TANH, "gelu8": L.EPI_GELU_TANH_FP8, "res": L.EPI_GATED_RES,
        "qkv": L.EPI_QKV_ROPE}


@pytest.mark.parametrize("fp8,kind,M,N,K,good", [(0,) + c for c in BF16] + [(1,) + c for c in FP8])
def test_default_tile_is_among_the_fastest(fp8, kind, M, N, K, good):
    assert L.lib().oasis_gemm_tile(M, N, K, KIND[kind], 1, fp8) in good


@pytest.mark.parametrize("args,code", [((0, 64, 64, 0, 1, 0), -2), ((64, 64, 96, 0, 1, 0), -2), ((64, 64, 64, 0, 1, 1), -2),
                                       ((64, 64, 128, 0, 3, 0), -2), ((64, 64, 128, 0, 0, 0), -2),
                                       ((64, 64, 128, 12, 1, 0), -5), ((64, 64, 128, -1, 1, 0), -5)])
def test_tile_query_errors(args, code):
    assert L.lib().oasis_gemm_tile(*args) == code


def test_linear_shapes_reach_every_kernel():
    """The [K, N] linear layer's GPU test runs each kernel of its table, on at least one shape with partial last
    tiles of rows and of columns."""
    tile = L.lib().oasis_linear_tile
    assert {tile(*s) for s in LINEAR_SHAPES} == set(range(8))
    assert {tile(M, K, N) for M, K, N in LINEAR_SHAPES if M % 16 and N % 64} == set(range(8))
    assert tile(3, 64, (1 << 24) + 8) == tile(3, 1 << 23, 64) == 8
    assert tile(0, 64, 64) == tile(1, 96, 64) == tile(1, 64, 60) == -2
