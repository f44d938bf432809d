"""The GEMM tiles used above 320 tokens (bf16 18-29, fp8 12-23) on ragged shapes against a tile that
other tests hold to the oracle, and whole sub-blocks at row counts where the tile choice changes."""
import ctypes

import pytest
import torch

from helpers import L, cuda, pkg, stream, sync
from test_gpu_model import _check_sub_block, _single_block_dit

pytestmark = pytest.mark.gpu

# rows: 600 leaves a partial last tile on every tile height, 100-row frames change the gate row and the
# RoPE position inside 16-row groups; K = 640: 10 (fp8: 5) K tiles, not a multiple of any ring's stages
M, P, T, K, H = 600, 100, 3, 640, 4
D = 64 * H


def _operands(fp8):
    g = torch.Generator().manual_seed(5)
    A = cuda(torch.randn(M, K, generator=g), torch.bfloat16)
    W = cuda(torch.randn(3 * D, K, generator=g) * 0.05, torch.bfloat16)
    t = {"bias": cuda(torch.randn(3 * D, generator=g) * 0.1), "x": cuda(torch.randn(M, 3 * D, generator=g)),
         "gate": cuda(torch.randn(M // P, 3 * D, generator=g)), "cos": cuda(torch.randn(P, 64, generator=g)),
         "sin": cuda(torch.randn(P, 64, generator=g)), "A": A, "W": W}
    if fp8:
        u8 = dict(dtype=torch.uint8, device="cuda")
        t.update(q=torch.empty(3 * D, K, **u8), s=torch.empty(3 * D, device="cuda"), a8=torch.empty(M, K, **u8),
                 a8s=torch.empty(M, K // 32, **u8))
        L.call("oasis_quantize_fp8_rows", L.ptr(W), 3 * D, K, L.ptr(t["q"]), L.ptr(t["s"]), stream())
        L.call("oasis_quantize_act_fp8", L.ptr(A), K, M, K, L.ptr(t["a8"]), K, L.ptr(t["a8s"]), K // 32, stream())
    return t


def _run(t, kind, tile, fp8, N, splits=1):
    """One product of N columns (fewer than 3D: a partial last tile column) with the given epilogue."""
    e = L.Epilogue()
    e.rows_per_frame, e.frames_per_stream, e.bias = P, T, t["bias"].data_ptr()
    out = None
    if kind == "qkv":
        out = [torch.zeros(M * D, dtype=torch.bfloat16, device="cuda") for _ in range(3)]
        e.kind, e.n_heads = L.EPI_QKV_ROPE, H
        e.q, e.k, e.v = (o.data_ptr() for o in out)
        e.s_b, e.s_t, e.s_p, e.s_h = P * H * T * 64, 64, H * T * 64, T * 64
        e.rope_cos, e.rope_sinp, e.rope_by_frame = t["cos"].data_ptr(), t["sin"].data_ptr(), 1
    elif kind == "gelu" and fp8:
        out = [torch.zeros(M, N, dtype=torch.uint8, device="cuda"), torch.zeros(M, N // 32, dtype=torch.uint8, device="cuda")]
        e.kind, e.out_fp8, e.out_scale, e.ld_out, e.ld_scale = (L.EPI_GELU_TANH_FP8, out[0].data_ptr(),
                                                               out[1].data_ptr(), N, N // 32)
    elif kind in ("gelu", "erf"):
        out = [torch.zeros(M, N, dtype=torch.bfloat16, device="cuda")]
        e.kind, e.out_bf16, e.ld_out = L.EPI_GELU_TANH if kind == "gelu" else L.EPI_GELU_ERF, out[0].data_ptr(), N
    elif kind == "part":
        out = [torch.zeros(splits, M, N, device="cuda")]
        e.kind, e.out_f32, e.ld_out, e.split_stride = L.EPI_PARTIAL_F32, out[0].data_ptr(), N, M * N
    else:
        out = [t["x"][:, :N].contiguous()]
        e.kind = {"gated": L.EPI_GATED_RES, "res": L.EPI_RESIDUAL, "store": L.EPI_STORE_F32}[kind]
        e.out_f32, e.ld_out, e.gate, e.gate_fstride = out[0].data_ptr(), N, t["gate"].data_ptr(), 3 * D
    if fp8:
        L.call("oasis_gemm_fp8_a8", L.ptr(t["a8"]), K, L.ptr(t["a8s"]), K // 32, L.ptr(t["q"]), K, L.ptr(t["s"]), M, N,
               K, ctypes.byref(e), tile, splits, stream())
    else:
        L.call("oasis_gemm_bf16_config", L.ptr(t["A"]), K, L.ptr(t["W"]), K, M, N, K, ctypes.byref(e), tile, splits,
               stream())
    sync()
    return out


@pytest.mark.parametrize("tile", list(range(18, 30)))
def test_bf16_tiles_equal_the_96x64_tile(tile):
    """Every epilogue, bit for bit: all these tiles add the K steps of an output in the same order. The
    GELUs may differ in the last bf16 place where a tile reads its epilogue kind at run time."""
    t = _operands(False)
    for kind, N, splits in (("store", 520, 1), ("gelu", 520, 1), ("erf", 520, 1), ("part", 520, 1), ("part", 520, 5),
                            ("gated", 520, 1), ("res", 520, 1), ("qkv", 3 * D, 1)):
        for a, b in zip(_run(t, kind, tile, False, N, splits), _run(t, kind, 2, False, N, splits)):
            assert torch.equal(a, b), (tile, kind, splits, (a.float() - b.float()).abs().max().item())


@pytest.mark.parametrize("tile", list(range(12, 24)))
def test_fp8_tiles_equal_the_4_wave_tile(tile):
    t = _operands(True)
    for kind, N, splits in (("store", 520, 1), ("gelu", 544, 1), ("part", 520, 1), ("part", 520, 5), ("gated", 520, 1),
                            ("res", 520, 1), ("qkv", 3 * D, 1)):
        if kind == "gelu" and tile == 22:   # 48-column wave tiles: lanes do not cover 32-column blocks
            with pytest.raises(L.OasisError, match="GELU_TANH_FP8"):
                _run(t, kind, tile, True, N)
            continue
        for a, b in zip(_run(t, kind, tile, True, N, splits), _run(t, kind, 0, True, N, splits)):
            assert torch.equal(a, b), (tile, kind, splits)


@pytest.mark.parametrize("kind,T", [("s", 3), ("t", 5), ("s", 7), ("t", 8), ("t", 10), ("s", 24), ("t", 28)])
def test_sub_blocks_across_tile_choices(kind, T):
    """Sub-blocks from 432 tokens up: split-K partials (below 1024 tokens), then O and FC2 unsplit with the
    residual in their epilogue, on the tiles the costs pick."""
    dr = pkg.synth.Draw(170 + T)
    x, cond = dr.normal(T, 144, 1024), dr.normal(T, 1024)
    w = _single_block_dit(pkg.synth.config0()["w"], kind, spatial_freqs=pkg.synth.theta_freqs(16, 32),
                          temporal_freqs=pkg.synth.theta_freqs(32, 64))
    _check_sub_block(x, cond, w, kind, T, "%s sub-block T=%d" % (kind, T))
