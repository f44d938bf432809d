"""Projections of many conditioning rows (a long window, several streams, a video batch): the row-batched
kernels behind oasis_gemv_bf16_tiled and oasis_gemv_f32 against fp64, at the edges of their row groups,
passes and tiles."""
import pytest
import torch

from helpers import L, cuda, pkg, stream, sync

pytestmark = pytest.mark.gpu


def _silu(x):
    return x * torch.sigmoid(x)


@pytest.mark.parametrize("R,N,K,off,act_in,act_out,acc", [(9, 8192, 64, 0, 1, 0, 0), (17, 8208, 320, 0, 0, 1, 0),
                                                          (33, 9216, 1024, 0, 1, 0, 1), (80, 8224, 1024, 0, 1, 0, 0),
                                                          (96, 8400, 192, 1, 1, 0, 0), (97, 8400, 448, 0, 1, 1, 1),
                                                          (200, 8192, 2048, 3, 0, 0, 0), (40, 8176, 128, 0, 1, 0, 0),
                                                          (33, 8192, 64, 0, 1, 0, 0), (12, 8192, 1024, 2, 1, 0, 1),
                                                          (9, 24592, 1024, 0, 1, 0, 0), (11, 8192, 2048, 0, 0, 1, 0)])
def test_tiled_rows(R, N, K, off, act_in, act_out, acc):
    """off: x rows that start `off` floats past a 16-byte boundary. N = 8176 and 9 rows of K = 64 are below the
    kernel's range, the last four shapes its fewest rows. The row-major kernel gives the same bits."""
    g = torch.Generator().manual_seed(R + N)
    W = (torch.randn(N, K, generator=g) * 0.05).to(torch.bfloat16)
    x, b, o0 = torch.randn(R, K, generator=g) * 2, torch.randn(N, generator=g), torch.randn(R, N + 4, generator=g)
    xd = torch.zeros(R, K + 8, device="cuda")
    xd[:, off:off + K] = x.cuda()
    out, Wt, bd = cuda(o0), cuda(pkg.model.tile_rows16(W)), cuda(b)
    L.call("oasis_gemv_bf16_tiled", L.ptr(xd[:, off:]), K + 8, R, L.ptr(Wt), N, K, L.ptr(bd), L.ptr(out), N + 4,
           act_in, act_out, acc, stream())
    sync()
    y = (_silu(x.double()) if act_in else x.double()) @ W.double().t() + b.double()
    y = _silu(y) if act_out else y
    y = y + o0[:, :N].double() if acc else y
    # x as hi + lo bf16 keeps 2^-17 of each value, fp32 sums: 1e-5 of the row's scale
    assert (out[:, :N].cpu().double() - y).norm() <= 1e-5 * y.norm()
    assert torch.equal(out[:, N:].cpu(), o0[:, N:])
    rm, Wr = cuda(o0), cuda(W)
    L.call("oasis_gemv_bf16", L.ptr(xd[:, off:]), K + 8, R, L.ptr(Wr), N, K, L.ptr(bd), L.ptr(rm), N + 4, act_in,
           act_out, acc, stream())
    sync()
    assert torch.equal(rm, out)


@pytest.mark.parametrize("R,N,K,act_in,act_out,acc", [(9, 16, 16, 0, 0, 0), (32, 48, 1088, 0, 1, 0),
                                                      (33, 2048, 1024, 1, 0, 1), (80, 1024, 1088, 0, 0, 0),
                                                      (40, 1000, 256, 1, 0, 0), (17, 40, 260, 0, 0, 0),
                                                      (70, 64, 256, 2, 1, 0)])
def test_f32_rows(R, N, K, act_in, act_out, acc):
    """More than 8 rows: the MFMA kernel, and (N or K without whole 16-tiles, the timestep embedding) the
    vector kernel with every row group in one launch."""
    g = torch.Generator().manual_seed(R + K)
    W, b, o0 = torch.randn(N, K, generator=g) * 0.05, torch.randn(N, generator=g), torch.randn(R, N, generator=g)
    if act_in == 2:
        x = torch.randint(0, 1000, (R, 1), generator=g).float()
        f = torch.exp(-torch.log(torch.tensor(10000.0, dtype=torch.float64)) * torch.arange(K // 2) / (K // 2))
        xe = torch.cat([torch.cos(x.double() * f), torch.sin(x.double() * f)], 1)
    else:
        x = torch.randn(R, K, generator=g) * 2
        xe = _silu(x.double()) if act_in else x.double()
    out, xd, Wd, bd = cuda(o0), cuda(x), cuda(W), cuda(b)
    L.call("oasis_gemv_f32", L.ptr(xd), x.shape[1], R, L.ptr(Wd), N, K, L.ptr(bd), L.ptr(out), N, act_in, act_out, acc,
           stream())
    sync()
    y = xe @ W.double().t() + b.double()
    y = _silu(y) if act_out else y
    y = y + o0.double() if acc else y
    # fp32 products and sums over K terms; the embedding's fp32 angles (t up to 1000) are good to ~3e-5
    assert (out.cpu().double() - y).norm() <= (1e-4 if act_in == 2 else 2e-6) * y.norm()


@pytest.mark.parametrize("R", [8, 9])
@pytest.mark.parametrize("x", [-80.0, -87.0, -87.5, -88.0, -88.5])
def test_f32_rows_of_tiny_silu(R, x):
    """1 + exp(-x) from 2^126 up: its reciprocal is no normal number, x over it still is."""
    xd, W, out = torch.full((R, 64), x, device="cuda"), torch.full((64, 64), 2.0 ** 100, device="cuda"), torch.zeros(R, 64, device="cuda")
    L.call("oasis_gemv_f32", L.ptr(xd), 64, R, L.ptr(W), 64, 64, None, L.ptr(out), 64, 1, 0, 0, stream())
    sync()
    ref = 64 * 2.0 ** 100 * _silu(torch.tensor(x, dtype=torch.float64)).item()
    # the fp32 exponent -x log2(e) = 127 holds 2^-18: 3e-6 of the exponential
    assert ((out.double() - ref).abs() <= 1e-5 * abs(ref)).all()


@pytest.mark.parametrize("R", [9, 41, 96, 97])
def test_conditioning_rows_do_not_depend_on_the_batch(R):
    """The rows of one conditioning call (the MFMA kernels, [hid | action] side by side, and the adaLN rows kernel
    from its fewest rows to a second pass) against the same rows 8 at a time (the step's kernels): fp32 sums in
    another order."""
    dr = pkg.synth.Draw(3)
    # 4 sub-blocks of D = 1024: 24576 stacked adaLN outputs
    w = pkg.synth.dit_weights(dr, n_blocks=2, d=1024, n_heads=16, d_mlp=1024)
    dit = pkg.DiT(w, "cuda")
    ws = dit.workspace(144, max_cond=112)
    t, a = dr.randint(0, 1000, (R,)).float().cuda(), pkg.synth.one_hot_actions(dr, R).cuda()
    many = dit.conditioning(t, a, ws).clone()
    few = torch.cat([dit.conditioning(t[i:i + 8], a[i:i + 8], ws).clone() for i in range(0, R, 8)])
    sync()
    assert (many - few).abs().max() <= 2e-5 * few.abs().max()
