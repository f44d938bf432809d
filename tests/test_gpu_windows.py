"""Temporal attention windows of 3 to 32 frames: tile edges, ragged last tiles and non-finite rows against fp64."""
import pytest
import torch

from helpers import L, cuda, stream, sync

pytestmark = pytest.mark.gpu


def _run(q, k, v):
    B, P, H, T, _ = q.shape
    out = torch.full((B * T * P, H * 64), float("nan"), device="cuda", dtype=torch.bfloat16)
    L.call("oasis_temporal_attention", L.ptr(q), L.ptr(k), L.ptr(v), L.ptr(out), B, T, P, H, 0.125, stream())
    sync()
    return out.view(B, T, P, H, 64).permute(0, 2, 3, 1, 4)


def _inputs(B, P, H, T):
    g = torch.Generator().manual_seed(B * 1000 + P * 10 + T)
    return [cuda(torch.randn(B, P, H, T, 64, generator=g) * 2, torch.bfloat16) for _ in range(3)]


# every window length; 5 x 7 x 3 = 105 groups leave the last tile, the last wave and the last block partly empty.
# Above 3072 tiles a workgroup takes four of them: 6201 groups two to a tile, 3101 one to a tile
@pytest.mark.parametrize("B,P,H,T", [(B, P, H, T) for T in range(3, 34) for B, P, H in ((1, 1, 1), (5, 7, 3))]
                         + [(3, 689, 3, 8), (7, 443, 1, 11), (7, 443, 1, 16), (7, 443, 1, 17), (7, 443, 1, 24)])
def test_temporal_windows(B, P, H, T):
    q, k, v = _inputs(B, P, H, T)
    out = _run(q, k, v).double()
    s = (q.double().unsqueeze(-2) * k.double().unsqueeze(-3)).sum(-1) * 0.125
    p = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device="cuda").tril(), float("-inf")).softmax(-1)
    ref = (p.unsqueeze(-1) * v.double().unsqueeze(-3)).sum(-2)
    # bf16 holds 8 significant bits (ulp 2^-7 in [1, 2)), so rounding to nearest costs at most 2^-8 of the value:
    # once for each probability (the sum divided by is of the unrounded ones) and once for the output; 1.02 covers
    # the fp32 scores and sums
    bound = 1.02 * 2.0 ** -8 * ((p.unsqueeze(-1) * v.double().abs().unsqueeze(-3)).sum(-2) + ref.abs())
    assert torch.isfinite(out).all() and ((out - ref).abs() <= bound).all()


@pytest.mark.parametrize("T", [5, 8, 9, 16, 17, 32])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_temporal_windows_keep_non_finite_values_apart(T, bad):
    """An infinite or NaN value in one frame of one group leaves earlier frames and other groups as they were."""
    q, k, v = _inputs(2, 3, 2, T)
    clean = _run(q, k, v).double()
    v[1, 1, 1, T - 2, 5] = bad
    out = _run(q, k, v).double()
    hit = torch.zeros_like(out, dtype=torch.bool)
    hit[1, 1, 1, T - 2:, 5] = True
    assert not torch.isfinite(out[hit]).any()
    # the finite elements may be summed in another order: one bf16 step
    assert torch.isfinite(out[~hit]).all()
    assert ((out - clean)[~hit].abs() <= 2.0 ** -7 * clean[~hit].abs() + 1e-4).all()


@pytest.mark.parametrize("T", [8, 11, 16, 17, 24, 32, 33])
@pytest.mark.parametrize("big", [2.0 ** 33, 2.0 ** 120])
def test_temporal_windows_of_huge_scores(T, big):
    """Scores beyond what exp2 holds, finite in fp32: the key of the largest score gets probability 1."""
    q, k, v = _inputs(2, 5, 3, T)
    k[..., T // 2, 9] = big
    out = _run(q, k, v).double()
    s = (q.double().unsqueeze(-2) * k.double().unsqueeze(-3)).sum(-1) * 0.125
    p = s.masked_fill(~torch.ones(T, T, dtype=torch.bool, device="cuda").tril(), float("-inf")).softmax(-1)
    ref = (p.unsqueeze(-1) * v.double().unsqueeze(-3)).sum(-2)
    # as test_temporal_windows
    bound = 1.02 * 2.0 ** -8 * ((p.unsqueeze(-1) * v.double().abs().unsqueeze(-3)).sum(-2) + ref.abs())
    assert torch.isfinite(out).all() and ((out - ref).abs() <= bound).all()
