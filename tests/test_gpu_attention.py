"""Attention without bias or causal mask: every staging variant at its edges, and non-finite values, against fp64."""
import pytest
import torch

from helpers import L, cuda, stream, sync

pytestmark = pytest.mark.gpu


def _inputs(n, sq, sk):
    g = torch.Generator().manual_seed(n + 3 * sq + 7 * sk)
    return [cuda(torch.randn(n, r, 64, generator=g) * 2, torch.bfloat16) for r in (sq, sk, sk)]


def _run(q, k, v):
    n, sq, _ = q.shape
    out = torch.full((n, sq, 64), float("nan"), device="cuda", dtype=torch.bfloat16)
    L.call("oasis_sdpa", L.ptr(q), L.ptr(k), L.ptr(v), L.ptr(out), n, sq, k.shape[1], 64, 0.125, None, 0, L.BF16,
           stream())
    sync()
    return out.double()


def _ref(q, k, v):
    s = torch.matmul(q.double(), k.double().transpose(-1, -2).contiguous()) * 0.125
    p = s.softmax(-1)
    return torch.matmul(p, v.double()), torch.matmul(p, v.double().abs())


# one stage of 96 to 192 keys with and without the probabilities' remainders, the two rings on either side of 256
# workgroups; one key past a stage, one short of it, one key in the last stage, and partial query tiles
@pytest.mark.parametrize("n,sq,sk", [(1, 1, 65), (2, 97, 96), (300, 48, 95), (3, 64, 97), (2, 65, 128), (260, 130, 127),
                                     (1, 1, 129), (200, 160, 160), (171, 150, 146), (129, 64, 145), (3, 144, 143),
                                     (256, 144, 144), (255, 144, 144), (257, 65, 1), (3, 97, 64),
                                     (2, 49, 144), (2, 47, 145), (3, 48, 160), (256, 128, 160), (256, 33, 159),
                                     (256, 48, 152), (2, 70, 161), (5, 200, 192), (2, 65, 193), (1, 16, 256),
                                     (3, 100, 257), (4, 4096, 385), (129, 100, 193), (128, 65, 320), (300, 1, 576),
                                     (30, 576, 576), (28, 576, 576), (300, 20, 641)])
def test_attention_variants(n, sq, sk):
    q, k, v = _inputs(n, sq, sk)
    out = _run(q, k, v)
    ref, mass = _ref(q, k, v)
    # bf16 rounds to within 2^-8: each probability (the sum divided by is of the unrounded ones) and the output;
    # 1.02 covers the fp32 scores and sums
    bound = 1.02 * 2.0 ** -8 * (mass + ref.abs())
    assert torch.isfinite(out).all() and ((out - ref).abs() <= bound).all()


@pytest.mark.parametrize("n,sq,sk", [(2, 144, 144), (256, 144, 144), (2, 96, 160), (2, 70, 192), (2, 64, 576),
                                     (2, 96, 96), (2, 100, 128), (200, 160, 160)])
def test_attention_keeps_infinite_values(n, sq, sk):
    """An infinite value gives infinity in its dim, whatever rounding left of its probability, and in no other."""
    q, k, v = _inputs(n, sq, sk)
    q = q * 0.25  # no probability underflows
    v[1, sk // 2, 9] = float("inf")
    out = _run(q, k, v)
    assert (out[1, :, 9] == float("inf")).all()
    out[1, :, 9] = 0
    assert torch.isfinite(out).all()


# every staging variant with keys past the sequence in its last stage
@pytest.mark.parametrize("n,sq,sk", [(3, 96, 32), (3, 144, 64), (2, 70, 65), (2, 100, 97), (2, 48, 143), (256, 144, 129),
                                     (2, 48, 159), (256, 64, 145), (2, 70, 161), (128, 65, 320), (16, 576, 576),
                                     (2, 40, 448), (300, 20, 641)])
def test_attention_keeps_an_infinite_last_value(n, sq, sk):
    """The rows that fill up the last stage repeat the last key with probability 0, and 0 x inf is not finite."""
    q, k, v = _inputs(n, sq, sk)
    q = q * 0.25  # no probability underflows
    v[1, sk - 1, 9] = float("inf")
    out = _run(q, k, v)
    assert (out[1, :, 9] == float("inf")).all()
    out[1, :, 9] = 0
    assert torch.isfinite(out).all()


# every staging variant, each chunk of keys holding both kinds of rounded key
@pytest.mark.parametrize("n,sq,sk", [(2, 144, 144), (256, 144, 144), (2, 48, 160), (256, 128, 160), (2, 70, 192),
                                     (3, 100, 257), (2, 64, 576), (300, 20, 640), (2, 96, 96), (2, 100, 128),
                                     (200, 160, 160)])
def test_attention_divides_by_the_unrounded_sum(n, sq, sk):
    """Keys whose probability bf16 rounds by nearly half a step, all in one direction, and whose values are zero
    reach the output through the softmax sum alone: the sum is of the fp32 probabilities."""
    s = torch.arange(-1.0, 0.0, 2.0 ** -8, dtype=torch.float64)   # scores that bf16 holds
    p = s.exp()
    off = (p.float().bfloat16().double() / p - 1)
    s = s[off.argmax()].item()
    assert off.max() > 0.003
    scores = torch.full((sk,), s, dtype=torch.float64)
    scores[::16] = 0                            # the largest score of every chunk: a probability of 1
    q, k, v = (torch.zeros(n, r, 64) for r in (sq, sk, sk))
    q[:, :, 0], k[:, :, 0] = 8, scores.float()  # q . k / 8
    v[:, sk - sk % 16 - 16] = torch.rand(n, 64, generator=torch.Generator().manual_seed(sk)).bfloat16().float() + 1
    v = v.bfloat16().float()
    out = _run(*(cuda(t, torch.bfloat16) for t in (q, k, v)))
    ref = (v.double().sum(1) / scores.exp().sum()).unsqueeze(1).cuda().expand_as(out)
    # one value with probability 1: exact but for fp32 (1e-5) and the output's rounding, to within 2^-8 of the
    # power of two below it (half a step of 2^-7)
    half_step = torch.exp2(torch.floor(torch.log2(ref))) * 2.0 ** -8
    assert ((out - ref).abs() <= half_step + 1e-5 * ref).all()
