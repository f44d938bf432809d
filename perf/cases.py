"""Performance cases of the framework: what a program that uses it has it do, through its public
entry points, from the smallest calls to the largest.

Kinds of case (the listed ones are samples of the ranges that `draw` covers):
  norm          the per-kernel surface's LayerNorm + adaLN modulate on T padded frames' rows
  linear        the per-kernel surface's linear layer ([K, N] weights)
  sdpa          the per-kernel surface's attention: spatial, temporal (causal bias), VAE
  conditioning  timestep / action conditioning and every adaLN projection of the model
  step          a captured denoising step of B streams x T frames (bf16 or fp8 weights)
  kv            a multi-stream K/V-cache pass: context prefill, then the current frames (decode)
  frame         one generated frame: DDIM steps, bridge, VAE decode
  vae           a captured batched VAE decode
Weights and inputs are synthetic, of the model's shapes and with the spread that a trained model has
where it matters (adaLN gates and modulations of order one).
"""
import math

import torch

from __graft_entry__ import load_package

oasis = load_package()

D, H, HD, DM = 1024, 16, 64, 4096   # model width, heads, head dim, MLP width
P, PATCH = 144, 64                  # tokens of a frame, values of a patch
GRID, VGRID = (9, 16), (18, 32)     # DiT and VAE token grids
PPAD = 160                          # rows of a frame in the per-kernel surface's padded layout
VL, VLAT, VPATCH = 576, 32, 20      # VAE tokens, latent width, patch side
EXT, FREQ = 25, 256                 # action width, timestep embedding width
SCALING = 0.07843137255             # latent scaling factor
DEV = "cuda"


# ---- the cases -------------------------------------------------------------------------------

def listed():
    return [
        # two padded frames' rows through one LayerNorm and one modulate: the smallest calls a program
        # on the per-kernel surface makes, where the launch and its latency are all there is
        {"name": "norm_320", "kind": "norm", "rows": 320, "dtype": "bf16"},
        # the QKV projection of two padded frames on the per-kernel surface
        {"name": "linear_320_qkv", "kind": "linear", "rows": 320, "k": 1024, "n": 3072, "out": "bf16"},
        # spatial attention of two padded frames on the per-kernel surface
        {"name": "sdpa_spatial_2", "kind": "sdpa", "layout": "spatial", "frames": 2, "dtype": "bf16"},
        # conditioning of a 16-frame video batch of 4 DDIM steps: 16 x (1 + 4) rows in one call
        {"name": "conditioning_80", "kind": "conditioning", "rows": 80},
        # the denoising step of one stream with its two-frame window, the whole model
        {"name": "step_b1_t2", "kind": "step", "blocks": 16, "b": 1, "t": 2, "weights": "bf16"},
        # one frame of an interactive session: 4 DDIM steps on the K/V cache and the decode
        {"name": "frame_4", "kind": "frame", "steps": 4, "kv": True, "ctx_t": 14},
        # three sessions served together on the K/V cache: context prefill and one denoising pass
        {"name": "kv_b3", "kind": "kv", "blocks": 4, "b": 3},
        # two streams with a five-frame window: an ordinary batch between the tuned sizes
        {"name": "step_b2_t5", "kind": "step", "blocks": 4, "b": 2, "t": 5, "weights": "bf16"},
        # one stream with the longest window, 32 frames
        {"name": "step_b1_t32", "kind": "step", "blocks": 4, "b": 1, "t": 32, "weights": "bf16"},
        # three two-frame streams on fp8 weights
        {"name": "step_fp8_b3_t2", "kind": "step", "blocks": 4, "b": 3, "t": 2, "weights": "fp8"},
        # eight streams with eight-frame windows on fp8 weights: the largest batch
        {"name": "step_fp8_b8_t8", "kind": "step", "blocks": 4, "b": 8, "t": 8, "weights": "fp8"},
        # the decodes of three sessions' frames in one batch
        {"name": "vae_3", "kind": "vae", "latents": 3},
    ]


def _log_int(rng, lo, hi):
    """An integer in [lo, hi], spread over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo - 0.49), math.log(hi + 0.49)))))))


def draw(rng):
    kind = rng.choice(["norm", "linear", "sdpa", "conditioning", "step", "step", "step", "kv", "frame", "vae"])
    if kind == "norm":
        return {"kind": kind, "rows": _log_int(rng, 144, 5120), "dtype": rng.choice(["bf16", "f32"])}
    if kind == "linear":
        k, n = rng.choice([(1024, 3072), (1024, 1024), (1024, 4096), (4096, 1024), (1024, 64)])
        return {"kind": kind, "rows": _log_int(rng, 32, 5120), "k": k, "n": n, "out": rng.choice(["bf16", "f32"])}
    if kind == "sdpa":
        layout = rng.choice(["spatial", "temporal", "vae"])
        frames = (rng.choice([2, 4, 8, 16, 32]) if layout == "temporal"
                  else _log_int(rng, 1, 32) if layout == "spatial" else _log_int(rng, 1, 8))
        return {"kind": kind, "layout": layout, "frames": frames, "dtype": rng.choice(["bf16", "f32"])}
    if kind == "conditioning":
        return {"kind": kind, "rows": _log_int(rng, 1, 96)}
    if kind == "kv":
        return {"kind": kind, "blocks": 4, "b": _log_int(rng, 1, 16)}
    if kind == "frame":
        kv = rng.random() < 0.75
        return {"kind": kind, "steps": rng.randint(1, 4 if kv else 3), "kv": kv, "ctx_t": rng.randint(1, 50)}
    if kind == "vae":
        return {"kind": kind, "latents": _log_int(rng, 1, 8)}
    t = _log_int(rng, 1, 32)
    return {"kind": "step", "blocks": 4, "b": _log_int(rng, 1, max(1, 64 // t)), "t": t,
            "weights": rng.choice(["bf16", "fp8"])}


# ---- weights and inputs, from the seed alone ----------------------------------------------------

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(seed)

    def n(self, *shape, std=1.0, dtype=torch.float32):
        return (torch.randn(*shape, generator=self.g, device=DEV) * std).to(dtype)

    def w(self, *shape):
        return self.n(*shape, std=0.02, dtype=torch.bfloat16)

    def ints(self, hi, n):
        return torch.randint(0, hi, (n,), generator=self.g, device=DEV)


def _theta(n, dim):
    return (10000.0 ** (-2.0 * torch.arange(n, dtype=torch.float64) / dim)).float()


def _dit_weights(r, blocks):
    w = {"t_emb.w0": r.w(D, FREQ), "t_emb.b0": r.w(D), "t_emb.w2": r.w(D, D), "t_emb.b2": r.w(D),
         "ext.w": r.w(D, EXT), "ext.b": r.w(D), "x_emb.w": r.n(D, 16, 2, 2, std=0.1, dtype=torch.bfloat16),
         "x_emb.b": r.w(D)}
    for i in range(blocks):
        for kind in "st":
            p = "blocks.%d.%s." % (i, kind)
            w[p + "ada_w"], w[p + "ada_b"] = r.w(6 * D, D), r.n(6 * D, std=0.3, dtype=torch.bfloat16)
            w[p + "qkv_w"] = r.w(3 * D, D)
            w[p + "out_w"], w[p + "out_b"] = r.w(D, D), r.w(D)
            w[p + "fc1_w"], w[p + "fc1_b"] = r.w(DM, D), r.w(DM)
            w[p + "fc2_w"], w[p + "fc2_b"] = r.w(D, DM), r.w(D)
    w["final.ada_w"], w["final.ada_b"] = r.w(2 * D, D), r.n(2 * D, std=0.3, dtype=torch.bfloat16)
    w["final.w"], w["final.b"] = r.w(PATCH, D), r.w(PATCH)
    w["rope.spatial_freqs"], w["rope.temporal_freqs"] = _theta(HD // 4, HD // 2), _theta(HD // 2, HD)
    return w


def _vae_weights(r, depth=12):
    w = {"pq_w": r.n(D, VLAT, std=0.1, dtype=torch.bfloat16), "pq_b": r.w(D)}
    for i in range(depth):
        p = "dec.%d." % i
        for n in ("n1", "n2"):
            w[p + n + "_w"], w[p + n + "_b"] = 1 + r.n(D, std=0.1), r.n(D, std=0.02)
        w[p + "qkv_w"], w[p + "qkv_b"] = r.w(3 * D, D), r.w(3 * D)
        w[p + "proj_w"], w[p + "proj_b"] = r.w(D, D), r.w(D)
        w[p + "fc1_w"], w[p + "fc1_b"] = r.w(DM, D), r.w(DM)
        w[p + "fc2_w"], w[p + "fc2_b"] = r.w(D, DM), r.w(D)
    w["norm_w"], w["norm_b"] = 1 + r.n(D, std=0.1), r.n(D, std=0.02)
    w["pred_w"], w["pred_b"] = r.w(3 * VPATCH * VPATCH, D), r.w(3 * VPATCH * VPATCH)
    w["rope.vae_freqs"] = _theta(HD // 8, HD // 4)
    return w


def _actions(r, n):
    a = torch.zeros(n, EXT, device=DEV)
    a[torch.arange(n, device=DEV), r.ints(EXT, n)] = 1.0
    return a


def _dtype(name):
    return torch.bfloat16 if name == "bf16" else torch.float32


def _inputs(case, seed):
    """Everything a case draws: used by prepare and, in 64 bits, by exact."""
    r = _Rand(seed)
    k = case["kind"]
    if k == "norm":
        n, dt = case["rows"], _dtype(case["dtype"])
        return {"x": r.n(n, D, dtype=dt), "w": 1 + r.n(D, std=0.1), "b": r.n(D, std=0.1),
                "shift": r.n(n, D, std=0.3, dtype=dt), "scale": r.n(n, D, std=0.3, dtype=dt)}
    if k == "linear":
        return {"x": r.n(case["rows"], case["k"], dtype=torch.bfloat16), "w": r.w(case["k"], case["n"])}
    if k == "sdpa":
        dt = _dtype(case["dtype"])
        heads, seq = _sdpa_shape(case)
        q, kk, v = (r.n(heads * seq, HD, dtype=dt) for _ in range(3))
        i = torch.arange(seq, device=DEV)
        t = case["frames"]
        # the block-diagonal causal bias of positions whose t frames stand in consecutive rows
        keep = (i[:, None] // t == i[None] // t) & (i[None] <= i[:, None])
        bias = torch.where(keep, 0.0, -1e4) if case["layout"] == "temporal" else None
        return {"q": q, "k": kk, "v": v, "bias": bias}
    if k == "conditioning":
        n = case["rows"]
        return {"w": _dit_weights(r, 16), "t": r.ints(1000, n).float(), "a": _actions(r, n)}
    if k == "step":
        n = case["b"] * case["t"]
        return {"w": _dit_weights(r, case["blocks"]), "patches": r.n(n * P, PATCH), "t": r.ints(1000, n).float(),
                "a": _actions(r, n)}
    if k == "kv":
        b = case["b"]
        # rows [0, b) the context frames (lightly noised), [b, 2b) the current ones
        return {"w": _dit_weights(r, case["blocks"]), "ctx": r.n(b * P, PATCH), "cur": r.n(b * P, PATCH),
                "t": torch.cat([torch.full((b,), 14.0, device=DEV), r.ints(1000, b).float()]), "a": _actions(r, 2 * b)}
    if k == "frame":
        return {"w": _dit_weights(r, 16), "vw": _vae_weights(r), "noise": r.n(P, PATCH).clamp(-20, 20),
                "ctx": r.n(P, PATCH), "a": _actions(r, 2)}
    return {"vw": _vae_weights(r), "latents": r.n(case["latents"], VL, VLAT)}


def _sdpa_shape(case):
    """(heads stacked along the rows, rows of each)"""
    if case["layout"] == "spatial":
        return H * case["frames"], PPAD
    if case["layout"] == "vae":
        return H * case["frames"], VL
    return H * PPAD * case["frames"] // 32, 32


def _schedule(case):
    return oasis.schedule.ddim_steps(case["steps"]), oasis.schedule.sigmoid_alphas_cumprod()


# ---- prepare and run ----------------------------------------------------------------------------

_STREAM = []


def _stream():
    """The one stream that a program runs its captured graphs on (its passes follow one another)."""
    if not _STREAM:
        _STREAM.append(torch.cuda.Stream())
    return _STREAM[0]


def prepare(case, seed):
    k = case["kind"]
    x = _inputs(case, seed)
    st = {"kind": k}
    if k == "norm":
        st.update(x, ln=torch.empty_like(x["x"]), out=torch.empty_like(x["x"]))
    elif k == "linear":
        st.update(x, fn=oasis.kernels.make_linear_kernel(case["k"] // 32),
                  out=torch.empty(case["rows"], case["n"], device=DEV, dtype=_dtype(case["out"])))
    elif k == "sdpa":
        heads, seq = _sdpa_shape(case)
        st.update(x, out=torch.empty_like(x["q"]))
        if x["bias"] is None:
            st["fn"] = oasis.kernels.make_sdpa_kernel(seq // 32, seq // 32, 2, 0.125)
        else:
            st["fn"] = oasis.kernels.make_sdpa_causal_kernel(1, 1, 2, 0.125, heads)
    elif k == "conditioning":
        dit = oasis.DiT(x["w"], DEV)
        st.update(dit=dit, ws=dit.workspace(P, max_cond=max(16, case["rows"])), t=x["t"], a=x["a"])
    elif k == "step":
        dit = oasis.DiT(x["w"], DEV, weights=case["weights"])
        step = oasis.DiTStep(dit, B=case["b"], T=case["t"], stream=_stream())
        step.set_inputs(x["patches"], x["t"], x["a"])
        step.capture()
        st["step"] = step
    elif k == "kv":
        b = case["b"]
        dit = oasis.DiT(x["w"], DEV)
        ws = dit.workspace(2 * b * P, max_cond=max(16, 2 * b))
        kv = oasis.model.KVCache(dit, b)
        ws.t[:2 * b].copy_(x["t"])
        ws.act[:2 * b, :EXT].copy_(x["a"])
        s = _stream()

        def passes():
            dit.conditioning_inplace(2 * b, ws, s)
            dit.patch_embed(x["ctx"], ws.x, s)
            dit.precompute_past(ws, kv, b, ws.ada, dit.ada_width, s)
            dit.patch_embed(x["cur"], ws.x, s)
            dit.forward_current(ws, kv, b, ws.ada[b:], dit.ada_width, ws.v_out, s)
        st.update(graph=oasis.Graph(passes, s), stream=s, out=(ws.v_out[:b * P], kv.k, kv.v), keep=(dit, ws, kv, x))
    elif k == "frame":
        steps, alphas = _schedule(case)
        fp = oasis.FramePipeline(oasis.DiT(x["w"], DEV), oasis.VAE(x["vw"], DEV), steps, alphas, stream=_stream(),
                                 kv_cache=case["kv"])
        fp.set_inputs(x["noise"], x["ctx"], float(case["ctx_t"]), x["a"][0], x["a"][1])
        fp.capture()
        st.update(fp=fp, noise=x["noise"])
    else:
        vae = oasis.VAE(x["vw"], DEV)
        ws = vae.workspace(max_frames=case["latents"])
        frames = torch.empty(case["latents"], *vae.frame_shape, device=DEV)
        s = _stream()
        st.update(graph=oasis.Graph(lambda: vae.decode_batch(x["latents"], frames, ws, s), s), stream=s, out=frames,
                  keep=(vae, ws, x))
    torch.cuda.synchronize()
    return st


def run(st):
    k = st["kind"]
    if k == "norm":
        oasis.kernels.layernorm_d1024(st["x"], st["w"], st["b"], None, None, st["ln"])
        oasis.kernels.adaln_modulate_kernel(st["ln"], st["shift"], st["scale"], st["out"])
        return st["ln"], st["out"]
    if k == "linear":
        st["fn"](st["x"], st["w"], st["out"])
        return st["out"]
    if k == "sdpa":
        if st["bias"] is None:
            st["fn"](st["q"], st["k"], st["v"], None, None, st["out"])
        else:
            st["fn"](st["q"], st["k"], st["v"], None, st["bias"], None, st["out"])
        return st["out"]
    if k == "conditioning":
        return st["dit"].conditioning(st["t"], st["a"], st["ws"])
    if k == "step":
        return st["step"].run()
    if k == "frame":   # fresh noise for the frame, then its graph, on the pipeline's stream
        fp = st["fp"]
        with torch.cuda.stream(fp.stream):
            fp.chunk.copy_(st["noise"])
        return fp.chunk, fp.run()
    st["graph"].launch()
    torch.cuda.current_stream().wait_stream(st["stream"])
    return st["out"]


# ---- what a pass cannot do without ------------------------------------------------------------

_SUB = 3 * D * D + D * D + 2 * D * DM          # projection weights of a sub-block
_COND = 4 * (D * FREQ + D * (D + 64) + 2 * D)   # conditioning MLP, fp32


def _ada_bytes(blocks):
    return 2 * 2 * blocks * 6 * D * (D + 2) + 4 * 2 * D * (D + 1)


def _cond_flops(rows, blocks):
    return 2 * rows * (D * FREQ + D * (D + EXT) + (2 * blocks * 6 + 2) * D * D)


def _block_flops(b, t, blocks):
    m = b * t * P
    attn = 4 * m * P * D + 4 * b * P * D * (t * (t + 1) // 2)
    return blocks * (2 * 2 * m * _SUB + attn)


def _vae_work(n, depth=12):
    m = n * VL
    pred = 3 * VPATCH * VPATCH
    flops = depth * (2 * m * _SUB + 4 * m * VL * D) + 2 * m * D * (VLAT + pred)
    return 2 * (depth * _SUB + D * (VLAT + pred)) + 4 * m * (VLAT + pred), flops


def work(case):
    k = case["kind"]
    if k == "norm":
        n, e = case["rows"] * D, 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 5 * n * e + 8 * D, "flops": 11 * n}
    if k == "linear":
        m, kk, n = case["rows"], case["k"], case["n"]
        return {"bytes": 2 * (m * kk + kk * n) + m * n * (2 if case["out"] == "bf16" else 4), "flops": 2 * m * kk * n}
    if k == "sdpa":
        heads, seq = _sdpa_shape(case)
        e = 2 if case["dtype"] == "bf16" else 4
        return {"bytes": 4 * heads * seq * HD * e, "flops": 4 * heads * seq * seq * HD}
    if k == "conditioning":
        rows = case["rows"]
        return {"bytes": _COND + _ada_bytes(16) + 4 * rows * (32 * 6 + 2) * D, "flops": _cond_flops(rows, 16)}
    if k == "step":
        b, t, n = case["b"], case["t"], case["blocks"]
        e = 2 if case["weights"] == "bf16" else 1
        m = b * t * P
        return {"bytes": _COND + _ada_bytes(n) + e * 2 * n * _SUB + 4 * 2 * PATCH * D + 4 * 2 * m * PATCH,
                "flops": _cond_flops(b * t, n) + _block_flops(b, t, n) + 4 * m * PATCH * D}
    if k == "kv":
        b, n = case["b"], case["blocks"]
        m = b * P
        return {"bytes": _COND + _ada_bytes(n) + 2 * 2 * n * _SUB + 4 * 2 * PATCH * D + 4 * 3 * m * PATCH
                + 2 * 2 * n * 2 * m * D,
                "flops": _cond_flops(2 * b, n) + 2 * _block_flops(b, 1, n) + 6 * m * PATCH * D}
    if k == "frame":
        n = case["steps"]
        passes = (n + 1) if case["kv"] else 2 * n   # frames through the model
        vb, vf = _vae_work(1)
        return {"bytes": _COND + _ada_bytes(16) + 2 * 32 * _SUB + vb,
                "flops": _cond_flops(1 + n, 16) + passes * _block_flops(1, 1, 16) + vf}
    vb, vf = _vae_work(case["latents"])
    return {"bytes": vb, "flops": vf}


def tolerance(case):
    k = case["kind"]
    if k == "norm":
        return {"rel": 1e-2 if case["dtype"] == "bf16" else 1e-6}
    if k == "linear":
        return {"rel": 1e-2 if case["out"] == "bf16" else 1e-5}
    if k == "sdpa":
        return {"rel": 1e-2}
    if k == "conditioning":
        return {"rel": 1e-5}
    if k == "step" and case["weights"] == "fp8":   # measured against exact: 0.022
        return {"rel": 6e-2}
    if k == "vae":   # 0.0038, through 12 layers
        return {"rel": 1.5e-2}
    return {"rel": 1e-2}   # step, kv, frame: 0.0011 to 0.0026


# ---- the same results in 64 bits ----------------------------------------------------------------

def _d(t):
    return t.double()


def _silu(x):
    return x * torch.sigmoid(x)


def _ln(x, w=None, b=None):
    y = (x - x.mean(-1, keepdim=True)) / torch.sqrt(x.var(-1, unbiased=False, keepdim=True) + 1e-6)
    return y if w is None else y * _d(w) + _d(b)


def _softmax_attn(q, k, v, bias=None):
    s = torch.matmul(q, k.transpose(-1, -2).contiguous()) * 0.125
    if bias is not None:
        s = s + bias
    return torch.matmul(torch.softmax(s, -1), v)


def _rotate(x, ang):
    """Pairs (2i, 2i+1) of the last dim's first ang.shape[-1] values turned by their angles."""
    n = ang.shape[-1]
    a, b = x[..., 0:n:2], x[..., 1:n:2]
    c, s = torch.cos(ang[..., ::2]), torch.sin(ang[..., ::2])
    return torch.cat([torch.stack([a * c - b * s, b * c + a * s], -1).flatten(-2), x[..., n:]], -1)


def _axial(freqs, gh, gw):
    f = _d(freqs).to(DEV)
    y = torch.linspace(-1, 1, gh, device=DEV, dtype=torch.float64)[:, None] * f
    x = torch.linspace(-1, 1, gw, device=DEV, dtype=torch.float64)[:, None] * f
    y = y.repeat_interleave(2, 1)[:, None].expand(gh, gw, -1)
    x = x.repeat_interleave(2, 1)[None].expand(gh, gw, -1)
    return torch.cat([y, x], -1).reshape(gh * gw, -1)


def _cond64(w, t, a):
    half = FREQ // 2
    f = torch.exp(-math.log(10000.0) * torch.arange(half, device=DEV, dtype=torch.float64) / half)
    ang = _d(t)[:, None] * f
    emb = torch.cat([torch.cos(ang), torch.sin(ang)], -1)
    hid = _silu(emb @ _d(w["t_emb.w0"]).t() + _d(w["t_emb.b0"]))
    return hid @ _d(w["t_emb.w2"]).t() + _d(w["t_emb.b2"]) + _d(a) @ _d(w["ext.w"]).t() + _d(w["ext.b"])


def _proj(w, weights):
    """A projection weight in 64 bits, as the model holds it: bf16, or e4m3 with a scale per channel."""
    if weights != "fp8":
        return _d(w)
    s = w.float().abs().amax(1, keepdim=True) / 448.0
    s = torch.where(s > 0, s, torch.ones_like(s))
    return _d((w.float() / s).to(torch.float8_e4m3fn).float()) * _d(s)


def _blocks64(w, x, cond, blocks, weights="bf16"):
    """x [B, T, P, D], cond [B, T, D] -> (x after the sub-blocks, [(rotated k, v) of each temporal one])"""
    B, T = x.shape[:2]
    sc = _silu(cond)
    s_ang = _axial(w["rope.spatial_freqs"], *GRID)
    t_ang = (torch.arange(T, device=DEV, dtype=torch.float64)[:, None]
             * _d(w["rope.temporal_freqs"]).to(DEV)).repeat_interleave(2, 1)
    causal = torch.full((T, T), float("-inf"), device=DEV, dtype=torch.float64).triu(1)
    kvs = []
    for i in range(blocks):
        for kind in "st":
            p = "blocks.%d.%s." % (i, kind)
            ada = (sc @ _d(w[p + "ada_w"]).t() + _d(w[p + "ada_b"]))[:, :, None, :].split(D, -1)
            h = _ln(x) * (1 + ada[1]) + ada[0]
            q, k, v = (y.reshape(B, T, P, H, HD) for y in (h @ _proj(w[p + "qkv_w"], weights).t()).split(D, -1))
            # -> [B, T, H, P, HD] or [B, P, H, T, HD]
            order = (0, 1, 3, 2, 4) if kind == "s" else (0, 2, 3, 1, 4)
            q, k, v = (y.permute(order).contiguous() for y in (q, k, v))
            ang = s_ang if kind == "s" else t_ang
            k = _rotate(k, ang)
            o = _softmax_attn(_rotate(q, ang), k, v, None if kind == "s" else causal)
            if kind == "t":
                kvs.append((k, v))
            o = o.permute((0, 1, 3, 2, 4) if kind == "s" else (0, 3, 1, 2, 4)).reshape(B, T, P, D)
            x = x + ada[2] * (o @ _proj(w[p + "out_w"], weights).t() + _d(w[p + "out_b"]))
            h = _ln(x) * (1 + ada[4]) + ada[3]
            h = torch.nn.functional.gelu(h @ _proj(w[p + "fc1_w"], weights).t() + _d(w[p + "fc1_b"]),
                                         approximate="tanh")
            x = x + ada[5] * (h @ _proj(w[p + "fc2_w"], weights).t() + _d(w[p + "fc2_b"]))
    return x, kvs


def _embed64(w, patches):
    cw = _d(w["x_emb.w"]).permute(0, 2, 3, 1).reshape(D, PATCH)
    return _d(patches) @ cw.t() + _d(w["x_emb.b"])


def _final64(w, x, cond):
    shift, scale = (_silu(cond) @ _d(w["final.ada_w"]).t() + _d(w["final.ada_b"]))[:, :, None, :].split(D, -1)
    return (_ln(x) * (1 + scale) + shift) @ _d(w["final.w"]).t() + _d(w["final.b"])


def _vae64(w, latents, depth=12):
    n = latents.shape[0]
    x = _d(latents) @ _d(w["pq_w"]).t() + _d(w["pq_b"])
    ang = _axial(w["rope.vae_freqs"], *VGRID)
    for i in range(depth):
        p = "dec.%d." % i
        qkv = _ln(x, w[p + "n1_w"], w[p + "n1_b"]) @ _d(w[p + "qkv_w"]).t() + _d(w[p + "qkv_b"])
        q, k, v = (y.reshape(n, VL, H, HD).permute(0, 2, 1, 3).contiguous() for y in qkv.split(D, -1))
        o = _softmax_attn(_rotate(q, ang), _rotate(k, ang), v).permute(0, 2, 1, 3).reshape(n, VL, D)
        x = x + o @ _d(w[p + "proj_w"]).t() + _d(w[p + "proj_b"])
        h = _ln(x, w[p + "n2_w"], w[p + "n2_b"]) @ _d(w[p + "fc1_w"]).t() + _d(w[p + "fc1_b"])
        x = x + torch.nn.functional.gelu(h) @ _d(w[p + "fc2_w"]).t() + _d(w[p + "fc2_b"])
    y = _ln(x, w["norm_w"], w["norm_b"]) @ _d(w["pred_w"]).t() + _d(w["pred_b"])
    y = y.reshape(n, VGRID[0], VGRID[1], 3, VPATCH, VPATCH).permute(0, 3, 1, 4, 2, 5)
    return y.reshape(n, 3, VGRID[0] * VPATCH, VGRID[1] * VPATCH).clamp(-1, 1)


def exact(case, seed):
    k = case["kind"]
    x = _inputs(case, seed)
    if k == "norm":
        y = _ln(_d(x["x"]), x["w"], x["b"])
        return y, y * (1 + _d(x["scale"])) + _d(x["shift"])
    if k == "linear":
        return _d(x["x"]) @ _d(x["w"])
    if k == "sdpa":
        heads, seq = _sdpa_shape(case)
        q, kk, v = (_d(x[n]).reshape(heads, seq, HD) for n in "qkv")
        return _softmax_attn(q, kk, v, None if x["bias"] is None else _d(x["bias"])).reshape(heads * seq, HD)
    if k == "vae":
        return _vae64(x["vw"], x["latents"])
    w = x["w"]
    if k == "conditioning":
        sc = _silu(_cond64(w, x["t"], x["a"]))
        names = ["blocks.%d.%s." % (i, kind) for i in range(16) for kind in "st"] + ["final."]
        cols = []
        for p in names:
            y = sc @ _d(w[p + "ada_w"]).t() + _d(w[p + "ada_b"])
            y[:, D:2 * D] += 1.0   # the model's rows hold 1 + scale
            if y.shape[1] == 6 * D:
                y[:, 4 * D:5 * D] += 1.0
            cols.append(y)
        return torch.cat(cols, 1)
    if k == "step":
        b, t = case["b"], case["t"]
        cond = _cond64(w, x["t"], x["a"]).reshape(b, t, D)
        h, _ = _blocks64(w, _embed64(w, x["patches"]).reshape(b, t, P, D), cond, case["blocks"], case["weights"])
        return _final64(w, h, cond).reshape(b * t * P, PATCH)
    if k == "kv":
        b = case["b"]
        cond = _cond64(w, x["t"], x["a"]).reshape(2, b, D).transpose(0, 1).contiguous()
        z = torch.stack([_embed64(w, x["ctx"]).reshape(b, P, D), _embed64(w, x["cur"]).reshape(b, P, D)], 1)
        h, kvs = _blocks64(w, z, cond, case["blocks"])
        v = _final64(w, h, cond)[:, 1].reshape(b * P, PATCH)
        return v, torch.stack([y[0] for y in kvs]), torch.stack([y[1] for y in kvs])
    # frame: DDIM steps with the context frame beside the generated one, then the decode
    steps, alphas = _schedule(case)
    ctx = _embed64(w, x["ctx"])
    chunk = _d(x["noise"])
    for i, (t, tn) in enumerate(steps):
        ts = torch.tensor([float(case["ctx_t"]), float(t)], device=DEV)
        cond = _cond64(w, ts, x["a"])[None]
        h, _ = _blocks64(w, torch.stack([ctx, _embed64(w, chunk)])[None], cond, 16)
        v = _final64(w, h, cond)[0, 1]
        at = float(alphas[t])
        an = 1.0 if i == len(steps) - 1 else float(alphas[max(tn, 0)])
        x0 = math.sqrt(at) * chunk - math.sqrt(1 - at) * v
        eps = (chunk / math.sqrt(at) - x0) / math.sqrt(1 / at - 1)
        chunk = math.sqrt(an) * x0 + math.sqrt(1 - an) * eps
    lat = chunk.reshape(GRID[0], GRID[1], 2, 2, 16).permute(0, 2, 1, 3, 4).reshape(VL, 16) / SCALING
    lat = torch.nn.functional.pad(lat, (0, VLAT - 16))
    return chunk, _vae64(x["vw"], lat[None])[0]
