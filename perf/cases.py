"""The framework's work, as callers have it done: the attention layer from its smallest calls to
the full model shape, the attention entry points on their own, the sparse attention's training
step, the residual / LayerNorm pass and a whole transformer block.

Sizes follow the repository's own configurations: 1,560 tokens per latent frame (30 x 52), target
and source video side by side, 40 heads of 128 dims (or one of 8 GPUs' share of 5), 512 text
tokens, the 2 x 4,096-token correctness configuration, and odd lengths around them.
"""
import math
import os
import sys

import torch

_PKG = os.path.join(os.getcwd(), "lightning-unified-video-editor-via-in-context-sparse-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from icsa_hip import wan  # noqa: E402
from icsa_hip.editing_sparse_attention import editing_sparse_attention  # noqa: E402
from icsa_hip.hip_host import (SparsePiecewiseAttn1stIntervalsFunction, flash_attn_func,  # noqa: E402
                               sparse_piecewise_attn_1st_intervals_hip)

D = 128
BLK = 64
HW = (30, 52)              # latent rows and columns of one frame: 1,560 tokens
FREQS = wan.wan_freqs(D)   # a model's RoPE table, built once
DEV = "cuda"
BF = torch.bfloat16


# ------------------------------------------------------------------------------------------
# the cases
# ------------------------------------------------------------------------------------------
def listed():
    return [
        # the attention layer at the repository's correctness configuration: two heads, target and
        # source of 4,096 tokens each (a small test or debug run)
        dict(name="layer_2heads_8k", kind="layer", B=1, H=2, t=4096, s=4096, qk="bf16", v="bf16", alpha="one"),
        # one latent frame, the image-editing use: 3,120 tokens, all 40 heads, the types the model
        # code hands over (q / k in f32 after RoPE, v in bf16, one gate value per token)
        dict(name="layer_image_f32qk", kind="layer", B=1, H=40, t=1560, s=1560, qk="f32", v="bf16", alpha="token"),
        # one of 8 GPUs' share of the heads at the full 21-frame length
        dict(name="layer_5heads_64k", kind="layer", B=1, H=5, t=32768, s=32768, qk="bf16", v="bf16", alpha="one"),
        # the headline: 40 heads, 21 frames of target and of source, padded to whole blocks
        dict(name="layer_40heads_64k", kind="layer", B=1, H=40, t=32768, s=32768, qk="bf16", v="bf16", alpha="one"),
        # everything between the projections and the output projection for a 9-frame clip: RMSNorm,
        # RoPE, gate, block sums, the attention layer on a length that ends inside a block
        dict(name="self_attention_9frames", kind="self_attention", B=1, H=40, f=9, sf=9),
        # cross attention of the 21-frame model: every video token against 512 text tokens
        dict(name="cross_attention_text", kind="flash", B=1, H=40, Sq=65520, Sk=512),
        # dense self attention of a short clip with an odd length (the layer's dense counterpart)
        dict(name="dense_6frames", kind="flash", B=1, H=12, Sq=9373, Sk=9373),
        # the sparse kernel's host entry with its default sparsity, inference
        dict(name="sparse_host_16k", kind="sparse", B=1, H=40, TQ=16384, TKV=16384, sparsity=0.1),
        # training: forward and backward of the sparse attention, small and at a 5-frame length
        # that ends inside a block
        dict(name="sparse_train_4heads_2k", kind="train", B=1, H=4, TQ=2048, TKV=2048, sparsity=0.1),
        dict(name="sparse_train_5frames", kind="train", B=1, H=40, TQ=7800, TKV=7800, sparsity=0.1),
        # residual update + LayerNorm + affine of the 21-frame residual stream
        dict(name="residual_norm_21frames", kind="norm", B=1, S=65520, dim=5120, mode="affine"),
        # a whole transformer block (projections, both attentions, FFN) on a 2-frame clip
        dict(name="block_2frames", kind="block", B=1, H=40, f=2, sf=2, ffn=13824, text=512),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "layer", "self_attention", "flash", "flash", "sparse",
                       "train", "train", "norm"])
    H = rng.choice([1, 2, 3, 4, 5, 8, 10, 12, 20, 40])
    B = 2 if rng.random() < 0.2 else 1
    if kind == "layer":
        top = 32768 if B * H <= 20 else 24000
        t = _log(rng, 512, top)
        if rng.random() < 0.5:
            t = t // BLK * BLK
        s = t if rng.random() < 0.7 else max(BLK, int(t * rng.uniform(0.5, 1.0)))
        return dict(kind=kind, B=B, H=H, t=t, s=s, qk=rng.choice(["bf16", "bf16", "f32"]),
                    v=rng.choice(["bf16", "bf16", "f32"]), alpha=rng.choice(["one", "token", "token"]))
    if kind == "self_attention":
        f = rng.randint(1, 21 if B * H <= 20 else 14)
        return dict(kind=kind, B=B, H=H, f=f, sf=f if rng.random() < 0.7 else rng.randint(1, f))
    if kind == "flash":
        Sq = _log(rng, 256, 65536 if H <= 20 else 32768)
        if rng.random() < 0.5:                       # text keys
            Sk = rng.choice([77, 226, 256, 512, 512])
        else:
            Sq = Sk = min(Sq, 24000)
        return dict(kind=kind, B=B, H=H, Sq=Sq, Sk=Sk)
    if kind == "sparse":
        TQ = _log(rng, 16, 640) * BLK
        TKV = TQ if rng.random() < 0.7 else max(16, int(TQ // BLK * rng.uniform(0.5, 1.0))) * BLK
        return dict(kind=kind, B=1, H=H, TQ=TQ, TKV=TKV, sparsity=rng.choice([0.0625, 0.1, 0.125, 0.25]))
    if kind == "train":
        TQ = _log(rng, 512, 16384)
        TKV = TQ if rng.random() < 0.7 else max(512, int(TQ * rng.uniform(0.5, 1.0)))
        return dict(kind=kind, B=B, H=H, TQ=TQ, TKV=TKV, sparsity=rng.choice([0.0625, 0.1, 0.125]))
    return dict(kind="norm", B=B, S=_log(rng, 64, 32768), dim=128 * rng.choice([2, 12, 13, 24, 40]),
                mode=rng.choice(["affine", "modulate", "first", "update"]))


# ------------------------------------------------------------------------------------------
# inputs
# ------------------------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(1000003 * int(seed) + 17)
    return g


def _n(g, *shape):
    return torch.randn(*shape, generator=g, device=DEV, dtype=torch.float32)


def _dt(name):
    return torch.float32 if name == "f32" else BF


def _paired(g, B, t, s, width, dtype):
    """Target rows first, then source rows; the target is a noisy copy of the source, as an edited
    clip is of its input."""
    src = _n(g, B, max(t, s), width)
    x = torch.empty(B, t + s, width, device=DEV, dtype=dtype)
    x[:, t:] = src[:, :s]
    x[:, :t] = src[:, :t] + 0.3 * _n(g, B, t, width)
    return x


def _inputs(case, seed):
    g = _gen(seed)
    kind, B = case["kind"], case["B"]
    st = {}
    if kind == "layer":
        H, t, s = case["H"], case["t"], case["s"]
        st["q"] = _n(g, B, t + s, H, D).to(_dt(case["qk"]))
        st["k"] = _paired(g, B, t, s, H * D, _dt(case["qk"])).view(B, t + s, H, D)
        st["v"] = _paired(g, B, t, s, H * D, _dt(case["v"])).view(B, t + s, H, D)
        st["alpha"] = 1.0
        if case["alpha"] == "token":
            st["alpha"] = (torch.sigmoid(_n(g, B, t + s, 1, 1)) - 0.5) * 0.5
    elif kind == "self_attention":
        H, t, s = case["H"], case["f"] * HW[0] * HW[1], case["sf"] * HW[0] * HW[1]
        st["yq"] = (1.5 * _n(g, B, t + s, H * D)).to(BF)
        st["yk"] = _paired(g, B, t, s, H * D, BF)
        st["yv"] = _paired(g, B, t, s, H * D, BF)
        st["logit"] = (2 * _n(g, B, t + s, 1)).to(BF)
        st["wq"] = 0.5 + torch.rand(H * D, generator=g, device=DEV)
        st["wk"] = 0.5 + torch.rand(H * D, generator=g, device=DEV)
    elif kind == "flash":
        st["q"] = _n(g, B, case["Sq"], case["H"], D).to(BF)
        st["k"] = _n(g, B, case["Sk"], case["H"], D).to(BF)
        st["v"] = _n(g, B, case["Sk"], case["H"], D).to(BF)
    elif kind in ("sparse", "train"):
        for name, T in (("q", case["TQ"]), ("k", case["TKV"]), ("v", case["TKV"])):
            st[name] = _n(g, B, case["H"], T, D).to(BF)
        if kind == "train":
            st["do"] = _n(g, B, case["H"], case["TQ"], D).to(BF)
    elif kind == "norm":
        S, dim = case["S"], case["dim"]
        st["x"] = _n(g, B, S, dim) * 1.5 + 0.2
        if case["mode"] == "first":                   # the patch embedding's output
            st["x"] = st["x"].to(BF)
        st["y"] = _n(g, B, S, dim).to(BF)
        for name in ("gate", "shift", "scale"):
            st[name] = 0.3 * _n(g, B, 1, dim)
        st["weight"] = 0.5 + torch.rand(dim, generator=g, device=DEV)
        st["bias"] = 0.1 * _n(g, dim)
    elif kind == "block":
        dim, ffn = case["H"] * D, case["ffn"]
        t, s = case["f"] * HW[0] * HW[1], case["sf"] * HW[0] * HW[1]
        st["x"] = _paired(g, B, t, s, dim, torch.float32)
        st["e"] = 0.3 * _n(g, B, 6, dim)
        st["context"] = _n(g, B, case["text"], dim).to(BF)
        W = {"modulation": (_n(g, 1, 6, dim) / dim ** 0.5).to(BF)}
        for a in ("self_attn", "cross_attn"):
            for p in ("q", "k", "v", "o"):
                W[f"{a}.{p}.weight"] = (_n(g, dim, dim) / dim ** 0.5).to(BF)
                W[f"{a}.{p}.bias"] = (0.02 * _n(g, dim)).to(BF)
            W[f"{a}.alpha_1.weight"] = (2 * _n(g, 1, dim) / dim ** 0.5).to(BF)
            W[f"{a}.alpha_2.weight"] = torch.zeros(1, dim, device=DEV, dtype=BF)
            for p in ("norm_q", "norm_k"):
                W[f"{a}.{p}.weight"] = (0.5 + torch.rand(dim, generator=g, device=DEV)).to(BF)
        W["norm3.weight"] = (0.5 + torch.rand(dim, generator=g, device=DEV)).to(BF)
        W["norm3.bias"] = (0.1 * _n(g, dim)).to(BF)
        W["ffn.0.weight"] = (_n(g, ffn, dim) / dim ** 0.5).to(BF)
        W["ffn.0.bias"] = (0.02 * _n(g, ffn)).to(BF)
        W["ffn.2.weight"] = (_n(g, dim, ffn) / ffn ** 0.5).to(BF)
        W["ffn.2.bias"] = (0.02 * _n(g, dim)).to(BF)
        st["W"] = W
    return st


def prepare(case, seed):
    st = _inputs(case, seed)
    st["case"] = case
    kind = case["kind"]
    if kind in ("self_attention", "block"):
        st["grid"] = [(case["f"],) + HW] * case["B"]
        st["src_grid"] = [(case["sf"],) + HW] * case["B"]
    if kind == "train":
        for name in ("q", "k", "v"):
            st[name].requires_grad_(True)
    if kind == "norm" and case["mode"] in ("affine", "first", "update"):
        st["x_out"] = torch.empty_like(st["x"], dtype=torch.float32)
    if kind == "block":
        dim = case["H"] * D
        with torch.device("meta"):
            blk = wan.WanAttentionBlock("t2v_cross_attn", dim, case["ffn"], case["H"], cross_attn_norm=True)
        blk.load_state_dict(st.pop("W"), strict=True, assign=True)
        st["blk"] = blk.requires_grad_(False).eval()
        st["lens"] = torch.tensor([st["x"].shape[1]] * case["B"])
    return st


# ------------------------------------------------------------------------------------------
# one pass
# ------------------------------------------------------------------------------------------
def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "layer":
        return editing_sparse_attention(st["q"], st["k"], st["v"], c["t"], c["s"], alpha_2=st["alpha"], backend="hip")
    if kind == "self_attention":
        return wan.wan_self_attention_core(st["yq"], st["yk"], st["yv"], st["logit"], st["wq"], st["wk"],
                                           st["grid"], st["src_grid"], 1, FREQS, c["H"], out_dtype=BF)
    if kind == "flash":
        return flash_attn_func(st["q"], st["k"], st["v"])
    if kind == "sparse":
        return sparse_piecewise_attn_1st_intervals_hip(st["q"], st["k"], st["v"], c["sparsity"])
    if kind == "train":
        out = SparsePiecewiseAttn1stIntervalsFunction.apply(st["q"], st["k"], st["v"], c["sparsity"], BLK)
        dq, dk, dv = torch.autograd.grad(out, (st["q"], st["k"], st["v"]), st["do"])
        return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}
    if kind == "norm":
        if c["mode"] == "affine":          # x + y * gate, then norm3
            o = wan.ln_modulate(st["x"], y=st["y"], gate=st["gate"], weight=st["weight"], bias=st["bias"],
                                x_out=st["x_out"])
            return {"out": o, "x": st["x_out"]}
        if c["mode"] == "first":           # the first block's bf16 stream updated into f32, modulated
            o = wan.ln_modulate(st["x"], shift=st["shift"], scale=st["scale"], y=st["y"], gate=st["gate"],
                                x_out=st["x_out"])
            return {"out": o, "x": st["x_out"]}
        if c["mode"] == "update":          # the block's last residual update
            wan.ln_modulate(st["x"], y=st["y"], gate=st["gate"], out=False, x_out=st["x_out"])
            return {"x": st["x_out"]}
        return {"out": wan.ln_modulate(st["x"], shift=st["shift"], scale=st["scale"])}
    return st["blk"](st["x"], st["e"], st["lens"], st["grid"], FREQS, st["context"], None, st["src_grid"], 1)


# ------------------------------------------------------------------------------------------
# what a pass cannot do without
# ------------------------------------------------------------------------------------------
def _sizes(t, S, sparsity=0.0625):
    NB = -(-S // BLK)
    n_t = t // BLK
    z = dict(NB=NB, n_t=n_t, n_s=NB - n_t, ks=max(1, int(n_t * sparsity)), peaked=NB // 2)
    z["topK"] = z["n_s"] // 8
    z["Tkv"] = t + z["topK"] * BLK
    z["NKV"] = -(-z["Tkv"] // BLK)
    z["top_k"] = max(1, int(sparsity * z["NKV"]))
    z["diffuse"] = NB - z["peaked"]
    return z


def _layer_flops(B, H, t, S):
    z = _sizes(t, S)
    dense = 4.0 * z["peaked"] * BLK * z["Tkv"] * D
    sparse = 4.0 * z["diffuse"] * BLK * D * (z["top_k"] * BLK + z["NKV"])
    blocks = 4.0 * z["NB"] ** 2 * D + 2.0 * z["diffuse"] * z["NKV"] * D
    return B * H * (dense + sparse + blocks)


def work(case):
    kind, B = case["kind"], case["B"]
    if kind == "layer":
        H, S = case["H"], case["t"] + case["s"]
        es = {"f32": 4, "bf16": 2}
        n = B * S * H * D
        nbytes = n * (3 * es[case["qk"]] + es[case["v"]])          # q, k, v, and x in q's type
        return {"bytes": nbytes, "flops": _layer_flops(B, H, case["t"], S)}
    if kind == "self_attention":
        H, t = case["H"], case["f"] * HW[0] * HW[1]
        S = t + case["sf"] * HW[0] * HW[1]
        return {"bytes": B * S * H * D * 8, "flops": _layer_flops(B, H, t, S)}
    if kind == "flash":
        H, Sq, Sk = case["H"], case["Sq"], case["Sk"]
        return {"bytes": B * H * D * 4 * (Sq + Sk), "flops": 4.0 * B * H * Sq * Sk * D}
    if kind in ("sparse", "train"):
        H, TQ, TKV = case["H"], case["TQ"], case["TKV"]
        NQ, NKV = -(-TQ // BLK), -(-TKV // BLK)
        top_k = max(1, int(case["sparsity"] * (TKV // BLK if kind == "train" else NKV)))
        pairs = B * H * NQ * BLK * D * (top_k * BLK + NKV)
        rank = 2.0 * B * H * NQ * NKV * D
        if kind == "sparse":
            return {"bytes": B * H * D * 2 * (2 * TQ + 2 * TKV), "flops": 4.0 * pairs + rank}
        # forward: q, k, v, out; backward: do, q, k, v, out, dq, dk, dv; five products per pair
        return {"bytes": B * H * D * 2 * (6 * TQ + 6 * TKV), "flops": 14.0 * pairs + rank}
    if kind == "norm":
        n = B * case["S"] * case["dim"]
        per = {"affine": 4 + 2 + 4 + 2, "first": 2 + 2 + 4 + 2, "update": 4 + 2 + 4, "modulate": 4 + 2}
        return {"bytes": n * per[case["mode"]], "flops": 8.0 * n}
    H, t = case["H"], case["f"] * HW[0] * HW[1]
    S = t + case["sf"] * HW[0] * HW[1]
    dim, ffn, text = H * D, case["ffn"], case["text"]
    weights = 8 * dim * dim + 2 * dim * ffn
    flops = 2.0 * B * (S * (6 * dim * dim + 2 * dim * ffn) + text * 2 * dim * dim)
    flops += _layer_flops(B, H, t, S) + 4.0 * B * H * S * text * D
    return {"bytes": 2.0 * weights + 8.0 * B * S * dim, "flops": flops}


def tolerance(case):
    """Measured against the 64-bit result, 2.0e-3 to 2.7e-3 for bf16 operands, probabilities and
    outputs; the bounds are about four times that."""
    kind = case["kind"]
    if kind == "norm":          # x is an f32 sum, out its bf16 LayerNorm (single-ulp flips)
        return {"rel": 2e-3, "max": 1e-2}
    if kind == "block":         # a rounding may move a near-tied choice of the attention layer
        return {"rel": 1e-2, "max": 0.5}
    return {"rel": 1e-2, "max": 0.1}


# ------------------------------------------------------------------------------------------
# the same in 64 bits
# ------------------------------------------------------------------------------------------
def _softmax_rows(q, k, v):
    """softmax(q k^T / sqrt(D)) v of one head in float64, in row ranges."""
    out = torch.empty(q.shape[0], v.shape[1], dtype=torch.float64, device=q.device)
    step = max(64, int(2e8) // max(1, k.shape[0]))
    kt, sc = k.t().contiguous(), 1 / math.sqrt(D)
    for i in range(0, q.shape[0], step):
        out[i:i + step] = torch.softmax((q[i:i + step] @ kt).mul_(sc), dim=-1) @ v
    return out


def _blocks(x, n):
    """[T, D] rows as n blocks of 64, zero rows past T."""
    y = torch.zeros(n * BLK, x.shape[1], dtype=x.dtype, device=x.device)
    y[:x.shape[0]] = x
    return y.view(n, BLK, -1)


def _piecewise(qb, kb, vb, KC, VC, idx, real=None):
    """The sparse piecewise attention of one head: qb [n, 64, D] against the blocks kb / vb
    [NKV, 64, D] named by idx [n, top_k] exactly and against the block sums of all others to first
    order.  The block sums' numerator and weight, taken in chunks of 64 blocks, are not rescaled
    when a later chunk raises the running maximum (the algorithm's definition).  Returns out and
    the log of the weight (natural units)."""
    n, top_k = idx.shape
    NKV, sc = kb.shape[0], 1 / math.sqrt(D)
    out = torch.empty(n, BLK, D, dtype=torch.float64, device=qb.device)
    lse = torch.empty(n, BLK, dtype=torch.float64, device=qb.device)
    step = max(1, int(6e7) // (top_k * BLK * D))
    for i in range(0, n, step):
        q, ix = qb[i:i + step], idx[i:i + step]
        m_ = q.shape[0]
        kx = kb[ix].reshape(m_, top_k * BLK, D)
        s = torch.matmul(q, kx.transpose(1, 2).contiguous()) * sc
        if real is not None:
            s.masked_fill_(~real[ix].reshape(m_, 1, top_k * BLK), -math.inf)
        m0 = s.amax(-1, keepdim=True)
        p = torch.exp(s - m0)
        acc, l = torch.matmul(p, vb[ix].reshape(m_, top_k * BLK, D)), p.sum(-1, keepdim=True)
        z = torch.matmul(q.reshape(-1, D), KC.t().contiguous()).view(m_, BLK, NKV) * (sc / BLK)
        used = torch.zeros(m_, NKV, dtype=torch.bool, device=q.device).scatter_(1, ix, True)
        z.masked_fill_(used[:, None, :], -math.inf)
        m, g, gl = m0, 0.0, 0.0
        for c in range(0, NKV, BLK):
            zc = z[:, :, c:c + BLK]
            m = torch.maximum(m, zc.amax(-1, keepdim=True))
            pc = torch.exp(zc - m)
            g = g + torch.matmul(pc.reshape(-1, zc.shape[2]), VC[c:c + BLK]).view(m_, BLK, D)
            gl = gl + BLK * pc.sum(-1, keepdim=True)
        f = torch.exp(m0 - m)
        den = l * f + gl
        out[i:i + step] = (acc * f + g) / den
        lse[i:i + step] = (m + torch.log(den))[..., 0]
    return out, lse


def _layer_exact(q, k, v, alpha, t, qa, ka, va):
    """q, k, v: one batch entry [S, H, D] float64 as the block sums see it; qa, ka, va: as the
    attention sees it; alpha [S] or a number.  Returns [S, H, D] float64."""
    S, H, _ = q.shape
    z = _sizes(t, S)
    NB, n_t = z["NB"], z["n_t"]
    size = torch.full((NB, 1), float(BLK), dtype=torch.float64, device=q.device)
    size[-1] = S - (NB - 1) * BLK
    out = torch.empty(S, H, D, dtype=torch.float64, device=q.device)
    for h in range(H):
        qs, ks, vs = (_blocks(x[:, h], NB).sum(1) for x in (q, k, v))
        P = torch.softmax((qs / size) @ (ks / size).t() / math.sqrt(D), dim=-1)
        oc = P @ (vs / size)
        sharp = torch.topk(P[:, :n_t], z["ks"], dim=-1).values.sum(-1)
        order = torch.argsort(sharp, descending=True, stable=True)
        sel = torch.argsort(P[:n_t, n_t:].sum(0), descending=True, stable=True)[:z["topK"]] + n_t

        def new(x):                                  # target rows, then the selected source blocks
            return torch.cat([x[:t, h], _blocks(x[:, h], NB)[sel].reshape(-1, D)])

        qb = _blocks(qa[:, h], NB)
        res = torch.empty(NB, BLK, D, dtype=torch.float64, device=q.device)
        pk, df = order[:z["peaked"]], order[z["peaked"]:]
        kn, vn = new(ka), new(va)
        res[pk] = _softmax_rows(qb[pk].reshape(-1, D), kn, vn).view(-1, BLK, D)
        KC, VC = _blocks(new(k), z["NKV"]).sum(1), _blocks(new(v), z["NKV"]).sum(1)
        idx = torch.topk(qs[df] @ KC.t(), z["top_k"], dim=-1).indices
        res[df] = _piecewise(qb[df], _blocks(kn, z["NKV"]), _blocks(vn, z["NKV"]), KC, VC, idx)[0]
        a = alpha.view(-1, 1) if isinstance(alpha, torch.Tensor) else alpha
        out[:, h] = res.reshape(-1, D)[:S] + a * oc.repeat_interleave(BLK, 0)[:S]
    return out


def _rope(x, grid, src_grid):
    """x [S, H, D] float64 rotated by frame, row and column of its token on its own grid."""
    S = x.shape[0]
    tab = FREQS.to(x.device)
    n_hw = D // 2 // 3
    parts = torch.split(tab, [D // 2 - 2 * n_hw, n_hw, n_hw], dim=1)
    ang = torch.ones(S, D // 2, dtype=torch.complex128, device=x.device)
    at = 0
    for f, h, w in (grid, src_grid):
        i = torch.arange(f * h * w, device=x.device)
        pos = (i // (h * w), i // w % h, i % w)
        ang[at:at + len(i)] = torch.cat([p[j] for p, j in zip(parts, pos)], dim=1)
        at += len(i)
    xc = torch.view_as_complex(x.reshape(S, -1, D // 2, 2).contiguous())
    return torch.view_as_real(xc * ang[:, None]).reshape(x.shape)


def _rms(y, w, H, eps=1e-6):
    """WanRMSNorm of a bf16 projection: the normalised row returns to bf16, the weight is f32."""
    y = y.double()
    r = torch.rsqrt(y.square().mean(-1, keepdim=True) + eps)
    return ((y * r).to(BF).double() * w.double()).view(y.shape[0], H, D)


def _core_exact(yq, yk, yv, logit, wq, wk, grid, src_grid, H):
    q, k = (_rope(_rms(y, w, H), grid, src_grid) for y, w in ((yq, wq), (yk, wk)))
    v = yv.double().view(-1, H, D)
    # the gate's bf16 steps are part of its definition
    sg = torch.sigmoid(logit.double().view(-1)).to(BF).double()
    gate = (sg - 0.5).to(BF).double() * 0.5
    return _layer_exact(q, k, v, gate, grid[0] * grid[1] * grid[2], q, k, v)


def _train_exact(q, k, v, do, sparsity):
    """Output and gradients of one head, [T, D] float64 each."""
    TQ, TKV = q.shape[0], k.shape[0]
    NQ, NKV = -(-TQ // BLK), -(-TKV // BLK)
    top_k = max(1, int(sparsity * (TKV // BLK)))
    sc = 1 / math.sqrt(D)
    qb, kb, vb, dob = _blocks(q, NQ), _blocks(k, NKV), _blocks(v, NKV), _blocks(do, NQ)
    KC, VC = kb.sum(1), vb.sum(1)
    real = (torch.arange(NKV * BLK, device=q.device) < TKV).view(NKV, BLK)
    idx = torch.topk(qb.sum(1) @ KC.t(), top_k, dim=-1).indices
    out, lse = _piecewise(qb, kb, vb, KC, VC, idx, real)
    lse = lse[..., None]
    lse.view(-1)[TQ:] = 0
    dvec = (dob * out).sum(-1, keepdim=True)
    dk, dv = torch.zeros_like(kb), torch.zeros_like(vb)
    dq = torch.empty_like(qb)
    step = max(1, int(3e7) // (top_k * BLK * D))
    for i in range(0, NQ, step):
        ix, qq, dd = idx[i:i + step], qb[i:i + step], dob[i:i + step]
        m_ = ix.shape[0]
        kx, vx = kb[ix].reshape(m_, -1, D), vb[ix].reshape(m_, -1, D)
        p = torch.exp(torch.matmul(qq, kx.transpose(1, 2).contiguous()) * sc - lse[i:i + step])
        p = p * real[ix].reshape(m_, 1, -1)
        ds = p * (torch.matmul(dd, vx.transpose(1, 2).contiguous()) - dvec[i:i + step])
        dq[i:i + step] = torch.matmul(ds, kx) * sc
        flat = ix.reshape(-1)
        dk.index_add_(0, flat, (torch.matmul(ds.transpose(1, 2).contiguous(), qq) * sc).view(-1, BLK, D))
        dv.index_add_(0, flat, torch.matmul(p.transpose(1, 2).contiguous(), dd).view(-1, BLK, D))
    used = torch.zeros(NQ, NKV, dtype=torch.bool, device=q.device).scatter_(1, idx, True)
    qf, dof = qb.view(-1, D), dob.view(-1, D)
    p = torch.exp(qf @ KC.t() * (sc / BLK) - lse.view(-1, 1)).view(NQ, BLK, NKV)
    p = p.masked_fill(used[:, None, :], 0).view(-1, NKV)
    ds = p * (dof @ VC.t() - BLK * dvec.view(-1, 1))
    dq = dq.view(-1, D) + ds @ KC * (sc / BLK)
    dk = dk + (ds.t() @ qf * (sc / BLK))[:, None, :]
    dv = dv + (p.t() @ dof)[:, None, :]
    return out.reshape(-1, D)[:TQ], dq[:TQ], dk.reshape(-1, D)[:TKV], dv.reshape(-1, D)[:TKV]


def _ln(x, eps=1e-6):
    m = x.mean(-1, keepdim=True)
    return (x - m) / torch.sqrt((x - m).square().mean(-1, keepdim=True) + eps)


def _block_exact(st, case, b):
    W, H = st["W"], case["H"]
    grid, src = (case["f"],) + HW, (case["sf"],) + HW
    e = (W["modulation"].double()[0] + st["e"][b].double())

    def lin(x, name, rnd=True):
        bias = W.get(name + ".bias")
        y = x @ W[name + ".weight"].double().t() + (bias.double() if bias is not None else 0.0)
        return y.to(BF).double() if rnd else y

    x = st["x"][b].double()
    # the decisions depend on the projections' bf16 values, which are part of the model's definition
    h = (_ln(x) * (1 + e[1]) + e[0]).to(BF).double()
    a = "self_attn."
    y = _core_exact(lin(h, a + "q"), lin(h, a + "k"), lin(h, a + "v"), lin(h, a + "alpha_1"),
                    W[a + "norm_q.weight"], W[a + "norm_k.weight"], grid, src, H)
    x = x + lin(y.reshape(len(x), -1), a + "o", False) * e[2]
    h = _ln(x) * W["norm3.weight"].double() + W["norm3.bias"].double()
    a, ctx = "cross_attn.", st["context"][b].double()
    q = _rms(lin(h, a + "q"), W[a + "norm_q.weight"], H)
    k = _rms(lin(ctx, a + "k"), W[a + "norm_k.weight"], H)
    v = lin(ctx, a + "v").view(-1, H, D)
    y = torch.stack([_softmax_rows(q[:, i], k[:, i], v[:, i]) for i in range(H)], dim=1)
    x = x + lin(y.reshape(len(x), -1), a + "o", False)
    h = _ln(x) * (1 + e[4]) + e[3]
    h = torch.nn.functional.gelu(lin(h, "ffn.0", False), approximate="tanh")
    return x + lin(h, "ffn.2", False) * e[5]


@torch.no_grad()
def exact(case, seed):
    st = _inputs(case, seed)
    kind, B = case["kind"], case["B"]
    if kind == "layer":
        al = st["alpha"]
        res = []
        for b in range(B):
            q, k, v = (st[n][b].double() for n in "qkv")
            res.append(_layer_exact(q, k, v, al[b].double().view(-1) if isinstance(al, torch.Tensor) else al,
                                    case["t"], q, k, v))
        return torch.stack(res)
    if kind == "self_attention":
        grid, src = (case["f"],) + HW, (case["sf"],) + HW
        return torch.stack([_core_exact(st["yq"][b], st["yk"][b], st["yv"][b], st["logit"][b], st["wq"],
                                        st["wk"], grid, src, case["H"]) for b in range(B)])
    if kind == "flash":
        out = torch.empty(B, case["Sq"], case["H"], D, dtype=torch.float64, device=DEV)
        for b in range(B):
            for h in range(case["H"]):
                out[b, :, h] = _softmax_rows(*(st[n][b, :, h].double().contiguous() for n in "qkv"))
        return out
    if kind == "sparse":
        out = torch.empty(B, case["H"], case["TQ"], D, dtype=torch.float64, device=DEV)
        NQ, NKV = case["TQ"] // BLK, case["TKV"] // BLK
        for b in range(B):
            for h in range(case["H"]):
                qb, kb, vb = (_blocks(st[n][b, h].double(), m) for n, m in (("q", NQ), ("k", NKV), ("v", NKV)))
                KC, VC = kb.sum(1), vb.sum(1)
                idx = torch.topk(qb.sum(1) @ KC.t(), max(1, int(case["sparsity"] * NKV)), dim=-1).indices
                out[b, h] = _piecewise(qb, kb, vb, KC, VC, idx)[0].view(-1, D)
        return out
    if kind == "train":
        names = ("out", "dq", "dk", "dv")
        res = {n: torch.empty(B, case["H"], case["TQ" if n in ("out", "dq") else "TKV"], D,
                              dtype=torch.float64, device=DEV) for n in names}
        for b in range(B):
            for h in range(case["H"]):
                for n, x in zip(names, _train_exact(*(st[m][b, h].double() for m in ("q", "k", "v", "do")),
                                                    case["sparsity"])):
                    res[n][b, h] = x
        return res
    if kind == "norm":
        mode, x = case["mode"], st["x"].double()
        if mode == "modulate":
            return {"out": _ln(x) * (1 + st["scale"].double()) + st["shift"].double()}
        x += st["y"].double() * st["gate"].double()
        if mode == "update":
            return {"x": x}
        n = _ln(x)
        if mode == "affine":
            n = n.mul_(st["weight"].double()).add_(st["bias"].double())
        else:
            n = n * (1 + st["scale"].double()) + st["shift"].double()
        return {"out": n, "x": x}
    return torch.stack([_block_exact(st, case, b) for b in range(B)])
