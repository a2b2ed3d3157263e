"""The calls that a diffusion transformer makes of this package, as cases whose time is measured.

A case is a dict of plain values; ``kind`` names the path:

  self    self-attention over H heads and S tokens (joint image/text or video tokens): head_dim 64 and 128, other
          head_dims, bf16 and fp16, [B,H,S,D] and [B,S,H,D] memory, with and without the log-sum-exp, is_causal
  cross   attention of many query rows to a text prompt's or an image's tokens, with and without the additive
          padding bias that text encoders' masks become
  masked  self-attention under a mask: a padded prompt at the end of the keys ("prefix") or inside the gathered
          sequence of several ranks ("holes"), several samples packed into one sequence ("segments"), a relative
          bias per head ("bias")
  sparse  block-sparse attention (window, sinks and scattered blocks)
  ring    one rank's pass over the key/value blocks of a ring, resident or as they arrive
  cache   the First Block Cache step around a model's blocks: hit and miss, down-sampled, and with TaylorSeer

Sizes are those of the package's tests and benchmark, or lie between them.
"""
import math

import torch
import torch.nn.functional as F

import paraattention_amd
from paraattention_amd import TaylorSeer, UnifiedAttnMode, fbcache

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}


def _self(name, B, H, S, D, dtype="bf16", layout="bshd", lse=False, causal=False, norm=True):
    return {"name": name, "kind": "self", "B": B, "H": H, "S": S, "D": D, "dtype": dtype, "layout": layout, "lse": lse,
            "causal": causal, "norm": norm}


def listed():
    return [
        # the smallest calls: the text tokens of one prompt, where launches and the host count
        _self("small_self", 1, 24, 257, 128),
        # FLUX joint attention of one image (4096 image and 512 text tokens), called through the mode
        _self("image_joint", 1, 24, 4608, 128),
        # one rank's heads of a 119k-token video, output and log-sum-exp (the package's headline shape)
        _self("video_share", 1, 3, 119056, 128, layout="bhsd", lse=True),
        # a video model with head_dim 64 (CogVideoX)
        _self("video_head_dim_64", 1, 48, 17776, 64, norm=False),
        # the op test's own shape: fp16, is_causal, log-sum-exp
        _self("causal_fp16", 1, 24, 4096, 64, dtype="fp16", layout="bhsd", lse=True, causal=True, norm=False),
        # a head_dim that is neither 64 nor 128, two images of a guidance pair
        _self("image_head_dim_72", 2, 16, 4096, 72, norm=False),
        # Wan 2.1 cross-attention to the 512 tokens of a text prompt
        {"name": "cross_text", "kind": "cross", "B": 1, "H": 40, "Sq": 32760, "Skv": 512, "D": 128, "dtype": "bf16", "bias": False},
        # cross-attention to a padded prompt, the padding as an additive bias per key; a guidance pair
        {"name": "cross_padded", "kind": "cross", "B": 2, "H": 24, "Sq": 7800, "Skv": 256, "D": 128, "dtype": "bf16", "bias": True},
        # a boolean key mask with the prompt's padding inside the sequence gathered from two ranks
        {"name": "text_mask", "kind": "masked", "B": 1, "H": 24, "S": 4352, "D": 128, "dtype": "bf16", "mask": "holes"},
        # the benchmark's block-sparse shape: 128 x 128 tiles, about 30 % kept, a mask per head
        {"name": "block_sparse", "kind": "sparse", "B": 1, "H": 24, "blocks": 256, "block": 128, "D": 128, "dtype": "bf16",
         "density": 0.30, "per_head": True},
        # one rank's ring pass over eight resident blocks of the 119k-token video
        {"name": "ring_sweep", "kind": "ring", "B": 1, "H": 24, "S": 14882, "blocks": 8, "D": 128, "dtype": "bf16", "resident": True},
        # a cached step of a video model: residual, decision, residual added back
        {"name": "cache_hit", "kind": "cache", "B": 1, "rows": 32760, "width": 5120, "text": 512, "dtype": "bf16", "step": "hit", "stride": 1},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["self", "self", "self", "cross", "cross", "masked", "masked", "sparse", "ring", "cache", "cache"])
    dtype = rng.choice(["bf16", "bf16", "bf16", "fp16"])
    if kind == "self":
        D = rng.choice([128, 128, 128, 64, 64, rng.choice([40, 72, 80, 96])])
        B = rng.choice([1, 1, 2])
        H = rng.choice([3, 8, 12, 16, 24, 40])
        S = _log(rng, 200, 40000)
        while 4.0 * B * H * S * S * D > 1.5e13:
            S = S * 3 // 4
        case = _self("", B, H, S, D, dtype, rng.choice(["bhsd", "bshd"]), rng.random() < 0.3, rng.random() < 0.2, D == 128 and rng.random() < 0.7)
    elif kind == "cross":
        case = {"kind": "cross", "B": rng.choice([1, 2]), "H": rng.choice([12, 16, 24, 40]), "Sq": _log(rng, 1000, 33000),
                "Skv": rng.choice([77, 226, 256, 257, 333, 512, rng.randint(64, 512)]), "D": rng.choice([128, 128, 64]), "dtype": dtype,
                "bias": rng.random() < 0.5}
    elif kind == "masked":
        mask = rng.choice(["prefix", "holes", "holes", "segments", "bias"])
        B, H = rng.choice([1, 2]), rng.choice([8, 16, 24])
        S = _log(rng, 300, {"prefix": 12000, "holes": 12000, "segments": 8000, "bias": 3000}[mask])
        case = {"kind": "masked", "B": B, "H": H, "S": S, "D": rng.choice([128, 128, 64]), "dtype": dtype, "mask": mask}
    elif kind == "sparse":
        block = rng.choice([64, 128, 128, 256])
        case = {"kind": "sparse", "B": 1, "H": rng.choice([4, 8, 16, 24]), "blocks": max(8, _log(rng, 3000, 32768) // block), "block": block,
                "D": rng.choice([128, 128, 64]), "dtype": dtype, "density": round(rng.uniform(0.2, 0.5), 2), "per_head": rng.random() < 0.6}
    elif kind == "ring":
        case = {"kind": "ring", "B": 1, "H": rng.choice([6, 12, 24]), "S": _log(rng, 1000, 12000), "blocks": rng.choice([2, 4, 8]), "D": 128,
                "dtype": dtype, "resident": rng.random() < 0.5}
    else:
        case = {"kind": "cache", "B": rng.choice([1, 2]), "rows": _log(rng, 500, 16000), "width": rng.choice([1920, 3072, 5120]),
                "text": rng.choice([226, 256, 512]), "dtype": dtype, "step": rng.choice(["hit", "hit", "miss", "seer_hit", "seer_full"]),
                "stride": rng.choice([1, 1, 1, 2])}
    case.pop("name", None)
    return case


# ---------------------------------------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------------------------------------
class _Inputs:
    """Normally distributed tensors on the GPU from one seed."""

    def __init__(self, seed, dtype):
        self.device = torch.device("cuda")
        self.g = torch.Generator(device=self.device).manual_seed(seed)
        self.dtype = dtype

    def randn(self, *shape, dtype=None):
        return torch.randn(*shape, generator=self.g, device=self.device, dtype=dtype or self.dtype)

    def rows(self, B, H, S, D, layout="bhsd", norm=False):
        """Heads of queries, keys or values: [B,H,S,D], or a view of it on the [B,S,H,D] memory that a model's
        projection leaves; ``norm``: RMS-normalised per row, as models with a query/key norm hand them over."""
        shape = (B, H, S, D) if layout == "bhsd" else (B, S, H, D)
        t = self.randn(*shape)
        if norm:
            t = (t.float() * torch.rsqrt(t.float().square().mean(-1, keepdim=True) + 1e-6)).to(self.dtype)
        return t if layout == "bhsd" else t.transpose(1, 2)

    def uniform(self, *shape):
        return torch.rand(*shape, generator=self.g, device=self.device)


def _kept_lengths(x, B, n):
    """Per batch element the number of tokens that a prompt padded to n really has."""
    return ((0.15 + 0.8 * x.uniform(B)) * n).long().clamp(1, n)


def _padded_prompt_keys(x, case):
    """[B,S] boolean: which keys are kept.  "prefix": [image, text] with the padding at the end; "holes": the same
    sequence gathered from two ranks, each of which holds half of the image and half of the text."""
    B, S = case["B"], case["S"]
    ranks = 1 if case["mask"] == "prefix" else 2
    text = min(256, S // 4) // ranks * ranks
    length = _kept_lengths(x, B, text)[:, None]
    pos = torch.arange(S, device=x.device)
    shard = S // ranks
    in_shard = pos % shard
    in_text = (in_shard >= shard - text // ranks) & (pos < shard * ranks)
    index = (pos // shard) * (text // ranks) + in_shard - (shard - text // ranks)
    return ~in_text[None, :] | (index[None, :] < length)


def _block_mask(x, case):
    """bool [H or none, n, n]: a window of 4 blocks around the diagonal, two sink blocks, the rest scattered."""
    n = case["blocks"]
    i = torch.arange(n, device=x.device)
    base = ((i[:, None] - i[None, :]).abs() <= min(4, n // 8)) | (i[None, :] < min(2, n // 8))
    have = base.float().mean()
    fill = ((case["density"] - have) / (1.0 - have)).clamp(min=0.0)
    shape = (case["H"], n, n) if case["per_head"] else (n, n)
    return base | (x.uniform(*shape) < fill)


def prepare(case, seed):
    x = _Inputs(seed, DTYPES[case["dtype"]])
    kind = case["kind"]
    if kind == "self":
        B, H, S, D, layout = (case[n] for n in ("B", "H", "S", "D", "layout"))
        state = {"q": x.rows(B, H, S, D, layout, case["norm"]), "k": x.rows(B, H, S, D, layout, case["norm"]), "v": x.rows(B, H, S, D, layout)}
    elif kind == "cross":
        B, H, Sq, Skv, D = (case[n] for n in ("B", "H", "Sq", "Skv", "D"))
        state = {"q": x.rows(B, H, Sq, D, "bshd"), "k": x.rows(B, H, Skv, D, "bshd"), "v": x.rows(B, H, Skv, D, "bshd"), "bias": None}
        if case["bias"]:
            padding = torch.arange(Skv, device=x.device)[None, :] >= _kept_lengths(x, B, Skv)[:, None]
            state["bias"] = (padding.to(x.dtype) * -10000.0)[:, None, None, :]
    elif kind == "masked":
        B, H, S, D = (case[n] for n in ("B", "H", "S", "D"))
        state = {"q": x.rows(B, H, S, D, "bshd"), "k": x.rows(B, H, S, D, "bshd"), "v": x.rows(B, H, S, D, "bshd")}
        if case["mask"] == "bias":
            state["mask"] = 0.5 * x.randn(1, H, S, S)
        elif case["mask"] == "segments":
            # three samples of unequal length behind a prefix that all of them see
            cuts = (x.uniform(B, 2).sort(dim=1).values * S).long()
            pos = torch.arange(S, device=x.device)
            segment = (pos[None, :, None] >= cuts[:, None, :]).sum(-1)
            state["mask"] = ((segment[:, :, None] == segment[:, None, :]) | (pos < 64)[None, None, :])[:, None]
        else:
            state["mask"] = _padded_prompt_keys(x, case)[:, None, None, :]
    elif kind == "sparse":
        S = case["blocks"] * case["block"]
        state = {n: x.rows(case["B"], case["H"], S, case["D"]) for n in ("q", "k", "v")}
        state["mask"] = _block_mask(x, case)
    elif kind == "ring":
        shape = (case["B"], case["H"], case["S"], case["D"])
        state = {"q": x.rows(*shape), "k": [x.rows(*shape) for _ in range(case["blocks"])], "v": [x.rows(*shape) for _ in range(case["blocks"])]}
    else:
        shape = (case["B"], case["rows"], case["width"])
        before, prev = x.randn(*shape), x.randn(*shape)
        state = {"before": before, "after": before + prev + 0.05 * x.randn(*shape), "text": x.randn(case["B"], case["text"], case["width"])}
        seer = case["step"].startswith("seer")
        ctx = fbcache.create_cache_context(residual_diff_threshold=0.12, downsample_factor=case["stride"],
                                           warmup_steps=1 << 40 if case["step"] in ("miss", "seer_full") else 0)
        with fbcache.cache_context(ctx):
            ctx.mark_step_begin()
            fbcache.set_first_hidden_states_residual(prev)
            if not seer:
                state["rest"], state["rest_text"] = x.randn(*shape), x.randn(*state["text"].shape)
                fbcache.set_hidden_states_residual(state["rest"])
                fbcache.set_encoder_hidden_states_residual(state["rest_text"])
        state["context"] = ctx
        if seer:
            state["seer"] = TaylorSeer(n_derivatives=2, skip_interval_steps=3)
            for _ in range(3):  # three full steps: value, first and second difference
                state["seer"].mark_step_begin()
                state["seer"].update(x.randn(*shape))
            state["seer"].mark_step_begin()
    state["case"] = case
    return state


# ---------------------------------------------------------------------------------------------------------
# one pass
# ---------------------------------------------------------------------------------------------------------
def run(state):
    case = state["case"]
    kind = case["kind"]
    ns = torch.ops.para_attn
    if kind == "self":
        q, k, v = state["q"], state["k"], state["v"]
        if case["lse"]:
            return ns.attention_forward_with_lse(q, k, v, is_causal=case["causal"])
        with UnifiedAttnMode():
            return F.scaled_dot_product_attention(q, k, v, is_causal=case["causal"])
    if kind == "cross":
        with UnifiedAttnMode():
            return F.scaled_dot_product_attention(state["q"], state["k"], state["v"], attn_mask=state["bias"])
    if kind == "masked":
        if case["mask"] in ("prefix", "holes"):
            return ns.attention_forward_sparse_kv(state["q"], state["k"], state["v"], state["mask"])
        return ns.attention_forward_with_lse(state["q"], state["k"], state["v"], state["mask"])
    if kind == "sparse":
        return ns.attention_forward_block_sparse(state["q"], state["k"], state["v"], state["mask"])
    if kind == "ring":
        return paraattention_amd.ring_sweep(state["q"], state["k"], state["v"], fused=None if case["resident"] else True)
    return _cache_step(state)


def _cache_step(state):
    """What CachedTransformerBlocks does around a model's blocks in one denoising step."""
    case = state["case"]
    before, after, text = state["before"], state["after"], state["text"]
    with fbcache.cache_context(state["context"]):
        residual, hit = fbcache.first_block_step(after, before)
        if case["step"] == "hit":
            hidden, encoder = fbcache.apply_prev_hidden_states_residual(after, text)
            return residual, hit, hidden, encoder
        if case["step"] == "seer_hit":
            return residual, hit, state["seer"].approximate_value_plus(after)
        fbcache.set_first_hidden_states_residual(residual)
        if case["step"] == "seer_full":
            return residual, hit, state["seer"].approximate_derivative(residual)
        rest, _ = torch.ops.para_attn.fbcache_first_residual_diff(before, after, None)
        fbcache.set_hidden_states_residual(rest)
        return residual, hit, rest


# ---------------------------------------------------------------------------------------------------------
# the same in 64 bits
# ---------------------------------------------------------------------------------------------------------
def _attention64(q, k, v, keep=None, causal=False):
    """(out, lse) in 64 bits, a head and a slice of the query rows at a time.  ``keep(b, h, r0, r1)``: what is added to
    the scores of those rows, or where boolean which of them are kept."""
    B, H, Sq, D = q.shape
    Skv = k.shape[2]
    out = torch.empty(B, H, Sq, D, dtype=torch.float64, device=q.device)
    lse = torch.empty(B, H, Sq, dtype=torch.float64, device=q.device)
    rows = max(1, (1 << 28) // Skv)
    for b in range(B):
        for h in range(H):
            kt, vh = k[b, h].double().t().contiguous(), v[b, h].double()
            for r0 in range(0, Sq, rows):
                r1 = min(Sq, r0 + rows)
                s = q[b, h, r0:r1].double() @ kt
                s *= 1.0 / math.sqrt(D)
                if causal:
                    at = torch.arange(Skv, device=q.device)
                    s.masked_fill_(at[None, :] > at[r0:r1, None], -math.inf)
                if keep is not None:
                    m = keep(b, h, r0, r1)
                    if m.dtype == torch.bool:
                        s.masked_fill_(~m, -math.inf)
                    else:
                        s += m.double()
                top = s.amax(-1, keepdim=True)
                s.sub_(top).exp_()
                total = s.sum(-1, keepdim=True)
                out[b, h, r0:r1] = (s @ vh) / total
                lse[b, h, r0:r1] = (top + total.log())[:, 0]
    return out, lse


def exact(case, seed):
    state = prepare(case, seed)
    kind = case["kind"]
    if kind == "self":
        out, lse = _attention64(state["q"], state["k"], state["v"], causal=case["causal"])
        return (out, lse) if case["lse"] else out
    if kind == "cross":
        bias = state["bias"]
        return _attention64(state["q"], state["k"], state["v"], None if bias is None else lambda b, h, r0, r1: bias[b, 0])[0]
    if kind == "masked":
        mask = state["mask"]

        def keep(b, h, r0, r1):
            m = mask[b if mask.shape[0] > 1 else 0, h if mask.shape[1] > 1 else 0]
            return m[r0:r1] if m.shape[0] > 1 else m

        out, lse = _attention64(state["q"], state["k"], state["v"], keep)
        return out if case["mask"] in ("prefix", "holes") else (out, lse)
    if kind == "sparse":
        mask, block = state["mask"], case["block"]
        at = torch.arange(case["blocks"] * block, device=mask.device) // block
        return _attention64(state["q"], state["k"], state["v"], lambda b, h, r0, r1: (mask[h] if mask.dim() == 3 else mask)[at[r0:r1]][:, at])
    if kind == "ring":
        return _attention64(state["q"], torch.cat(state["k"], 2), torch.cat(state["v"], 2))
    residual = state["after"].double() - state["before"].double()
    if case["step"] == "hit":
        return residual, None, state["after"].double() + state["rest"].double(), state["text"].double() + state["rest_text"].double()
    return residual, None, -residual if case["step"] == "miss" else None  # the second residual is taken the other way round


# ---------------------------------------------------------------------------------------------------------
# what a pass cannot do without
# ---------------------------------------------------------------------------------------------------------
def _attention_work(B, H, Sq, Skv, D, kept=1.0, lse=False, more=0.0):
    return {"bytes": 2.0 * B * H * D * (2 * Sq + 2 * Skv) + (4.0 * B * H * Sq if lse else 0.0) + more,
            "flops": 4.0 * B * H * Sq * Skv * D * kept}


def work(case):
    kind = case["kind"]
    if kind == "self":
        return _attention_work(case["B"], case["H"], case["S"], case["S"], case["D"], 0.5 if case["causal"] else 1.0, case["lse"])
    if kind == "cross":
        return _attention_work(case["B"], case["H"], case["Sq"], case["Skv"], case["D"], more=2.0 * case["B"] * case["Skv"] if case["bias"] else 0.0)
    if kind == "masked":
        B, H, S = case["B"], case["H"], case["S"]
        mask = {"prefix": B * S, "holes": B * S, "segments": B * S * S, "bias": 2.0 * H * S * S}[case["mask"]]
        return _attention_work(B, H, S, S, case["D"], 0.5 if case["mask"] == "segments" else 1.0, case["mask"] in ("segments", "bias"), mask)
    if kind == "sparse":
        S = case["blocks"] * case["block"]
        mask = case["blocks"] ** 2 * (case["H"] if case["per_head"] else 1)
        return _attention_work(case["B"], case["H"], S, S, case["D"], case["density"], True, mask)
    if kind == "ring":
        return _attention_work(case["B"], case["H"], case["S"], case["S"] * case["blocks"], case["D"], 1.0, True)
    n, t = 2.0 * case["B"] * case["rows"] * case["width"], 2.0 * case["B"] * case["text"] * case["width"]
    compared = n / case["stride"]
    passes = {"hit": 3 * n + compared + 3 * n + 3 * t,        # after, before and the previous residual in, residual out; residual and state in, state out
              "miss": 3 * n + 3 * n,                          # two residuals
              "seer_hit": 3 * n + compared + 5 * n,           # three stored orders and the state in, state out
              "seer_full": 3 * n + 2 * n + 3 * n}[case["step"]]  # two older orders and the value in, two differences out
    return {"bytes": passes, "flops": 0.0}


def tolerance(case):
    if case["kind"] == "cache":
        return "exact"  # every operation rounds to the activation type, as the eager chain it stands for
    # Probabilities and output are rounded to the activation type.  Against the same attention in 64 bits the ops show
    # rel 2.1e-3..2.4e-3 and max 0.8e-2..1.6e-2 in bf16, 2.6e-4..3.0e-4 and 1.0e-3..2.3e-3 in fp16; four times that.
    return {"rel": 9.5e-3, "max": 0.06} if case["dtype"] == "bf16" else {"rel": 1.2e-3, "max": 0.009}
