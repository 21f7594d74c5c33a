"""The workloads this library's speed is followed on: what the attention parts of the supported models ask of it.

Each kind below is the sequence of public calls that one block (or block half) of a model makes per step, on operands of
that model's widths: the Stable Diffusion 1.5 U-Net and its VAE, PixArt-Sigma, Flux, Qwen-Image, Sana and Krea 2.
Image sizes run from thumbnails to the largest a user asks for, in any aspect ratio, so most token counts are no
multiple of anything. Activations are N(0, 1), weights N(0, 1) / sqrt(fan-in), biases and gains of their usual size.
Buffers that such a program keeps between steps (outputs, scratch, weights, tables, text keys and values, prefix cache)
are made once, in prepare().
"""
import torch

import brodiffusion_amd as bd

F16, BF16 = torch.float16, torch.bfloat16


def listed():
    return [
        # the deepest U-Net level at 512 x 512: a few microseconds of arithmetic, so launches and the host path are the cost
        {"name": "unet_self_8x8", "kind": "unet_self", "batch": 2, "h": 8, "w": 8, "channels": 1280, "heads": 8, "w8": False},
        # the shallowest level of the same network: the largest self-attention of a U-Net step, head_dim 40
        {"name": "unet_self_64x64", "kind": "unet_self", "batch": 2, "h": 64, "w": 64, "channels": 320, "heads": 8, "w8": False},
        # cross-attention to a 77-token prompt with the keys and values projected once per image, INT8 weights
        {"name": "unet_cross_32x32_w8", "kind": "unet_cross", "batch": 2, "h": 32, "w": 32, "channels": 640, "heads": 8, "keys": 77, "w8": True},
        # the feed-forward half of a U-Net block, 768 x 512 image
        {"name": "unet_ff_48x32", "kind": "unet_ff", "batch": 2, "h": 48, "w": 32, "channels": 640, "w8": False},
        # both attention halves of a PixArt-Sigma block at 1024 x 1024, a prompt of 120 of at most 300 tokens
        {"name": "pixart_block_64x64", "kind": "pixart_block", "h": 64, "w": 64, "channels": 1152, "heads": 16, "keys": 300, "valid": 120},
        # Flux double-stream attention at 1024 x 1024 with head norms and RoPE: the headline configuration
        {"name": "flux_joint_64x64", "kind": "flux_joint", "text": 512, "h": 64, "w": 64, "heads": 24},
        # the same at a small odd size
        {"name": "flux_joint_33x45", "kind": "flux_joint", "text": 512, "h": 33, "w": 45, "heads": 24},
        # Qwen-Image, first step: block-causal attention over [text ; reference image ; target], filling the prefix cache
        {"name": "qwen_prefill_64x64", "kind": "qwen_prefill", "text": 93, "ref_h": 24, "ref_w": 30, "h": 64, "w": 64, "heads": 24},
        # Qwen-Image, every later step: only the target rows run, the prefix comes from the cache
        {"name": "qwen_cached_40x57", "kind": "qwen_cached", "prefix": 669, "h": 40, "w": 57, "heads": 24},
        # Sana-1600M self-attention (ReLU linear attention) at 1024 x 1024, with the query / key norm of Sana-Sprint
        {"name": "sana_block_32x32", "kind": "sana_block", "h": 32, "w": 32, "heads": 20, "head_dim": 112, "qk_norm": True, "capture": False},
        # Krea 2 grouped-query attention at 1024 x 1024, the padding of the prompt hidden by a key mask
        {"name": "krea_gqa_64x64", "kind": "krea_gqa", "text": 512, "valid": 77, "h": 64, "w": 64, "heads": 48, "kv_heads": 12},
        # the VAE's mid-block for a 1024 x 1024 image: one head of 512 channels, once per image
        {"name": "vae_mid_128x128", "kind": "vae_mid", "h": 128, "w": 128, "channels": 512},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, round(lo * (hi / lo) ** rng.random())))


def draw(rng):
    most = max(_cost(c) for c in listed())
    while True:
        c = _draw(rng)
        if _cost(c) <= most:
            return c


def _draw(rng):
    kind = rng.choice(["unet_self", "unet_cross", "unet_ff", "pixart_block", "flux_joint", "qwen_prefill", "qwen_cached", "sana_block",
                       "krea_gqa", "vae_mid"])
    c = {"kind": kind}
    if kind.startswith("unet"):
        # images of 256 to 1024 pixels a side in steps of 64; the four resolutions of the network
        level = rng.randrange(4)
        c.update(batch=rng.choice([1, 2]), h=rng.randint(4, 16) * 8 >> level, w=rng.randint(4, 16) * 8 >> level,
                 channels=(320, 640, 1280, 1280)[level], w8=rng.random() < 0.4)
        if kind != "unet_ff":
            c["heads"] = 8
        if kind == "unet_cross":
            c["keys"] = 77 * rng.choice([1, 1, 2, 3])
        return c
    h = _log_int(rng, 16, 72)
    w = min(72, max(16, round(h * 2.0 ** rng.uniform(-1, 1))))
    if kind == "pixart_block":
        c.update(h=h, w=w, channels=1152, heads=16, keys=300, valid=_log_int(rng, 8, 300))
    elif kind == "flux_joint":
        c.update(text=rng.choice([256, 512, 512]), h=h, w=w, heads=24)
    elif kind == "qwen_prefill":
        c.update(text=_log_int(rng, 20, 512), ref_h=rng.randint(12, 32), ref_w=rng.randint(12, 32), h=h, w=w, heads=24)
    elif kind == "qwen_cached":
        c.update(prefix=_log_int(rng, 30, 1500), h=h, w=w, heads=24)
    elif kind == "sana_block":
        heads, head_dim = rng.choice([(20, 112), (70, 32)])
        c.update(h=h, w=w, heads=heads, head_dim=head_dim, qk_norm=rng.random() < 0.5, capture=rng.random() < 0.3)
    elif kind == "krea_gqa":
        c.update(text=512, valid=_log_int(rng, 10, 512), h=h, w=w, heads=48, kv_heads=12)
    else:
        c.update(h=rng.randint(4, 16) * 8, w=rng.randint(4, 16) * 8, channels=512)
    return c


class _Rand:
    """Operands of one case, from its seed."""

    def __init__(self, seed, dtype):
        self.g, self.dtype = torch.Generator(device="cuda").manual_seed(seed), dtype

    def __call__(self, *shape, scale=1.0, mean=0.0):
        x = torch.randn(*shape, generator=self.g, device="cuda", dtype=torch.float32)
        return (x * scale + mean).to(self.dtype)

    def weight(self, rows, cols, w8=False):
        """(weight, scales or None): INT8 with one scale per row, or of the compute type."""
        if not w8:
            return self(rows, cols, scale=cols ** -0.5), None
        x = torch.randn(rows, cols, generator=self.g, device="cuda", dtype=torch.float32) * cols ** -0.5
        s = x.abs().amax(dim=1, keepdim=True) / 127.0
        return torch.round(x / s).to(torch.int8), s


def prepare(case, seed):
    return globals()["_prepare_" + case["kind"]](case, seed)


def run(state):
    return state["run"](state)


# ── Stable Diffusion 1.5 U-Net and VAE (float16; float16 or INT8 weights) ──

def _prepare_unet_self(c, seed):
    r = _Rand(seed, F16)
    n, ch = c["h"] * c["w"], c["channels"]
    s = {"run": _run_unet_self_w8 if c["w8"] else _run_unet_self, "heads": c["heads"], "x": r(c["batch"], n, ch)}
    for p in "qkvo":
        s["w" + p], s["s" + p] = r.weight(ch, ch, c["w8"])
    s["bo"] = r(ch, scale=0.1)
    s["out"] = torch.empty_like(s["x"])
    s["scratch"] = torch.empty(bd.flash_attention_scratch_bytes(c["batch"], n, n, ch, True), dtype=torch.uint8, device="cuda")
    return s


def _run_unet_self(s):
    return bd.flash_attention_qkvo_forward(s["x"], None, s["wq"], None, s["wk"], None, s["wv"], None, s["wo"], s["bo"], None, s["heads"], False,
                                           out=s["out"], scratch=s["scratch"])


def _run_unet_self_w8(s):
    return bd.flash_attention_qkvo_int8w_fp16(s["x"], None, s["wq"], s["sq"], None, s["wk"], s["sk"], None, s["wv"], s["sv"], None,
                                              s["wo"], s["so"], s["bo"], None, s["heads"], False, out=s["out"], scratch=s["scratch"])


def _prepare_unet_cross(c, seed):
    r = _Rand(seed, F16)
    n, ch = c["h"] * c["w"], c["channels"]
    s = {"run": _run_unet_cross_w8 if c["w8"] else _run_unet_cross, "heads": c["heads"], "x": r(c["batch"], n, ch)}
    ctx = r(c["batch"], c["keys"], 768)
    for p, cols in (("q", ch), ("k", 768), ("v", 768), ("o", ch)):
        s["w" + p], s["s" + p] = r.weight(ch, cols, c["w8"])
    s["bo"] = r(ch, scale=0.1)
    if c["w8"]:
        s["k"], s["v"] = bd.flash_attention_project_kv_int8w_fp16(ctx, s["wk"], s["sk"], None, s["wv"], s["sv"], None)
    else:
        s["k"], s["v"] = bd.flash_attention_project_kv(ctx, s["wk"], None, s["wv"], None)
    s["out"] = torch.empty_like(s["x"])
    s["scratch"] = torch.empty(bd.flash_attention_scratch_bytes(c["batch"], n, c["keys"], ch, False), dtype=torch.uint8, device="cuda")
    return s


def _run_unet_cross(s):
    return bd.flash_attention_q_with_kv_cached_forward(s["x"], s["k"], s["v"], s["wq"], None, s["wo"], s["bo"], None, s["heads"], False,
                                                       out=s["out"], scratch=s["scratch"])


def _run_unet_cross_w8(s):
    return bd.flash_attention_q_with_kv_cached_int8w_fp16(s["x"], s["k"], s["v"], s["wq"], s["sq"], None, s["wo"], s["so"], s["bo"], None,
                                                          s["heads"], False, out=s["out"], scratch=s["scratch"])


def _prepare_unet_ff(c, seed):
    r = _Rand(seed, F16)
    n, ch = c["batch"] * c["h"] * c["w"], c["channels"]
    s = {"run": _run_unet_ff, "x": r(n, ch)}
    s["w1"], s["s1"] = r.weight(8 * ch, ch, c["w8"])
    s["w2"], s["s2"] = r.weight(ch, 4 * ch, c["w8"])
    s["b1"], s["b2"] = r(8 * ch, scale=0.1), r(ch, scale=0.1)
    s["y"], s["out"] = torch.empty(n, 4 * ch, dtype=F16, device="cuda"), torch.empty(n, ch, dtype=F16, device="cuda")
    return s


def _run_unet_ff(s):
    if s["s1"] is not None:
        y = bd.fused_linear_geglu_int8w(s["x"], s["w1"], s["s1"], s["b1"], s["y"])
        out = bd.linear_forward_batched_int8w_fp16(s["w2"], s["s2"], s["b2"], y, s["out"])
    else:
        y = bd.fused_linear_geglu(s["x"], s["w1"], s["b1"], s["y"])
        out = bd.linear_batched(s["w2"], s["b2"], y, s["out"])
    return bd.add_inplace_vec(out, s["x"])


def _prepare_vae_mid(c, seed):
    r = _Rand(seed, F16)
    n, ch = c["h"] * c["w"], c["channels"]
    s = {"run": _run_vae_mid, "x": r(n, ch)}
    for p in "qkvo":
        s["w" + p], s["b" + p] = r.weight(ch, ch)[0], r(ch, scale=0.1)
    s["out"] = torch.empty_like(s["x"])
    s["scratch"] = torch.empty(bd.flash_attention_scratch_bytes(1, n, n, ch, True), dtype=torch.uint8, device="cuda")
    return s


def _run_vae_mid(s):
    return bd.flash_attention_qkvo_forward(s["x"], None, s["wq"], s["bq"], s["wk"], s["bk"], s["wv"], s["bv"], s["wo"], s["bo"], None, 1, False,
                                           out=s["out"], scratch=s["scratch"])


# ── PixArt-Sigma (bfloat16) ──

def _prepare_pixart_block(c, seed):
    r = _Rand(seed, BF16)
    n, ch = c["h"] * c["w"], c["channels"]
    s = {"run": _run_pixart_block, "heads": c["heads"], "x": r(n, ch), "x2": r(n, ch)}
    for p in ("q", "k", "v", "o", "q2", "o2"):
        s["w" + p], s["b" + p] = r.weight(ch, ch)[0], r(ch, scale=0.1)
    s["kc"], s["vc"] = r(c["keys"], ch), r(c["keys"], ch)
    s["valid"] = torch.tensor([c["valid"]], dtype=torch.int32, device="cuda")
    for t in ("qh", "kh", "vh", "yc", "out", "q2", "y2", "out2"):
        s[t] = torch.empty_like(s["x"])
    return s


def _run_pixart_block(s):
    out = bd.mha_forward(s["x"], s["wq"], s["wk"], s["wv"], s["wo"], s["bq"], s["bk"], s["bv"], s["bo"], None, s["heads"],
                         qh=s["qh"], kh=s["kh"], vh=s["vh"], yc=s["yc"], out=s["out"])[0]
    q2 = bd.linear_batched(s["wq2"], s["bq2"], s["x2"], s["q2"])
    y2 = bd.sdpa_forward(q2, s["kc"], s["vc"], s["heads"], kv_valid_len=s["valid"], out=s["y2"])
    return out, bd.linear_batched(s["wo2"], s["bo2"], y2, s["out2"])


# ── Flux (bfloat16, head_dim 128) ──

def _prepare_flux_joint(c, seed):
    r = _Rand(seed, BF16)
    n, ch = c["text"] + c["h"] * c["w"], c["heads"] * 128
    s = {"run": _run_flux_joint, "heads": c["heads"], "q": r(n, ch), "k": r(n, ch), "v": r(n, ch),
         "gq": r(128, scale=0.1, mean=1.0), "gk": r(128, scale=0.1, mean=1.0)}
    s["cos"], s["sin"] = bd.build_axial_rope_tables(c["text"], c["h"], c["w"], 128, (16, 56, 56))
    for t in ("qn", "kn", "kr", "out"):
        s[t] = torch.empty_like(s["q"])
    return s


def _run_flux_joint(s):
    qn = bd.headnorm_rope(s["q"], s["gq"], 1e-6, None, None, 128, s["heads"], out=s["qn"])
    kn = bd.headnorm_rope(s["k"], s["gk"], 1e-6, None, None, 128, s["heads"], out=s["kn"])
    return bd.joint_attention(qn, kn, s["v"], s["cos"], s["sin"], 128, s["heads"], out=s["out"], Kr=s["kr"])


# ── Qwen-Image (bfloat16, head_dim 128) ──

def _prepare_qwen_prefill(c, seed):
    r = _Rand(seed, BF16)
    n_ref, n_img = c["ref_h"] * c["ref_w"], c["h"] * c["w"]
    prefix, ch = c["text"] + n_ref, c["heads"] * 128
    n = prefix + n_img
    s = {"run": _run_qwen_prefill, "heads": c["heads"], "q": r(n, ch), "k": r(n, ch), "v": r(n, ch),
         "gq": r(128, scale=0.1, mean=1.0), "gk": r(128, scale=0.1, mean=1.0)}
    s["cos"], s["sin"] = bd.build_qwen_rope_tables([("text", c["text"]), ("image", c["ref_h"], c["ref_w"])], c["h"], c["w"], 128)
    ends = [c["text"], prefix, n]
    s["mask"] = bd.SdpaMask.block_causal(0, ends, ends, [1, 0, 0])
    s["cache"] = torch.empty(prefix, ch, dtype=BF16, device="cuda")
    for t in ("qr", "kr", "out"):
        s[t] = torch.empty_like(s["q"])
    return s


def _run_qwen_prefill(s):
    qr = bd.headnorm_rope(s["q"], s["gq"], 1e-6, s["cos"], s["sin"], 128, s["heads"], out=s["qr"])
    kr = bd.headnorm_rope(s["k"], s["gk"], 1e-6, s["cos"], s["sin"], 128, s["heads"], out=s["kr"], cache_out=s["cache"])
    return bd.sdpa_forward(qr, kr, s["v"], s["heads"], mask=s["mask"], out=s["out"]), s["cache"]


def _prepare_qwen_cached(c, seed):
    r = _Rand(seed, BF16)
    n, prefix, ch = c["h"] * c["w"], c["prefix"], c["heads"] * 128
    s = {"run": _run_qwen_cached, "heads": c["heads"], "q": r(n, ch), "k": r(n, ch), "v": r(n, ch), "kp": r(prefix, ch), "vp": r(prefix, ch),
         "gq": r(128, scale=0.1, mean=1.0), "gk": r(128, scale=0.1, mean=1.0)}
    cos, sin = bd.build_qwen_rope_tables([("text", prefix)], c["h"], c["w"], 128)
    s["cos"], s["sin"] = cos[prefix:].contiguous(), sin[prefix:].contiguous()
    for t in ("qr", "kr", "out"):
        s[t] = torch.empty_like(s["q"])
    return s


def _run_qwen_cached(s):
    qr = bd.headnorm_rope(s["q"], s["gq"], 1e-6, s["cos"], s["sin"], 128, s["heads"], out=s["qr"])
    kr = bd.headnorm_rope(s["k"], s["gk"], 1e-6, s["cos"], s["sin"], 128, s["heads"], out=s["kr"])
    return bd.sdpa_forward(qr, kr, s["v"], s["heads"], k_prefix=s["kp"], v_prefix=s["vp"], out=s["out"])


# ── Sana (bfloat16) ──

def _prepare_sana_block(c, seed):
    r = _Rand(seed, BF16)
    n, ch = c["h"] * c["w"], c["heads"] * c["head_dim"]
    s = {"run": _run_sana_block, "heads": c["heads"], "x": r(n, ch), "bo": r(ch, scale=0.1), "nq": None, "nk": None, "state": None}
    for p in "qkvo":
        s["w" + p] = r.weight(ch, ch)[0]
    if c["qk_norm"]:
        s["nq"], s["nk"] = r(ch, scale=0.1, mean=1.0), r(ch, scale=0.1, mean=1.0)
    if c["capture"]:
        s["state"] = torch.empty(c["heads"] * (c["head_dim"] + 1) * c["head_dim"], dtype=torch.float32, device="cuda")
    s["out"] = torch.empty_like(s["x"])
    return s


def _run_sana_block(s):
    out = bd.sana_self_attention(s["x"], s["wq"], s["wk"], s["wv"], s["wo"], s["bo"], s["heads"], nq=s["nq"], nk=s["nk"],
                                 ref_mode="off" if s["state"] is None else "capture", ref_state=s["state"], out=s["out"])
    return out if s["state"] is None else (out, s["state"])


# ── Krea 2 (bfloat16, head_dim 128) ──

def _prepare_krea_gqa(c, seed):
    r = _Rand(seed, BF16)
    n = c["text"] + c["h"] * c["w"]
    s = {"run": _run_krea_gqa, "heads": c["heads"], "kv_heads": c["kv_heads"], "q": r(n, c["heads"] * 128),
         "k": r(n, c["kv_heads"] * 128), "v": r(n, c["kv_heads"] * 128)}
    s["cos"], s["sin"] = bd.build_axial_rope_tables(c["text"], c["h"], c["w"], 128, (16, 56, 56))
    s["mask"] = torch.ones(n, dtype=torch.float32, device="cuda")
    s["mask"][c["valid"]:c["text"]] = 0
    s["kr"], s["out"] = torch.empty_like(s["k"]), torch.empty_like(s["q"])
    return s


def _run_krea_gqa(s):
    return bd.gqa_attention_masked(s["q"], s["k"], s["v"], s["cos"], s["sin"], 128, s["heads"], s["kv_heads"], s["mask"], out=s["out"], Kr=s["kr"])


def work(case):
    """Bytes of the operands and results (weights, tables and caches included, intermediates not) and multiply-add FLOPs
    (two per multiply-add; projections and visible query-key pairs) of one pass."""
    k = case["kind"]
    if k in ("unet_self", "vae_mid"):
        b, n, ch = case.get("batch", 1), case["h"] * case["w"], case["channels"]
        return {"bytes": 4 * b * n * ch + 4 * ch * ch * (1 if case.get("w8") else 2), "flops": b * (8 * n * ch * ch + 4 * n * n * ch)}
    if k == "unet_cross":
        b, n, ch, keys = case["batch"], case["h"] * case["w"], case["channels"], case["keys"]
        return {"bytes": 4 * b * n * ch + 4 * b * keys * ch + 2 * ch * ch * (1 if case["w8"] else 2), "flops": b * (4 * n * ch * ch + 4 * n * keys * ch)}
    if k == "unet_ff":
        n, ch = case["batch"] * case["h"] * case["w"], case["channels"]
        return {"bytes": 4 * n * ch + 12 * ch * ch * (1 if case["w8"] else 2), "flops": 24 * n * ch * ch}
    if k == "pixart_block":
        n, ch, keys = case["h"] * case["w"], case["channels"], case["valid"]
        return {"bytes": 8 * n * ch + 12 * ch * ch + 4 * keys * ch, "flops": 12 * n * ch * ch + 4 * n * n * ch + 4 * n * keys * ch}
    if k == "flux_joint":
        n, ch = case["text"] + case["h"] * case["w"], case["heads"] * 128
        return {"bytes": 8 * n * ch + 512 * n, "flops": 4 * n * n * ch}
    if k == "qwen_prefill":
        t, ref, img, ch = case["text"], case["ref_h"] * case["ref_w"], case["h"] * case["w"], case["heads"] * 128
        n = t + ref + img
        pairs = t * (t + 1) // 2 + ref * (t + ref) + img * n
        return {"bytes": 8 * n * ch + 2 * (t + ref) * ch + 512 * n, "flops": 4 * pairs * ch}
    if k == "qwen_cached":
        n, prefix, ch = case["h"] * case["w"], case["prefix"], case["heads"] * 128
        return {"bytes": 8 * n * ch + 4 * prefix * ch + 512 * n, "flops": 4 * n * (n + prefix) * ch}
    if k == "sana_block":
        n, ch, d = case["h"] * case["w"], case["heads"] * case["head_dim"], case["head_dim"]
        return {"bytes": 4 * n * ch + 8 * ch * ch, "flops": 8 * n * ch * ch + 4 * n * ch * d}
    n, ch, keys = case["text"] + case["h"] * case["w"], case["heads"] * 128, case["valid"] + case["h"] * case["w"]
    return {"bytes": 4 * n * ch + 4 * n * case["kv_heads"] * 128 + 512 * n, "flops": 4 * n * keys * ch}


def _cost(case):
    w = work(case)
    return w["flops"] + 300 * w["bytes"]


def tolerance(case):
    """Two correct implementations round the operands of the matrix products, the probabilities and every intermediate
    tensor once to the compute type: 2^-12 (float16) or 2^-9 (bfloat16) relative each, a handful of them in sequence."""
    return {"rel": 2e-3} if case["kind"].startswith(("unet", "vae")) else {"rel": 1e-2}
