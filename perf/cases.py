"""The calls that a program makes of this framework, one pass of each, with their inputs and their 64-bit results.

Every case is one call (or the two or three calls of a block) through the public entry points, as a serving loop
makes them: a decode step of a whole model, a prompt read into the cache, a tree of drafts verified, and the single
operators of a decoder layer for programs that build their own loop.  Weights are random N(0, 0.02) (ternary ones in
{-1, 0, 1}) and packed by the framework's own packers; activations and cached keys and values are N(0, 1).
"""

from __future__ import annotations

import math

import torch

from axiomlm_amd.cache import StaticKVCache
from axiomlm_amd.kernels import (gqa_flash_decode_mps, pack_linear_q2_k, pack_linear_q2_k_gguf, pack_linear_q4_marlin,
                                 pack_linear_q8_g64, pack_linear_ternary, qmm_q4_marlin, qmv_q2_k, qmv_q2_k_gguf,
                                 qmv_q4_tile16, qmv_q4_tile16_swiglu, qmv_q8_g64, qmv_ternary, quantize_kv_fp8,
                                 quantize_kv_int4, repack_q4_marlin_tile16)
from axiomlm_amd.runner import DecodeRunner, QuantizedDecodeRunner
from axiomlm_amd.transformer import ModelConfig, Transformer

EPS = 1e-5
THETA = 10000.0
# (heads, KV heads, head size, MLP width, vocabulary): the small test model, the 7B shape of the benchmark, and the
# 7B shape with the grouped-query heads of the attention benchmark.
SHAPES = {"c1": (4, 4, 64, 704, 1024), "7b": (32, 32, 128, 11008, 32000), "gqa": (32, 8, 128, 11008, 32000)}
BYTES_PER_WEIGHT = {"q4": 0.5625, "q4_g128": 0.53125, "q4_marlin": 0.5625, "q4_tile16": 0.5625, "q8": 1.0625,
                    "fp16": 2.0, "ternary": 0.28125, "q2_k": 0.3125, "gguf": 84 / 256}
KV_BYTES = {"fp16": lambda hd: 2 * hd, "fp8": lambda hd: hd + hd // 32, "int4": lambda hd: hd // 2 + hd // 32}


def listed():
    return [
        # One token of the small test model: 20-odd short launches, where latency is everything.
        {"name": "step_small", "kind": "step", "shape": "c1", "layers": 4, "fmt": "q4", "kv": "fp16", "past": 100},
        # The headline: one token of the whole 7B model, MARLIN Q4 group 128, some hundred tokens into a chat.
        {"name": "step_7b", "kind": "step", "shape": "7b", "layers": 32, "fmt": "q4_g128", "kv": "fp16", "past": 600},
        # A long conversation on a grouped-query model with the mixed Q4 / Q8 weights and an FP8 cache (8 layers).
        {"name": "step_gqa_long", "kind": "step", "shape": "gqa", "layers": 8, "fmt": "q4_k_m", "kv": "fp8",
         "past": 6007},
        # A prompt of a page or two read into the cache (4 layers of the 7B shape, head, and the last token's logits).
        {"name": "prompt_7b", "kind": "prompt", "shape": "7b", "layers": 4, "fmt": "q4", "kv": "fp16", "T": 1000,
         "past": 0},
        # The next, short message of a conversation: Q8 weights, grouped heads, FP8 cache with the earlier turns in it.
        {"name": "prompt_q8_turn", "kind": "prompt", "shape": "gqa", "layers": 4, "fmt": "q8", "kv": "fp8", "T": 75,
         "past": 700},
        # Speculative decoding: a tree of 64 drafts verified against 2048 cached tokens (FP8 cache, 4 layers).
        {"name": "tree_64", "kind": "tree", "shape": "7b", "layers": 4, "fmt": "q4", "kv": "fp8", "T": 64,
         "past": 2048},
        # The MLP of a decoder layer for 16 tokens (a small batch, or a chain of drafts).
        {"name": "mlp_16", "kind": "mlp", "d": 4096, "hidden": 11008, "group": 64, "M": 16},
        # The QKV projection of a long prompt.
        {"name": "linear_q4_1024", "kind": "linear", "fmt": "q4_tile16", "M": 1024, "N": 12288, "K": 4096,
         "bias": False},
        # The 2-bit formats' feed-forward projection: one token, and the tokens of a short prompt.
        {"name": "linear_ternary_1", "kind": "linear", "fmt": "ternary", "M": 1, "N": 11008, "K": 4096,
         "bias": False},
        {"name": "linear_gguf_40", "kind": "linear", "fmt": "gguf", "M": 40, "N": 4096, "K": 11008, "bias": False},
        # Decode attention of a batch of long sequences over an INT4 cache.
        {"name": "attn_int4_8k", "kind": "attn", "B": 8, "heads": 32, "kv_heads": 8, "hd": 128, "kv": "int4",
         "len": 8192},
        # Decode attention of one sequence, one KV head per head, over an fp16 cache; an odd length.
        {"name": "attn_fp16_1", "kind": "attn", "B": 1, "heads": 32, "kv_heads": 32, "hd": 128, "kv": "fp16",
         "len": 3001},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["step", "prompt", "tree", "mlp", "linear", "linear", "attn"])
    if kind == "step":
        shape = rng.choice(["c1", "7b", "gqa"])
        fmt = rng.choice(["q4", "q4_g128", "q4_k_m", "q8", "fp16"] if shape != "c1" else ["q4", "q8", "fp16"])
        kv = rng.choice(["fp16", "fp8", "int4"])
        # (INT4 rows differ by a seventh of their largest value where a rounding falls the other way: with few
        # cached rows that is all of the result.)
        return {"kind": kind, "shape": shape, "layers": rng.randint(2, 8), "fmt": fmt, "kv": kv,
                "past": _log(rng, 500 if kv == "int4" else 1, 12000)}
    if kind == "prompt":
        return {"kind": kind, "shape": rng.choice(["c1", "7b", "gqa"]), "layers": rng.randint(2, 4),
                "fmt": rng.choice(["q4", "q8", "fp16"]), "kv": rng.choice(["fp16", "fp8"]),
                "T": _log(rng, 2, 1000), "past": rng.choice([0, _log(rng, 1, 2000)])}
    if kind == "tree":
        return {"kind": kind, "shape": rng.choice(["c1", "7b", "gqa"]), "layers": rng.randint(2, 4),
                "fmt": rng.choice(["q4", "q8"]), "kv": rng.choice(["fp16", "fp8"]), "T": rng.randint(2, 64),
                "past": _log(rng, 16, 4000)}
    if kind == "mlp":
        d, hidden = rng.choice([(4096, 11008), (2048, 5632), (256, 704)])
        return {"kind": kind, "d": d, "hidden": hidden, "group": 64 if d == 256 else rng.choice([64, 128]),
                "M": _log(rng, 1, 1024)}
    if kind == "linear":
        fmt = rng.choice(["q4_marlin", "q4_tile16", "q8", "ternary", "q2_k", "gguf"])
        return {"kind": kind, "fmt": fmt, "M": _log(rng, 1, 1024),
                "N": rng.choice([12288, 11008, 4096, 2048, 1000, 8 * rng.randint(20, 1200)]),
                "K": rng.choice([4096, 11008, 2048, 256 * rng.randint(1, 20)]), "bias": rng.random() < 0.3}
    heads, kv_heads, hd = rng.choice([(32, 8, 128), (32, 32, 128), (4, 4, 64), (32, 4, 64)])
    length = _log(rng, 16, 32768)
    return {"kind": kind, "B": rng.randint(1, max(1, min(8, 65536 // length))), "heads": heads, "kv_heads": kv_heads,
            "hd": hd, "kv": rng.choice(["fp16", "fp8", "int4"]), "len": length}


# ---- inputs ---------------------------------------------------------------------------------------------------------
class _Rand:
    def __init__(self, seed):
        self.dev = torch.device("cuda", torch.cuda.current_device())
        self.g = torch.Generator(device=self.dev)
        self.g.manual_seed(int(seed))

    def normal(self, *shape, std=1.0):
        return (torch.randn(*shape, generator=self.g, device=self.dev) * std).half()

    def norm_weight(self, n):
        return (1.0 + 0.1 * torch.randn(n, generator=self.g, device=self.dev)).half()

    def ints(self, high, *shape):
        return torch.randint(0, high, shape, generator=self.g, device=self.dev)

    def ternary(self, N, K):
        return (torch.randint(0, 4, (N, K), generator=self.g, device=self.dev) % 3 - 1).half() * 0.02


def _kind_fmt(fmt, name):
    """Format of one kind of matrix in a model of mode fmt (q4_k_m: Q8 down projection and head)."""
    if fmt == "q4_k_m":
        return "q8" if name in ("dn", "head") else "q4"
    return fmt


def _pack(fmt, w):
    if fmt == "fp16":
        return w, None
    if fmt == "q8":
        return pack_linear_q8_g64(w)
    return pack_linear_q4_marlin(w, clip_search=False, group_size=128 if fmt == "q4_g128" else 64)


def _rope(hd, n):
    inv = 1.0 / (THETA ** (torch.arange(0, hd, 2, dtype=torch.int64).float() / hd))
    a = torch.outer(torch.arange(n, dtype=torch.float32), inv)
    return torch.view_as_real(torch.polar(torch.ones_like(a), a)).contiguous()


def _matrices(case):
    heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
    d = heads * hd
    return d, hidden, vocab, {"qkv": ((heads + 2 * kvh) * hd, d), "o": (d, d), "gu": (2 * hidden, d),
                              "dn": (d, hidden)}


def _model(case, seed, keep_fp16):
    """Weights (fp16, or packed), cache and tokens of a model case, from the seed alone."""
    r = _Rand(seed)
    heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
    d, hidden, vocab, mats = _matrices(case)
    m = {"layers": []}
    for _ in range(case["layers"]):
        lay = {"ln1": r.norm_weight(d), "ln2": r.norm_weight(d)}
        for k, (n, kk) in mats.items():
            w = r.normal(n, kk, std=0.02)
            lay[k] = w if keep_fp16 else _pack(_kind_fmt(case["fmt"], k), w)
        m["layers"].append(lay)
    head, wte = r.normal(vocab, d, std=0.02), r.normal(vocab, d, std=0.02)
    m["head"] = head if keep_fp16 else _pack(_kind_fmt(case["fmt"], "head"), head)
    m["wte"] = wte if (keep_fp16 or case["fmt"] == "fp16") else pack_linear_q8_g64(wte)
    m["lnf"] = r.norm_weight(d)
    T, past = case.get("T", 1), case["past"]
    S = (past + T + 63) // 64 * 64 + 64
    m["S"], m["freqs"] = S, _rope(hd, S).to(r.dev)
    cache = StaticKVCache(1, S, case["layers"], kvh, hd, device=r.dev, cache_dtype=case["kv"])
    cache.cache.zero_()
    for i in range(case["layers"]):
        k, v = r.normal(1, kvh, S, hd), r.normal(1, kvh, S, hd)
        if case["kv"] == "fp16":
            cache.cache[i, 0].copy_(k)
            cache.cache[i, 1].copy_(v)
        else:
            kc, ks, vc, vs = (quantize_kv_fp8 if case["kv"] == "fp8" else quantize_kv_int4)(k, v)
            for j, (c, s) in enumerate(((kc, ks), (vc, vs))):
                cache.cache[i, j].copy_(c)
                cache.scales[i, j].copy_(s)
    m["cache"] = cache
    m["tokens"] = r.ints(vocab, 1, T)
    parent = [0] + [int(x) for x in (torch.rand(T, generator=torch.Generator().manual_seed(int(seed)))[1:]
                                     * torch.arange(1, T)).long()]
    depth, mask = [0] * T, [1] * T
    for u in range(1, T):  # a random tree: every node hangs off an earlier one
        depth[u], mask[u] = depth[parent[u]] + 1, mask[parent[u]] | (1 << u)
    m["depth"], m["mask"] = depth, mask
    return m


def _runner(case, m):
    heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
    P = lambda k: [lay[k][0] for lay in m["layers"]]  # noqa: E731
    S = lambda k: [lay[k][1] for lay in m["layers"]]  # noqa: E731
    ln1, ln2 = [lay["ln1"] for lay in m["layers"]], [lay["ln2"] for lay in m["layers"]]
    c = m["cache"]
    kv = dict(k_scales=c.k_scales, v_scales=c.v_scales, kv_dtype=case["kv"])
    if case["fmt"] == "fp16":
        return DecodeRunner(m["wte"], m["freqs"], ln1, P("qkv"), P("o"), ln2, P("gu"), P("dn"), m["lnf"], c.k_caches,
                            c.v_caches, heads, kvh, hd, EPS, lm_head_w=m["head"][0], max_tokens=64, **kv)
    return QuantizedDecodeRunner(None, m["head"][0], m["head"][1], m["freqs"], ln1, P("qkv"), S("qkv"), P("o"), S("o"),
                                 ln2, P("gu"), S("gu"), P("dn"), S("dn"), m["lnf"], c.k_caches, c.v_caches, heads, kvh,
                                 hd, case["fmt"] != "q8", EPS, [], vocab, wte_p=m["wte"][0], wte_s=m["wte"][1],
                                 max_tokens=64, **kv)


def _transformer(case, m):
    heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
    sd = {"transformer.wte.weight": m["wte"], "lm_head.weight": m["head"], "transformer.ln_f.weight": m["lnf"]}
    for i, lay in enumerate(m["layers"]):
        pre = f"transformer.h.{i}."
        sd.update({pre + "ln_1.weight": lay["ln1"], pre + "ln_2.weight": lay["ln2"],
                   pre + "attn.c_attn.weight": lay["qkv"], pre + "attn.c_proj.weight": lay["o"],
                   pre + "mlp.w_gate.weight": lay["gu"][:hidden], pre + "mlp.w_up.weight": lay["gu"][hidden:],
                   pre + "mlp.w_down.weight": lay["dn"]})
    cfg = ModelConfig(block_size=m["S"], vocab_size=vocab, n_layer=case["layers"], n_head=heads, n_embd=heads * hd,
                      n_kv_head=kvh, rope_theta=THETA, intermediate_size=hidden, rms_norm_eps=EPS,
                      tie_word_embeddings=False)
    model = Transformer(cfg, sd, device=m["freqs"].device)
    model.quantize({"q4": "q4_rtn", "q8": "q8", "fp16": None}[case["fmt"]])
    model.get_decode_runner(m["cache"])
    return model


def _linear_weight(case, r):
    N, K, fmt = case["N"], case["K"], case["fmt"]
    if fmt == "ternary":
        return pack_linear_ternary(r.ternary(N, K))
    w = r.normal(N, K, std=0.02)
    if fmt == "q8":
        return pack_linear_q8_g64(w)
    if fmt == "q2_k":
        return pack_linear_q2_k(w)
    if fmt == "gguf":
        return (pack_linear_q2_k_gguf(w),)
    return pack_linear_q4_marlin(w, clip_search=False)


def _attn_cache(case, r):
    k = r.normal(case["B"], case["kv_heads"], case["len"], case["hd"])
    v = r.normal(case["B"], case["kv_heads"], case["len"], case["hd"])
    if case["kv"] == "fp16":
        return k, None, v, None
    return (quantize_kv_fp8 if case["kv"] == "fp8" else quantize_kv_int4)(k, v)


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("step", "tree"):
        m = _model(case, seed, False)
        return {"case": case, "runner": _runner(case, m), "cache": m["cache"], "tokens": m["tokens"],
                "depth": m["depth"], "mask": m["mask"], "keep": m}
    if kind == "prompt":
        m = _model(case, seed, True)
        return {"case": case, "model": _transformer(case, m), "cache": m["cache"], "tokens": m["tokens"]}
    r = _Rand(seed)
    if kind == "mlp":
        d, H = case["d"], case["hidden"]
        s = {"case": case, "x": r.normal(case["M"], d), "ln": r.norm_weight(d)}
        for k, (n, kk) in (("gu", (2 * H, d)), ("dn", (d, H))):
            s[k] = repack_q4_marlin_tile16(*pack_linear_q4_marlin(r.normal(n, kk, std=0.02), clip_search=False,
                                                                  group_size=case["group"]), n, kk)
        return s
    if kind == "linear":
        s = {"case": case, "x": r.normal(case["M"], case["K"]), "w": _linear_weight(case, r)}
        s["bias"] = r.normal(case["N"], std=0.1) if case["bias"] else None
        if case["fmt"] == "q4_tile16":
            s["w"] = repack_q4_marlin_tile16(*s["w"], case["N"], case["K"])
        return s
    kc, ks, vc, vs = _attn_cache(case, r)
    return {"case": case, "q": r.normal(case["B"], case["heads"], 1, case["hd"]), "k": kc, "v": vc, "ks": ks, "vs": vs}


# ---- one pass -------------------------------------------------------------------------------------------------------
class _Outputs(dict):
    """Outputs of a model's pass.  The logits are a view of a buffer that the runner owns and frees with itself, so
    whoever holds them holds the runner too."""

    def __init__(self, state, **outputs):
        super().__init__(outputs)
        self.state = state


def _written(case, cache, past, T):
    """The cache rows that a pass wrote (FP8 codes as the numbers that they stand for)."""
    c = cache.cache[:, :, 0, :, past:past + T]
    if case["kv"] == "fp16":
        return {"kv": c}
    if case["kv"] == "fp8":
        c = c.view(torch.float8_e4m3fn)
    else:
        c = None  # INT4 codes: pairs of nibbles, no numbers by themselves
    return {"kv": c, "kv_scales": cache.scales[:, :, 0, :, past:past + T]}


def run(state):
    case, kind = state["case"], state["case"]["kind"]
    if kind == "step":
        past = case["past"]
        logits = state["runner"].step(state["tokens"], past, past, past + 1)
        return _Outputs(state, logits=logits, **_written(case, state["cache"], past, 1))
    if kind == "tree":
        past = case["past"]
        logits = state["runner"].verify_tree_step(state["tokens"], past, past, past, state["depth"], state["mask"])
        return _Outputs(state, logits=logits, **_written(case, state["cache"], past, case["T"]))
    if kind == "prompt":
        past, cache = case["past"], state["cache"]
        cache.total_seen_tokens[:] = [past] * cache.n_layer
        cache.layer_seq_lens[:] = [past] * cache.n_layer
        logits = state["model"].forward(state["tokens"], kv_caches=cache)[0]
        return _Outputs(state, logits=logits, **_written(case, cache, past, case["T"]))
    if kind == "mlp":
        h = qmv_q4_tile16_swiglu(state["x"], state["ln"], EPS, *state["gu"], case["hidden"])
        return [h, qmv_q4_tile16(h, *state["dn"], case["d"])]
    if kind == "linear":
        x, w, b, fmt = state["x"], state["w"], state["bias"], case["fmt"]
        if fmt == "q4_marlin":
            return qmm_q4_marlin(x, *w, case["N"], b)
        if fmt == "q4_tile16":
            return qmv_q4_tile16(x, *w, case["N"], b)
        return {"q8": qmv_q8_g64, "ternary": qmv_ternary, "q2_k": qmv_q2_k, "gguf": qmv_q2_k_gguf}[fmt](x, *w, b)
    return gqa_flash_decode_mps(state["q"], state["k"], state["v"], case["len"], 0, state["ks"], state["vs"],
                                case["kv"])


def work(case):
    kind = case["kind"]
    if kind in ("step", "tree", "prompt"):
        heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
        d, hidden, vocab, mats = _matrices(case)
        T, past, L = case.get("T", 1), case["past"], case["layers"]
        head_rows = T if kind == "tree" else 1
        b = vocab * d * BYTES_PER_WEIGHT[_kind_fmt(case["fmt"], "head")] + 2 * head_rows * vocab
        f = 2.0 * head_rows * vocab * d
        for k, (n, kk) in mats.items():
            b += L * n * kk * BYTES_PER_WEIGHT[_kind_fmt(case["fmt"], k)]
            f += 2.0 * T * L * n * kk
        b += L * 2 * kvh * (past + 2 * T) * KV_BYTES[case["kv"]](hd)
        f += L * 4.0 * heads * hd * (T * past + T * (T + 1) / 2)
        return {"bytes": b, "flops": f}
    if kind == "mlp":
        M, d, H = case["M"], case["d"], case["hidden"]
        w = 3 * d * H * (0.5625 if case["group"] == 64 else 0.53125)
        return {"bytes": w + 2 * M * (2 * d + 2 * H), "flops": 6.0 * M * d * H}
    if kind == "linear":
        M, N, K = case["M"], case["N"], case["K"]
        return {"bytes": N * K * BYTES_PER_WEIGHT[case["fmt"]] + 2 * M * (N + K), "flops": 2.0 * M * N * K}
    B, n, hd = case["B"], case["len"], case["hd"]
    return {"bytes": B * (2 * case["kv_heads"] * n * KV_BYTES[case["kv"]](hd) + 4 * case["heads"] * hd),
            "flops": 4.0 * B * case["heads"] * n * hd}


def tolerance(case):
    """fp16 activations between the layers of a model and fp16 results of a single operator (2^-11 each, and a
    few of them); FP8 rows written by a model move by a whole code where the value lies at a rounding boundary."""
    kind = case["kind"]
    if kind in ("step", "tree", "prompt"):
        return {"rel": 0.01 if case["kv"] == "fp16" else 0.03, "max": 0.3}
    if kind == "mlp":
        return {"rel": 3e-3, "max": 0.02}
    return {"rel": 1.2e-3, "max": 8e-3}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------
def _marlin_codes(p):
    """4-bit codes [N][K] of a MARLIN pack int32 [N/8][K/64][32 lanes][2]: column k = 64 g + 32 j + 8 s + r of row c
    of a tile is nibble s of half c % 2 of word j of the lane that holds (r, c - c % 2)."""
    nt, KG = p.shape[:2]
    dev = p.device
    r, c = torch.meshgrid(torch.arange(8, device=dev), torch.arange(8, device=dev), indexing="ij")
    lane = ((r >> 2) << 4) | ((c >> 2) << 3) | ((r & 3) << 1) | ((c >> 1) & 1)
    w = p.to(torch.int64)[:, :, lane]  # [nt][KG][r][c][j]
    half = (16 * (c & 1))[None, None, :, :, None]
    out = torch.stack([(w >> (half + 4 * s)) & 15 for s in range(4)], dim=-1)  # [nt][KG][r][c][j][s]
    return out.permute(0, 3, 1, 4, 5, 2).reshape(nt * 8, KG * 64)


def _decode(fmt, packed, N):
    if fmt == "fp16":
        return packed[0].double()
    if fmt in ("q4", "q4_g128", "q4_marlin", "q4_tile16"):
        q = _marlin_codes(packed[0]).double()
        sb = packed[1].double().transpose(1, 2).reshape(q.shape[0], -1, 2)
        q = q.reshape(q.shape[0], sb.shape[1], -1)
        return (q * sb[..., 0:1] + sb[..., 1:2]).reshape(q.shape[0], -1)[:N]
    if fmt == "q8":
        q = packed[0].contiguous().view(torch.uint8).reshape(N, -1, 64).double()
        sb = packed[1].double()
        return (q * sb[..., 0:1] + sb[..., 1:2]).reshape(N, -1)
    if fmt == "gguf":
        b = packed[0]
        e = torch.arange(256, device=b.device)
        q = (b[..., 16:80][..., 32 * (e // 128) + e % 32] >> (2 * ((e // 32) % 4)).to(torch.uint8)) & 3
        sc = b[..., :16][..., e // 16]
        d = b[..., 80:82].contiguous().view(torch.float16).double()
        dmin = b[..., 82:84].contiguous().view(torch.float16).double()
        return (d * (sc & 15).double() * q.double() - dmin * (sc >> 4).double()).reshape(N, -1)
    codes = torch.stack([(packed[0] >> (2 * j)) & 3 for j in range(4)], dim=-1).reshape(N, -1, 64)
    if fmt == "ternary":
        q = (codes == 1).double() - (codes == 2).double()
        return (q * packed[1].double()[..., None]).reshape(N, -1)
    return (codes.double() * packed[1].double()[..., 0:1] + packed[1].double()[..., 1:2]).reshape(N, -1)


def _kv_values(codes, scales, kv):
    if kv == "fp16":
        return codes.double()
    if kv == "fp8":
        q = codes.view(torch.float8_e4m3fn).double()
    else:
        q = torch.stack([codes & 15, codes >> 4], dim=-1).reshape(*codes.shape[:-1], -1).double()
        q = torch.where(q > 7, q - 16, q)
    return (q.reshape(*q.shape[:-1], -1, 64) * scales.double()[..., None]).reshape(q.shape)


def _kv_round(x, kv):
    """What a cache of type kv keeps of the rows x."""
    if kv == "fp16":
        return x
    g = x.reshape(*x.shape[:-1], -1, 64)
    s = (g.abs().amax(-1, keepdim=True) / (448.0 if kv == "fp8" else 7.0)).half().double()
    q = g / s
    q = q.float().to(torch.float8_e4m3fn).double() if kv == "fp8" else q.round().clamp(-8, 7)
    return (q * s).reshape(x.shape)


def _attend(q, k, v, visible=None):
    """q [T][Hq][hd], k and v [Hkv][n][hd], visible [T][n] -> [T][Hq][hd]."""
    T, Hq, hd = q.shape
    rep = Hq // k.shape[0]
    out = torch.empty_like(q)
    for h in range(k.shape[0]):
        qh = q[:, h * rep:(h + 1) * rep].reshape(T * rep, hd)
        s = (qh @ k[h].T.contiguous()) / math.sqrt(hd)
        if visible is not None:
            s = s.masked_fill(~visible.repeat_interleave(rep, 0), -math.inf)
        out[:, h * rep:(h + 1) * rep] = (torch.softmax(s, -1) @ v[h]).reshape(T, rep, hd)
    return out


def _rms(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _exact_model(case, seed):
    m = _model(case, seed, case["kind"] == "prompt")
    heads, kvh, hd, hidden, vocab = SHAPES[case["shape"]]
    d, hidden, vocab, mats = _matrices(case)
    T, past, kv, fmt, tok = case.get("T", 1), case["past"], case["kv"], case["fmt"], m["tokens"][0]
    dev = tok.device

    def weight(name, w, n):
        f = _kind_fmt(fmt, name)
        return _decode(f, _pack(f, w) if case["kind"] == "prompt" else w, n)

    if fmt == "fp16":
        x = m["wte"][tok].double()
    else:
        p, s = pack_linear_q8_g64(m["wte"]) if case["kind"] == "prompt" else m["wte"]
        x = _decode("q8", (p[tok], s[tok]), T)
    ar = torch.arange(T, device=dev)
    if case["kind"] == "tree":
        pos = past + torch.tensor(m["depth"], device=dev)
        vis = torch.tensor([[bool((b >> j) & 1) for j in range(T)] for b in m["mask"]], device=dev)
    else:
        pos, vis = past + ar, ar[None, :] <= ar[:, None]
    vis = torch.cat([torch.ones(T, past, dtype=torch.bool, device=dev), vis], 1)
    f = m["freqs"][pos].double()
    rot = torch.complex(f[..., 0], f[..., 1])[:, None, :]

    def rope(t):
        return torch.view_as_real(torch.view_as_complex(t.reshape(*t.shape[:-1], -1, 2).contiguous()) * rot).reshape(
            t.shape)

    c, rows = m["cache"], []
    for i, lay in enumerate(m["layers"]):
        y = _rms(x, lay["ln1"]) @ weight("qkv", lay["qkv"], mats["qkv"][0]).T
        q, k, v = (t.reshape(T, -1, hd) for t in y.split([d, kvh * hd, kvh * hd], 1))
        k, v = rope(k).transpose(0, 1).contiguous(), v.transpose(0, 1).contiguous()
        rows.append(torch.stack([k, v]))
        old = [_kv_values(c.cache[i, j, 0, :, :past], None if kv == "fp16" else c.scales[i, j, 0, :, :past], kv)
               for j in range(2)]
        a = _attend(rope(q), torch.cat([old[0], _kv_round(k, kv)], 1), torch.cat([old[1], _kv_round(v, kv)], 1), vis)
        x = x + a.reshape(T, d) @ weight("o", lay["o"], d).T
        y = _rms(x, lay["ln2"]) @ weight("gu", lay["gu"], 2 * hidden).T
        x = x + (torch.nn.functional.silu(y[:, :hidden]) * y[:, hidden:]) @ weight("dn", lay["dn"], d).T
    if case["kind"] == "prompt":
        x = x[-1:]
    logits = (_rms(x, m["lnf"]) @ weight("head", m["head"], vocab).T)[None]
    if kv == "fp16":
        return {"logits": logits, "kv": torch.stack(rows)}
    return {"logits": logits, "kv": None, "kv_scales": None}


def exact(case, seed):
    kind = case["kind"]
    if kind in ("step", "tree", "prompt"):
        return _exact_model(case, seed)
    r = _Rand(seed)
    if kind == "mlp":
        d, H, g = case["d"], case["hidden"], case["group"]
        x, ln = r.normal(case["M"], d), r.norm_weight(d)
        w = [_decode("q4", pack_linear_q4_marlin(r.normal(n, kk, std=0.02), clip_search=False, group_size=g), n)
             for n, kk in ((2 * H, d), (d, H))]
        y = _rms(x.double(), ln) @ w[0].T
        h = torch.nn.functional.silu(y[:, :H]) * y[:, H:]
        return [h, h @ w[1].T]
    if kind == "linear":
        x, w = r.normal(case["M"], case["K"]), _linear_weight(case, r)
        y = x.double() @ _decode(case["fmt"], w, case["N"]).T
        return y + r.normal(case["N"], std=0.1).double() if case["bias"] else y
    kc, ks, vc, vs = _attn_cache(case, r)
    q = r.normal(case["B"], case["heads"], 1, case["hd"]).double()
    return torch.stack([
        _attend(q[b].transpose(0, 1), _kv_values(kc[b], None if ks is None else ks[b], case["kv"]),
                _kv_values(vc[b], None if vs is None else vs[b], case["kv"])).transpose(0, 1)
        for b in range(case["B"])])
