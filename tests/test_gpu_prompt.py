"""Prompts read in one pass (prompt_step) against the oracle's multi-token forward, and Transformer.forward's choice
between prompt steps and verify chunks."""

import numpy as np
import pytest
import torch

from oracle import model as om
from test_gpu_runner import (TOL, _check_codes, _check_logits, _code_diffs, _gqa128_model, _prefill,
                             _sync_frozen, build_runner, c1_model, run_steps)

pytestmark = pytest.mark.gpu


def _models(name):
    return c1_model() if name == "c1" else _gqa128_model()


# 4: the smallest; 33, 64: the 64-row GEMM; 65, 150: the many-row GEMM with a ragged last row tile and, with heads of
# 128, its K splits summed by the RoPE launch; attention row blocks of 64 that end inside a token's heads (GQA 4).
@pytest.mark.parametrize("name", ["c1", "gqa128"])
@pytest.mark.parametrize("kv", ["fp16", "fp8", "int4"])
@pytest.mark.parametrize("T,past", [(4, 0), (33, 7), (64, 0), (65, 40), (150, 0)])
def test_prompt_step_matches_oracle(dev, name, kv, T, past):
    print(f"[prompt_step] {name} kv={kv} T={T} past={past}", flush=True)
    cfg, ow, cos, sin = _models(name)
    model = om.OracleModel(cfg, ow, cos, sin)
    S = 192
    runner, cache = build_runner(cfg, ow, cos, sin, dev, S, kv)
    ocache = om.OracleKVCache(S, cfg.n_layer, cfg.n_kv_head, cfg.head_dim, kv)
    frozen = kv != "fp16"  # the oracle attends over the GPU's codes, as in the verify tests
    ocache.frozen = frozen
    rng = np.random.default_rng(T + past)
    prefix = rng.integers(0, cfg.vocab, past).tolist()
    if frozen:
        run_steps(runner, cache, prefix, dev)
    else:
        _prefill(runner, cache, ocache, model, prefix, dev)
    toks = rng.integers(0, cfg.vocab, T).tolist()
    idx = torch.tensor([toks], device=dev)
    got = runner.prompt_step(idx, past, past, "all", min(T, 32))[0].float().cpu().numpy()
    if frozen:
        _sync_frozen(ocache, cache, past, S)
    ref = model.forward(toks, ocache, return_all_logits=True)
    for t in range(T):
        _check_logits(got[t], ref[t], f"prompt token {t} of {T}")
    if frozen:
        _check_codes(kv, _code_diffs(kv, ocache), f"prompt {name} T={T}")
    norm = runner.get_last_norm(min(T, 32))
    last = runner.prompt_step(idx, past, past, "last", 1)[0, 0].float().cpu().numpy()
    _check_logits(last, ref[-1], "last token's logits alone")
    assert np.abs(norm[0, -1].float().cpu().numpy() - runner.get_last_norm(1)[0, 0].float().cpu().numpy()).max() == 0
    cache.total_seen_tokens[:] = [past + T] * cfg.n_layer
    tok = int(rng.integers(0, cfg.vocab))
    got = run_steps(runner, cache, [tok], dev)[0]
    if frozen:
        _sync_frozen(ocache, cache, past + T, S)
    _check_logits(got, model.forward([tok], ocache)[-1], "step after the prompt")


def test_prompt_step_rejects_rows_past_the_cache(dev):
    cfg, ow, cos, sin = c1_model()
    runner, _ = build_runner(cfg, ow, cos, sin, dev, 64)
    idx = torch.zeros((1, 40), dtype=torch.int64, device=dev)
    with pytest.raises(RuntimeError, match="rows at slot"):
        runner.prompt_step(idx, 25, 25)
    with pytest.raises(RuntimeError, match="below"):
        runner.prompt_step(idx[:, :3], 0, 0)
    with pytest.raises(RuntimeError, match="norm_rows"):
        runner.prompt_step(idx, 0, 0, "last", 41)


@pytest.mark.parametrize("ring,S,T", [(False, 128, 100), (True, 64, 150), (True, 128, 150), (False, 96, 70)])
@pytest.mark.parametrize("every", [False, True])
def test_forward_prompt_equals_verify_chunks(dev, ring, S, T, every):
    """Transformer.forward against the same tokens as 32-token verify chunks: contiguous prompts, and ring caches
    whose end falls inside the prompt (the chunks after it attend over all slots, as verify_step's do)."""
    from axiomlm_amd.cache import StaticKVCache
    from axiomlm_amd.transformer import ModelConfig, Transformer

    cfg = ModelConfig(block_size=256, vocab_size=1024, n_layer=2, n_head=4, n_embd=256, rms_norm_eps=1e-5,
                      tie_word_embeddings=False)
    g = torch.Generator(device=dev)
    g.manual_seed(2)
    r = lambda *s: (torch.randn(*s, generator=g, device=dev) * 0.02).half()  # noqa: E731
    sd = {"transformer.wte.weight": r(1024, 256), "lm_head.weight": r(1024, 256),
          "transformer.ln_f.weight": 1 + r(256)}
    for i in range(2):
        pre = f"transformer.h.{i}."
        sd.update({pre + "ln_1.weight": 1 + r(256), pre + "ln_2.weight": 1 + r(256), pre + "attn.c_attn.weight": r(768, 256),
                   pre + "attn.c_proj.weight": r(256, 256), pre + "mlp.w_gate.weight": r(cfg.hidden, 256),
                   pre + "mlp.w_up.weight": r(cfg.hidden, 256), pre + "mlp.w_down.weight": r(256, cfg.hidden)})
    idx = torch.randint(0, 1024, (1, T), generator=g, device=dev)

    def run(chunks):
        model = Transformer(cfg, sd, device=dev).quantize("q4_rtn")
        cache = StaticKVCache(1, S, 2, 4, 64, device=dev, ring_buffer=ring)
        if not chunks:
            out = model.forward(idx, kv_caches=cache, return_all_logits=every)[0].clone()
        else:
            out = torch.cat([model.forward(idx[:, t:t + 32], kv_caches=cache, return_all_logits=True)[0].clone()
                             for t in range(0, T, 32)], dim=1)
            out = out if every else out[:, -1:]
        n = (T - 1) % 32 + 1
        return out, cache, model.get_decode_runner(cache).get_last_norm(n)

    a, ca, na = run(False)
    b, cb, nb = run(True)
    assert a.shape == b.shape == (1, T if every else 1, 1024)
    assert ca.total_seen_tokens == cb.total_seen_tokens and ca.layer_seq_lens == cb.layer_seq_lens
    # both within the oracle bar of the same values
    assert (a.float() - b.float()).abs().max().item() <= 2 * TOL
    assert (na.float() - nb.float()).abs().max().item() <= 2e-2
    used = min(T, S)
    assert (ca.cache[..., :used, :].float() - cb.cache[..., :used, :].float()).abs().max().item() <= 2e-2


# Rows per GEMM: 5 the smallest, 16-64-row tiles with remainders, several row blocks; K = 704 ends inside a stage.
@pytest.mark.parametrize("T", [5, 17, 40, 64, 131])
def test_fp16_weights_prompt_matches_oracle(dev, T):
    print(f"[fp16_prompt] T={T}", flush=True)
    cfg = om.OracleConfig(n_layer=2, n_head=4, n_kv_head=2, d_model=256, hidden=704, vocab=1000, eps=1e-5,
                          block_size=256)
    ow = om.fp16_model(cfg, om.make_float_weights(cfg, seed=7))
    rng = np.random.default_rng(T)
    ow.c_attn_b = [(rng.standard_normal((cfg.n_head + 2 * cfg.n_kv_head) * cfg.head_dim) * 0.1).astype(np.float16)
                   for _ in range(cfg.n_layer)]
    cos, sin = om.rope_tables(cfg.head_dim, cfg.block_size)
    runner, cache = _fp16_runner(cfg, ow, cos, sin, dev, 192)
    toks = rng.integers(0, cfg.vocab, T).tolist()
    got = runner.prompt_step(torch.tensor([toks], device=dev), 0, 0, "all", 1)[0].float().cpu().numpy()
    model = om.OracleModel(cfg, ow, cos, sin)
    ref = model.forward(toks, om.OracleKVCache(192, cfg.n_layer, cfg.n_kv_head, cfg.head_dim, "fp16"),
                        return_all_logits=True)
    for t in range(T):
        _check_logits(got[t], ref[t], f"fp16 prompt token {t} of {T}")


def test_fp16_weights_long_prompt_matches_four_token_steps(dev):
    """Four weight tiles per wave (64-row tiles of a large launch) against the GEMVs, four tokens at a time."""
    cfg = om.OracleConfig(n_layer=1, n_head=8, n_kv_head=4, d_model=512, hidden=5632, vocab=1000, eps=1e-5,
                          block_size=1024)
    ow = om.fp16_model(cfg, om.make_float_weights(cfg, seed=3))
    cos, sin = om.rope_tables(cfg.head_dim, cfg.block_size)
    T = 932
    idx = torch.from_numpy(np.random.default_rng(4).integers(0, cfg.vocab, (1, T))).to(dev)
    runner, cache = _fp16_runner(cfg, ow, cos, sin, dev, 1024)
    got = runner.prompt_step(idx, 0, 0, "all", 1)[0].float().cpu().numpy()
    runner, cache = _fp16_runner(cfg, ow, cos, sin, dev, 1024)
    for t0 in range(0, T, 4):
        ref = runner.prompt_step(idx[:, t0:t0 + 4], t0, t0, "all", 1)[0].float().cpu().numpy()
        for t in range(4):
            _check_logits(got[t0 + t], ref[t], f"fp16 prompt token {t0 + t}")


def _fp16_runner(cfg, ow, cos, sin, dev, S):
    from axiomlm_amd.cache import StaticKVCache
    from axiomlm_amd.runner import DecodeRunner

    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).to(dev)  # noqa: E731
    cache = StaticKVCache(1, S, cfg.n_layer, cfg.n_kv_head, cfg.head_dim, device=dev, cache_dtype="fp16")
    runner = DecodeRunner(t(ow.wte_p), t(np.stack([cos, sin], axis=-1).astype(np.float32)), [t(x) for x in ow.ln1],
                          [t(x) for x in ow.c_attn_p], [t(x) for x in ow.c_proj_p], [t(x) for x in ow.ln2],
                          [t(x) for x in ow.gu_p], [t(x) for x in ow.wd_p], t(ow.lnf), cache.k_caches, cache.v_caches,
                          cfg.n_head, cfg.n_kv_head, cfg.head_dim, cfg.eps, lm_head_w=t(ow.lmh_p),
                          c_attn_bs=[t(b) for b in (ow.c_attn_b or [])], k_scales=cache.k_scales,
                          v_scales=cache.v_scales, kv_dtype="fp16")
    return runner, cache


# 33: 48-row tiles; 64: one block of 64; 75 and 150: several blocks with a ragged last one; with heads of 128 the QKV
# splits are summed by the RoPE launch; SwiGLU and residual epilogues (fused with the norm) of split and unsplit K.
@pytest.mark.parametrize("mode,kv,hd", [("q8", "fp16", 64), ("q8", "fp16", 128), ("q8", "fp8", 128),
                                        ("q4_k_m", "fp16", 128)])
@pytest.mark.parametrize("T,past", [(33, 0), (64, 20), (75, 7), (150, 0)])
def test_q8_prompt_matches_oracle(dev, mode, kv, hd, T, past):
    print(f"[q8_prompt] {mode} kv={kv} hd={hd} T={T} past={past}", flush=True)
    cfg = om.OracleConfig(n_layer=2, n_head=512 // hd, n_kv_head=256 // hd, d_model=512, hidden=1408, vocab=1000,
                          eps=1e-5, block_size=256)
    ow = om.pack_model(cfg, om.make_float_weights(cfg, seed=6), mode)
    cos, sin = om.rope_tables(cfg.head_dim, cfg.block_size)
    model = om.OracleModel(cfg, ow, cos, sin)
    S = 192
    runner, cache = build_runner(cfg, ow, cos, sin, dev, S, kv)
    ocache = om.OracleKVCache(S, cfg.n_layer, cfg.n_kv_head, cfg.head_dim, kv)
    ocache.frozen = kv != "fp16"
    rng = np.random.default_rng(T + past)
    prefix = rng.integers(0, cfg.vocab, past).tolist()
    if ocache.frozen:
        run_steps(runner, cache, prefix, dev)
    else:
        _prefill(runner, cache, ocache, model, prefix, dev)
    toks = rng.integers(0, cfg.vocab, T).tolist()
    got = runner.prompt_step(torch.tensor([toks], device=dev), past, past, "all", 1)[0].float().cpu().numpy()
    if ocache.frozen:
        _sync_frozen(ocache, cache, past, S)
    ref = model.forward(toks, ocache, return_all_logits=True)
    for t in range(T):
        _check_logits(got[t], ref[t], f"{mode} prompt token {t} of {T}")
    if ocache.frozen:
        _check_codes(kv, _code_diffs(kv, ocache), f"{mode} prompt T={T}")


@pytest.mark.parametrize("mode", ["q4_rtn", "q8"])
def test_long_prompt_equals_verify_chunks(dev, mode):
    """700 tokens: many row blocks of the GEMMs, split K with the residual and norm reduced together, causal attention
    of many row blocks; against verify chunks of 32 tokens, both within the oracle bar of the same values."""
    cfg = om.OracleConfig(n_layer=2, n_head=8, n_kv_head=2, d_model=1024, hidden=2816, vocab=1000, eps=1e-5,
                          block_size=1024)
    ow = om.pack_model(cfg, om.make_float_weights(cfg, seed=8), mode)
    cos, sin = om.rope_tables(cfg.head_dim, cfg.block_size)
    T = 700
    idx = torch.from_numpy(np.random.default_rng(3).integers(0, cfg.vocab, (1, T))).to(dev)
    runner, cache = build_runner(cfg, ow, cos, sin, dev, 768)
    got = runner.prompt_step(idx, 0, 0, "all", 1)[0].float()
    runner2, cache2 = build_runner(cfg, ow, cos, sin, dev, 768)
    for t0 in range(0, T, 32):
        n = min(32, T - t0)
        ref = runner2.verify_step(idx[:, t0:t0 + n], t0, t0, t0 + n)[0].float()
        assert (got[t0:t0 + n] - ref).abs().max().item() <= 2 * TOL, f"tokens {t0}.."
    assert (cache.cache[..., :T, :].float() - cache2.cache[..., :T, :].float()).abs().max().item() <= 2e-2


@pytest.mark.parametrize("H,Hkv,hd", [(32, 32, 64), (32, 8, 128)])
def test_prompt_attention_is_a_mean_of_values(dev, H, Hkv, hd):
    """Equal values under unequal scores come out as they went in, whatever fp16 makes of the weights: the weights are
    summed as they are multiplied (2^-22 of the value at most, far below its own rounding).  The first 40 tokens set a
    maximum that later keys exceed by five to seven powers of two, another amount for each head.

    An fp16 model that shows the attention output in dims 8 and up: embeddings have a one in coordinate 0 (query and
    value) and in coordinate 1 or 2 (the key's score), the O projection and the head are the identity, the MLP is zero and
    RoPE does not rotate.  The first token sees its own value only."""
    from axiomlm_amd.cache import StaticKVCache
    from axiomlm_amd.runner import DecodeRunner

    d, T, S = H * hd, 600, 640
    z = lambda *s: torch.zeros(*s, dtype=torch.float16, device=dev)  # noqa: E731
    wte = z(2, d)
    wte[:, 0] = 1
    wte[0, 1] = wte[1, 2] = 1
    n0 = (d / 2) ** 0.5  # a normalized one
    qkv = z(d + 2 * Hkv * hd, d)
    qkv[0:d:hd, 0] = 1 / n0
    kv = d + Hkv * hd
    qkv[d:kv:hd, 2] = (torch.linspace(5, 7, Hkv, device=dev) * np.log(2) * hd ** 0.5 / n0).half()
    qkv[kv:, 0] = 1.97 / n0
    for h in range(Hkv):
        qkv[kv + h * hd:kv + h * hd + 8, 0] = 0
    one = torch.ones(d, dtype=torch.float16, device=dev)
    eye = torch.eye(d, dtype=torch.float16, device=dev)
    freqs = torch.stack([torch.ones(S, hd // 2), torch.zeros(S, hd // 2)], -1).to(dev)
    cache = StaticKVCache(1, S, 1, Hkv, hd, device=dev)
    runner = DecodeRunner(wte, freqs, [one], [qkv], [eye], [one], [z(512, d)], [z(d, 256)], one, cache.k_caches,
                          cache.v_caches, H, Hkv, hd, 1e-5, lm_head_w=eye, kv_dtype="fp16")
    idx = (torch.arange(T, device=dev) >= 40).long()[None]
    got = runner.prompt_step(idx, 0, 0, "all", 1)[0].view(T, H, hd)[:, :, 8:]
    v = cache.cache[0, 1, 0, :, :T, 8:]
    assert (v == v[:, :1]).all() and v.min() > 1.9 and (cache.cache[0, 0, 0, :, 40, 0] > 0).all()
    assert (got[0] != 0).all()
    assert (got == got[0]).all(), (got != got[0]).float().mean().item()


# Row blocks of 64 tokens, whose second half starts at token 32; keys aligned to the blocks of 32 and not.
@pytest.mark.parametrize("heads", [4, 2])
@pytest.mark.parametrize("past", [0, 7])
@pytest.mark.parametrize("at", [32, 47, 75])
def test_token_that_is_not_finite_leaves_earlier_tokens_alone(dev, heads, past, at):
    """A token whose keys and values are NaN reaches no token before its own 16, in any layer."""
    cfg = om.OracleConfig(n_layer=2, n_head=heads, n_kv_head=heads, d_model=256, hidden=704, vocab=1000, eps=1e-5,
                          block_size=256)
    ow = om.fp16_model(cfg, om.make_float_weights(cfg, seed=7))
    ow.wte_p = ow.wte_p.copy()
    ow.wte_p[999] = np.inf
    cos, sin = om.rope_tables(cfg.head_dim, cfg.block_size)
    toks = torch.from_numpy(np.random.default_rng(at).integers(0, 999, (1, past + 150))).to(dev)
    out = []
    for tok in (999, 998):
        runner, _ = _fp16_runner(cfg, ow, cos, sin, dev, 192)
        toks[0, past + at] = tok
        if past:
            runner.prompt_step(toks[:, :past], 0, 0)
        out.append(runner.prompt_step(toks[:, past:], past, past, "all", 1)[0].clone())
    before = at // 16 * 16
    assert torch.isnan(out[0][at]).all() and torch.isfinite(out[1]).all()
    assert torch.equal(out[0][:before], out[1][:before])
