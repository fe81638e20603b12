"""Decode steps whose attention takes the reduce-merged splits: grouped-query heads at every length (one to 64 splits),
and few heads over a long cache, against the oracle on the same cache."""

import numpy as np
import pytest
import torch

from oracle import model as om
from test_gpu_runner import _check_logits, _sync_frozen, build_runner

pytestmark = pytest.mark.gpu


def _model(n_head, n_kv_head, hd):
    cfg = om.OracleConfig(n_layer=1, n_head=n_head, n_kv_head=n_kv_head, d_model=n_head * hd, hidden=256, vocab=256,
                          eps=1e-5, block_size=9000)
    ow = om.pack_model_rtn(cfg, om.make_float_weights(cfg, seed=5))
    return (cfg, ow, *om.rope_tables(hd, 9000, 10000.0))


# The smallest caches (fewer keys than splits), block edges, each doubling of the split count and its last length.
GQA = [0, 1, 3, 30, 31, 32, 127, 255, 256, 512, 513, 1025, 2100]


@pytest.mark.parametrize("heads,lengths", [((4, 2, 64), GQA), ((8, 2, 128), GQA), ((16, 1, 64), GQA),
                                           # two and four groups of four rows for both head sizes, a ragged group
                                           ((6, 1, 64), [40, 300]), ((8, 1, 128), [40, 300]), ((12, 1, 128), [40, 300]),
                                           ((4, 4, 64), [7998, 7999, 8100]),
                                           # more than sixteen query heads per KV head: the vector kernel
                                           ((32, 1, 64), [0, 40, 600, 8010])])
@pytest.mark.parametrize("kv", ["fp16", "fp8", "int4"])
def test_step_attention_matches_oracle(dev, heads, lengths, kv):
    cfg, ow, cos, sin = _model(*heads)
    S = lengths[-1] + 1
    model = om.OracleModel(cfg, ow, cos, sin)
    runner, cache = build_runner(cfg, ow, cos, sin, dev, S, kv)
    g = torch.Generator(device=dev)
    g.manual_seed(1)
    if kv == "fp16":
        cache.cache.normal_(generator=g)
    else:
        from axiomlm_amd.kernels import quantize_kv_fp8, quantize_kv_int4

        k, v = (torch.randn(1, cfg.n_kv_head, S, heads[2], generator=g, device=dev).half() for _ in range(2))
        kc, ks, vc, vs = (quantize_kv_fp8 if kv == "fp8" else quantize_kv_int4)(k, v)
        for j, (c, s) in enumerate(((kc, ks), (vc, vs))):
            cache.cache[0, j].copy_(c)
            cache.scales[0, j].copy_(s)
    rng = np.random.default_rng(2)
    for n in lengths:
        ocache = om.OracleKVCache(S, 1, cfg.n_kv_head, cfg.head_dim, kv)
        ocache.frozen = True  # the oracle reads the GPU's rows, the new one too
        tok = int(rng.integers(0, cfg.vocab))
        got = runner.step(torch.tensor([[tok]], device=dev), n, n, n + 1)[0, 0].float().cpu().numpy()
        _sync_frozen(ocache, cache, n, S)
        _check_logits(got, model.forward([tok], ocache)[-1], f"{heads} {kv} {n + 1} keys")


@pytest.mark.parametrize("heads", [(4, 2, 64), (4, 1, 128), (8, 1, 128), (16, 1, 64)])
@pytest.mark.parametrize("n", [200, 600])
def test_step_attention_keeps_small_weights(dev, heads, n):
    """Grouped-query softmax weights stay fp32: keys 2^-22 below the largest, whose values fill dims in which the
    large keys have none, keep the full precision of the result (weights as fp16 parts keep two bits of them).

    An fp16 model that shows the attention output: the token's normalized row is n0 in coordinate 0, q = n0 / 2 in dim 0
    of every head, the O projection and the head are the identity, the MLP and the new key are zero, and RoPE does not
    rotate.  The output, its sum with the residual, the norm's two products and the head round to fp16: 5 x 2^-11."""
    from axiomlm_amd.cache import StaticKVCache
    from axiomlm_amd.runner import DecodeRunner

    H, Hkv, hd = heads
    d, S = H * hd, 640
    z = lambda *s: torch.zeros(*s, dtype=torch.float16, device=dev)  # noqa: E731
    wte = z(8, d)
    wte[:, 0] = 1
    qkv = z(d + 2 * Hkv * hd, d)
    qkv[0:d:hd, 0] = 0.5
    qkv[d + Hkv * hd, 0] = 1  # the new value's dim 0: n0 itself, read back from the cache
    one = torch.ones(d, dtype=torch.float16, device=dev)
    eye = torch.eye(d, dtype=torch.float16, device=dev)
    freqs = torch.stack([torch.ones(S, hd // 2), torch.zeros(S, hd // 2)], -1).to(dev)
    cache = StaticKVCache(1, S, 1, Hkv, hd, device=dev)
    cache.cache.zero_()
    g = torch.Generator(device=dev)
    g.manual_seed(4)
    low = torch.arange(n, device=dev) % 8 != 0
    # scores q0 k0 / sqrt(hd) with q0 = sqrt(d) / 2: 0 to 0.5 of the low keys, 15.25 of the others
    k0 = torch.where(low, torch.rand(n, generator=g, device=dev) * 0.5, 15.25) * 2 / H ** 0.5
    cache.cache[0, 0, 0, :, :n, 0] = k0.half()
    v = (torch.rand(Hkv, n, hd, generator=g, device=dev) * 20000 + 10000).half()
    # each dim from three keys only, so that no two dims share a weight's error
    pick = torch.rand(Hkv, n, hd, generator=g, device=dev).masked_fill(~low[None, :, None], -1).topk(3, dim=1).indices
    v = v * z(Hkv, n, hd).scatter_(1, pick, 1)
    v[:, :, 0] = 0
    cache.cache[0, 1, 0, :, :n] = v
    runner = DecodeRunner(wte, freqs, [one], [qkv], [eye], [one], [z(512, d)], [z(d, 256)], one, cache.k_caches,
                          cache.v_caches, H, Hkv, hd, 1e-5, lm_head_w=eye, kv_dtype="fp16")
    got = runner.step(torch.zeros(1, 1, dtype=torch.int64, device=dev), n, n, n + 1)[0, 0].double()
    n0 = cache.cache[0, 1, 0, 0, n, 0].double()
    kk, vv = cache.cache[0, 0, 0, :, : n + 1, 0].double(), cache.cache[0, 1, 0, :, : n + 1].double()
    p = torch.softmax(n0 / 2 * kk / hd ** 0.5, -1)
    o = torch.matmul(p[:, None, :], vv)[:, 0].repeat_interleave(H // Hkv, 0).reshape(-1)
    x = wte[0].double() + o
    want = x / (x.square().mean() + 1e-5).sqrt()
    on = (o > 0) & (want.abs() > 2.0 ** -14)  # (below, fp16 itself has fewer bits)
    on[::hd] = False
    assert on.sum() > 0.9 * (d - H)
    assert ((got - want).abs() <= 5 * 2.0 ** -11 * want.abs())[on].all()


@pytest.mark.parametrize("heads,n", [((4, 2, 64), 40), ((4, 2, 64), 300), ((4, 2, 64), 2100), ((8, 2, 128), 600), ((4, 4, 64), 600),
                                     ((4, 4, 64), 8010)])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_step_over_a_key_that_is_not_finite(dev, heads, n, value):
    """A cached key of NaN (or of infinite score) makes the step's logits NaN, whichever launch merges the splits."""
    cfg, ow, cos, sin = _model(*heads)
    runner, cache = build_runner(cfg, ow, cos, sin, dev, n + 1)
    cache.cache.normal_()
    cache.cache[0, 0, 0, :, n // 2] = value
    got = runner.step(torch.tensor([[3]], device=dev), n, n, n + 1)
    assert torch.isnan(got).all()
