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
GQA = [0, 1, 3, 31, 32, 127, 512, 513, 1025, 2100]


@pytest.mark.parametrize("heads,lengths", [((4, 2, 64), GQA), ((8, 2, 128), GQA), ((16, 1, 64), GQA),
                                           ((4, 4, 64), [7998, 7999, 8100])])
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
