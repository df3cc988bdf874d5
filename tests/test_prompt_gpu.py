"""Prompts of more than 16 rows (many-row GEMMs and the prompt attention) against
a float64 forward, at the edges of their tiles: rows around 32 / 48 / 64 / 128,
behind an empty, a ragged and a long prefix (keys in one range or split), head
dims 64 and 128, grouped-query heads, mixed weight types."""
import numpy as np
import pytest

from llama_util import NumpyLlama, load, make_mixed_tensors, make_tensors

pytestmark = pytest.mark.gpu

BASE = dict(n_layers=2, vocab=640, max_ctx=1024, rms_eps=1e-5, rope_base=10000.0)
CONFIGS = {
    "d64_gqa_q4_0": (dict(BASE, dim=512, n_heads=8, n_kv_heads=2, ffn=1376), lambda o, c: make_tensors(o, c, 2, 5)),
    "d128_q4_k": (dict(BASE, dim=512, n_heads=4, n_kv_heads=4, ffn=1536), lambda o, c: make_tensors(o, c, 12, 6,
                                                                                              norm_std=0.1)),
    "d128_gqa_mixed": (dict(BASE, dim=768, n_heads=6, n_kv_heads=2, ffn=1536), lambda o, c: make_mixed_tensors(o, c, 7)),
}
# rows of consecutive calls on one cache
CALLS = [(17,), (48, 49), (3, 64, 65), (128, 129), (300, 33, 16, 211), (700, 17, 307)]


@pytest.mark.parametrize("name", CONFIGS)
def test_prompt_forward_matches_float64(pkg, ctx, ora, name):
    cfg, make = CONFIGS[name]
    tensors = make(ora, cfg)
    # max error / rms of the logits and of the cache.  Fp16 Q, K and V on both sides round the other way where fp32 and
    # float64 straddle a rounding boundary, as in the 16-row forward (the same bounds there).  Mixed fused weights and
    # Q6_K are held rounded to fp16 besides (2^-11 of each weight: about 3e-4 of a dot product's rms, 5 sigma of it
    # through two layers)
    ltol, ctol = (1e-2, 5e-3) if "mixed" in name else (2e-3, 1e-3)
    g = pkg.Model(ctx, **cfg)
    load(g, tensors)
    tokens = np.random.default_rng(8).integers(0, cfg["vocab"], cfg["max_ctx"]).astype(np.int32)
    ref = NumpyLlama(ora, tensors, cfg)  # causal: the last rows of any call are rows of one forward
    # the reference's logits of every position (its forward returns them all)
    want = ref.forward(tokens, 0)
    scale = np.sqrt((want ** 2).mean())
    for rows in CALLS:
        pos = 0
        for m in rows:
            n = min(16, m)
            print(f"{name}: {m} rows at {pos}", flush=True)
            got = g.forward(tokens[pos:pos + m], pos, n_logits=n).astype(np.float64)
            pos += m
            assert np.abs(got - want[pos - n:pos]).max() / scale <= ltol
        for layer in range(cfg["n_layers"]):
            k, v = (ora.h2f_fast(x).astype(np.float64).reshape(pos, cfg["n_kv_heads"], -1)
                    for x in g.kv_io(layer, 0, 0, pos))
            for a, b in ((k, ref.kc[layer][:pos]), (v, ref.vc[layer][:pos])):
                assert (np.abs(a - b) <= np.abs(b) * 2.0 ** -10 + ctol * np.sqrt((b ** 2).mean())).all()
    g.close()
