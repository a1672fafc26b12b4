"""One-token steps of an int8 model around the contexts at which a head's
positions stop fitting one workgroup of the split attention: each step's
logits against those of the same tokens fed as one prompt (other kernels
throughout: exact-split products and tile attention), within the forward
pass tests' 1e-4 of the largest logit; the chunks' merge inside the launch
and in its own launch give the same bits."""
import numpy as np
import pytest

from tests import engine, inputs

em = engine.load()
pytestmark = pytest.mark.gpu


def build(heads, kv_heads, hs, seed):
    D, H, V = heads * hs, 320, 500
    KV = kv_heads * hs
    n = iter(range(seed, seed + 100))
    w = lambda *s: inputs.normal(s, 0.05, next(n))  # noqa: E731
    ones = np.ones(D, np.float32)
    cfg = dict(dim=D, hidden_dim=H, n_layers=2, n_heads=heads, n_kv_heads=kv_heads, vocab_size=V,
               seq_len=320)
    weights = dict(token_embedding=inputs.normal((V, D), 1.0, next(n)), rms_final=ones,
                   wcls=w(D, V), layers=[dict(rms_att=ones, wqkv=w(D, D + 2 * KV), wo=w(D, D),
                                              rms_ffn=ones, w13=w(D, 2 * H), w2=w(H, D))
                                         for _ in range(2)])
    return cfg, weights


@pytest.mark.parametrize("heads,kv_heads,hs", [(4, 4, 48), (2, 2, 64), (4, 4, 32), (4, 2, 48)])
def test_steps_match_prompts(heads, kv_heads, hs, monkeypatch):
    cfg, w = build(heads, kv_heads, hs, 9100 + hs)
    w["wcls"] = np.ascontiguousarray(w["wcls"][:, :496])  # strips need 16-column groups
    cfg["vocab_size"] = 496
    w["token_embedding"] = w["token_embedding"][:496]
    model = em.Model(cfg, w, q8=True)
    monkeypatch.setenv("EM_DECODE_MERGE_KERNEL", "1")
    apart = em.Model(cfg, w, q8=True)
    monkeypatch.setenv("EM_DECODE_MERGE_KERNEL", "0")
    inside = em.Model(cfg, w, q8=True)
    monkeypatch.delenv("EM_DECODE_MERGE_KERNEL")
    tokens = [(p * 17 + 3) % 496 for p in range(300)]
    for ctx in (30, 62, 63, 64, 127, 128, 129, 254, 255, 256, 257, 299):
        for m in (model, apart, inside):
            m.forward(tokens[:ctx], 0)
        got = model.forward(tokens[ctx], ctx)
        assert np.array_equal(got, apart.forward(tokens[ctx], ctx)), ctx
        assert np.array_equal(got, inside.forward(tokens[ctx], ctx)), ctx
        want = model.forward(tokens[:ctx + 1], 0)
        assert np.abs(got - want).max() <= 1e-4 * np.abs(want).max(), ctx
