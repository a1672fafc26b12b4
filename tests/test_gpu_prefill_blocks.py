"""Prompts of an int8 model at row counts where its products take three 16-row
blocks a workgroup with the RoPE and cache write of the qkv product, and the
SwiGLU of the gate | up product, in their epilogues: the same bits as the plain
products followed by the separate kernels (whose own epilogue test_gpu_split_blocks.py
holds against 64-bit products), over two layers, so that every row's q, k, v and
SwiGLU reach the logits, and for a decode step on the cache that the prompt left."""
import numpy as np
import pytest

from tests import engine, inputs

em = engine.load()
pytestmark = pytest.mark.gpu


# 16 heads of 128, hidden 2816: gate | up three-block from 369 rows; qkv from
# 337 to 480 rows on 16 kv heads, from 513 on 8. 370 and 401 leave the last
# workgroup's rows ragged, 480 fills them.
@pytest.mark.parametrize("kv_heads,rows", [(16, (370, 401, 480)), (8, (513, 515))])
def test_fused_epilogues_give_the_same_bits(kv_heads, rows, monkeypatch):
    D, H, V, hs = 2048, 2816, 512, 128
    KV = kv_heads * hs
    w = lambda i, *s: inputs.normal(s, 0.03, 9500 + i)  # noqa: E731
    layer = dict(rms_att=inputs.uniform((D,), 0.5, 1.5, 9501), wqkv=w(2, D, D + 2 * KV),
                 wo=w(3, D, D), rms_ffn=inputs.uniform((D,), 0.5, 1.5, 9504), w13=w(5, D, 2 * H),
                 w2=w(6, H, D))
    cfg = dict(dim=D, hidden_dim=H, n_layers=2, n_heads=16, n_kv_heads=kv_heads, vocab_size=V,
               seq_len=max(rows) + 1)
    weights = dict(token_embedding=inputs.normal((V, D), 1.0, 9507),
                   rms_final=np.ones(D, np.float32), wcls=w(8, D, V), layers=[layer, layer])
    monkeypatch.setenv("EM_PREFILL_ROPE_FUSION", "0")
    monkeypatch.setenv("EM_MODEL_SWIGLU_FUSION", "0")
    apart = em.Model(cfg, weights, q8=True)
    monkeypatch.delenv("EM_PREFILL_ROPE_FUSION")
    monkeypatch.delenv("EM_MODEL_SWIGLU_FUSION")
    fused = em.Model(cfg, weights, q8=True)
    tokens = [(p * 17 + 3) % V for p in range(max(rows) + 1)]
    for n in rows:
        want, got = apart.forward(tokens[:n], 0), fused.forward(tokens[:n], 0)
        assert np.isfinite(got).all() and np.abs(got).max() > 0.1
        assert np.array_equal(got, want), n
        assert np.array_equal(fused.forward(tokens[n], n), apart.forward(tokens[n], n)), n
