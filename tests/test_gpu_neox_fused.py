"""GPU: the Q/K/V launch that rotates Neox pairs (rows i and i + head_size / 2 of a head) against the level below it,
which has one rope launch per layer, over head sizes that are no powers of two and the smallest and largest.

Both levels do the same arithmetic but for the order of a row's fp32 sums (level 2 runs the same products one
matrix per launch): logits agree to 1e-5 of the largest (16-bit activations quantize alike on both sides)."""
import numpy as np
import pytest

import wgml_amd as W
from wgml_amd.models import Llama2, Llama2Config, LlamaModelType, synth_llama

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scheme,heads,kv_heads,dim", [("q8_0", 128, 64, 256), ("q4_k_m", 64, 16, 256), ("q8_0", 2, 2, 512),
                                                       ("q4_k_m", 8, 4, 768), ("q8_0", 10, 5, 960), ("q8_0", 16, 16, 96),
                                                       ("q4_k_m", 24, 8, 768), ("f32", 4, 2, 256)])
def test_neox_pairs_in_the_qkv_launch(gpu, scheme, heads, kv_heads, dim):
    cfg = Llama2Config(dim=dim, hidden_dim=512, n_layers=2, n_q_heads=heads, n_kv_heads=kv_heads, vocab_size=320,
                       seq_len=64, rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=5, scheme=scheme)
    rng = np.random.default_rng(3)
    for layer in w.layers:
        for name, n in (("attn_q_bias", dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
            layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    got = {}
    for level in (3, 2):
        m = Llama2(gpu, cfg, LlamaModelType.Qwen2).load(w)
        m.set_fusion(level)
        for pos, tok in enumerate((5, 17, 200, 3, 111)):
            m.forward(tok, pos)
        got[level] = [m.logits()] + [np.asarray(m.kv_download(l, 0, 0, 5)) for l in range(2)]
    for a, b in zip(got[3], got[2]):
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()
