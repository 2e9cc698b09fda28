"""GPU: the Q/K/V launch that rotates Neox pairs (rows i and i + head_size / 2 of a head) against the level below it,
which has one rope launch per layer, over head sizes that are no powers of two and the smallest and largest, every
format, and both workgroup sizes (768 threads run where a launch has 2049 to 4096 row pairs: 3584 + 2 x 512 rows).

Both levels do the same arithmetic but for the order of a row's fp32 sums (level 2 runs the same products one
matrix per launch): logits agree to 1e-5 of the largest (16-bit activations quantize alike on both sides)."""
import numpy as np
import pytest

import npref
import wgml_amd as W
from wgml_amd.models import HostMatrix, Llama2, Llama2Config, LlamaModelType, synth_llama

pytestmark = pytest.mark.gpu
SIMPLE = [W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1, W.Q5_K, W.Q8_K]


def compare(gpu, scheme, heads, kv_heads, dim, n_layers=2):
    cfg = Llama2Config(dim=dim, hidden_dim=512, n_layers=n_layers, n_q_heads=heads, n_kv_heads=kv_heads, vocab_size=320,
                       seq_len=64, rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=5, scheme=scheme if isinstance(scheme, str) else "f32")
    rng = np.random.default_rng(3)
    for layer in w.layers:
        for name, v in list(layer.items()):
            if not isinstance(scheme, str) and isinstance(v, HostMatrix):
                layer[name] = HostMatrix(scheme, v.nrows, v.ncols, npref.encode_simple(scheme, v.data.view(np.float32)))
        for name, n in (("attn_q_bias", dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
            layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    got = {}
    for level in (3, 2):
        m = Llama2(gpu, cfg, LlamaModelType.Qwen2).load(w)
        m.set_fusion(level)
        for pos, tok in enumerate((5, 17, 200, 3, 111)):
            m.forward(tok, pos)
        if level == 3:  # as many launches as with neighbouring pairs (f32 matrices have a rope launch per layer)
            neighbours = Llama2(gpu, cfg, LlamaModelType.Llama).load(w)
            neighbours.set_fusion(3)
            neighbours.forward(5, 4)
            assert m.launches_per_token() == neighbours.launches_per_token() + (n_layers if scheme == "f32" else 0)
        got[level] = [m.logits()] + [np.asarray(m.kv_download(l, 0, 0, 5)) for l in range(n_layers)]
    for a, b in zip(got[3], got[2]):
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


@pytest.mark.parametrize("scheme,heads,kv_heads,dim", [("q8_0", 128, 64, 256), ("q4_k_m", 64, 16, 256), ("q8_0", 2, 2, 512),
                                                       ("q4_k_m", 8, 4, 768), ("q8_0", 10, 5, 960), ("q8_0", 16, 16, 96),
                                                       ("q4_k_m", 24, 8, 768), ("f32", 4, 2, 256)])
def test_neox_pairs_in_the_qkv_launch(gpu, scheme, heads, kv_heads, dim):
    compare(gpu, scheme, heads, kv_heads, dim)


@pytest.mark.parametrize("waves", [12, 16])
@pytest.mark.parametrize("scheme", ["q8_0", "q4_k", "q6_k", "q4_k_m"] + SIMPLE)
def test_formats_and_workgroup_sizes(gpu, scheme, waves):
    gpu.set_tuning(gpu.TUNE_GEMV_WAVES_PER_WG, waves)
    try:
        compare(gpu, scheme, 8, 4, 768)
    finally:
        gpu.set_tuning(gpu.TUNE_GEMV_WAVES_PER_WG, 0)


def test_launch_that_takes_the_smaller_workgroups(gpu):
    compare(gpu, "q8_0", 28, 4, 3584, n_layers=1)
