"""GPU: Q4_0, Q4_1, Q5_0 and Q5_1 as planes, on both sides of the line between tiles of one and of two blocks (more than 2048
columns, whole pairs of blocks): single products, slices and pairs of a fused launch, Neox pairs, and the batched product over
rows that end inside a unit of 256 columns.

The bound of single products is the rounding of the activations to 16-bit fixed point per block (2^-16 of a block's largest
value per element, far below it after summation): 5e-4 of the largest result, as in test_gpu_gemv.py."""
import numpy as np
import pytest

import npref
import oracle as orc
import wgml_amd as W

pytestmark = pytest.mark.gpu
LEGACY = [W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1]


@pytest.mark.parametrize("qtype", LEGACY)
@pytest.mark.parametrize("ncols", [32, 64, 96, 2016, 2048, 2080, 2112, 4064, 4096, 4128, 4160, 8224, 12352])
def test_products_around_the_tile_line(gpu, qtype, ncols):
    nrows = 21
    raw = npref.random_blocks(qtype, nrows * ncols // 32, seed=qtype + ncols)
    x = W.rng_normal(ncols, ncols)
    m = W.GpuQuantMatrix(gpu, qtype, nrows, ncols, raw)
    out = W.GpuVector.uninit(gpu, nrows)
    W.GemvQuant.from_device(gpu).dispatch(out, m, W.GpuVector.init(gpu, x))
    _, ref = orc.gemv_quant(qtype, raw, nrows, ncols, x)
    assert np.abs(out.read() - ref).max() <= 5e-4 * np.abs(ref).max()


@pytest.mark.parametrize("qtype", LEGACY)
@pytest.mark.parametrize("dim,hidden", [(2048, 2112), (2112, 2080), (2304, 4160)])
@pytest.mark.parametrize("neox", [False, True])
def test_models_around_the_tile_line(gpu, qtype, dim, hidden, neox):
    # the fused Q/K/V and gate/up launches against one launch per matrix, which differ in the order of a row's sums only
    from wgml_amd.models import HostMatrix, Llama2, Llama2Config, LlamaModelType, synth_llama

    cfg = Llama2Config(dim=dim, hidden_dim=hidden, n_layers=1, n_q_heads=dim // 64, n_kv_heads=dim // 64, vocab_size=320,
                       seq_len=64, rope_base_freq=10000.0, rms_norm_eps=1e-5)
    w = synth_llama(cfg, seed=7, scheme="f32")
    rng = np.random.default_rng(5)
    for layer in w.layers:
        for name, v in list(layer.items()):
            if isinstance(v, HostMatrix):
                layer[name] = HostMatrix(qtype, v.nrows, v.ncols, npref.encode_simple(qtype, v.data.view(np.float32)))
        if neox:
            for name, n in (("attn_q_bias", dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
                layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    got = {}
    for level in (3, 2):
        m = Llama2(gpu, cfg, LlamaModelType.Qwen2 if neox else LlamaModelType.Llama).load(w)
        m.set_fusion(level)
        for pos, tok in enumerate((5, 17, 200)):
            m.forward(tok, pos)
        got[level] = m.logits()
        if level == 3:  # the batched products see the same weights: within the rounding of the steps' activations
            m.prefill(np.array([5, 17, 200], np.uint32), 0)
            assert np.abs(m.logits() - got[3]).max() <= 1e-3 * np.abs(got[3]).max()
    assert np.abs(got[3] - got[2]).max() <= 1e-5 * np.abs(got[2]).max()
