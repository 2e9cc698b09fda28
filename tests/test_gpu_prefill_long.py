"""GPU parity: runs of more than 128 prompt tokens (tiles of 128 rows x 256 tokens) against the same
prompt fed in calls of at most 128 tokens (tiles of 64 rows x all tokens), which
test_gpu_prefill.py holds against the oracle's single-token steps.

Both sides take the same operands and differ in the order of their fp32 sums only (split
precision: within 2e-4 of the largest value each, the bound of that file), or see operands whose
rounding to f16 differs where such a difference tips it (plain f16: 3e-3 each).
"""
import numpy as np
import pytest

import npref
import wgml_amd as W
from wgml_amd.models import HostMatrix, Llama2, Llama2Config, LlamaModelType, synth_llama


pytestmark = pytest.mark.gpu
SIMPLE = [W.Q4_0, W.Q4_1, W.Q5_0, W.Q5_1, W.Q5_K, W.Q8_K]


def config(dim=256, hidden=768, heads=4, kv_heads=2, seq_len=1400):
    return Llama2Config(dim=dim, hidden_dim=hidden, n_layers=2, n_q_heads=heads, n_kv_heads=kv_heads,
                        vocab_size=320, seq_len=seq_len, rope_base_freq=10000.0, rms_norm_eps=1e-5)


def weights(cfg, scheme, biases):
    rng = np.random.default_rng(11)
    w = synth_llama(cfg, seed=4, scheme="f32" if not isinstance(scheme, str) else scheme)
    for layer in w.layers:
        for name, v in list(layer.items()):
            if not isinstance(scheme, str) and isinstance(v, HostMatrix):
                layer[name] = HostMatrix(scheme, v.nrows, v.ncols, npref.encode_simple(scheme, v.data.view(np.float32)))
        layer["attn_norm"] = (1 + 0.2 * rng.standard_normal(cfg.dim)).astype(np.float32)
        if biases:
            for name, n in (("attn_q_bias", cfg.dim), ("attn_k_bias", cfg.kv_dim), ("attn_v_bias", cfg.kv_dim)):
                layer[name] = (0.1 * rng.standard_normal(n)).astype(np.float32)
    return w


def state(model, cfg, n):
    return [model.logits().copy()] + [np.asarray(model.kv_download(l, which, 0, n)).copy()
                                      for l in range(cfg.n_layers) for which in (0, 1)]


def compare(gpu, cfg, w, model_type, n, start=0, precision=1):
    toks = W.prompt_tokens(9, n, cfg.vocab_size)
    short, wide = Llama2(gpu, cfg, model_type).load(w), Llama2(gpu, cfg, model_type).load(w)
    gpu.set_gemm_precision(precision)
    try:
        for at in range(0, n, 128):
            short.prefill(toks[at:at + 128], start_pos=at)
        if start:
            wide.prefill(toks[:start])
        wide.prefill(toks[start:], start_pos=start)
    finally:
        gpu.set_gemm_precision(1)
    # the long runs are there: fewer launches than with runs of 128 (of the same length each, but for
    # the kernels that add partial sums; 257 tokens are two runs instead of three)
    assert wide.launches_per_token() < 0.8 * short.launches_per_token() * -(-(n - start) // 128)
    tol = 2 * (2e-4 if precision else 3e-3)
    for got, want in zip(state(wide, cfg, n), state(short, cfg, n)):
        assert np.isfinite(got).all()
        assert np.abs(got - want).max() <= tol * np.abs(want).max()


@pytest.mark.parametrize("precision", [1, 0], ids=["split_f16", "plain_f16"])
@pytest.mark.parametrize("n", [129, 255, 256, 257, 390, 1024, 1153])
def test_run_lengths(gpu, n, precision):
    # one tile with padding, exactly one, one and a short run, two, the longest run, a run after it
    cfg = config()
    compare(gpu, cfg, weights(cfg, "q4_k_m", False), LlamaModelType.Llama, n, precision=precision)


@pytest.mark.parametrize("precision", [1, 0], ids=["split_f16", "plain_f16"])
@pytest.mark.parametrize("scheme", ["q8_0", "q4_k", "q6_k"] + SIMPLE)
def test_formats_biases_and_context(gpu, scheme, precision):
    cfg = config()
    compare(gpu, cfg, weights(cfg, scheme, True), LlamaModelType.Qwen2, 300, start=37, precision=precision)


@pytest.mark.parametrize("k_split", [0, 1, 3, 8])
@pytest.mark.parametrize("dim,heads,kv_heads,hidden", [(96, 3, 1, 160), (320, 4, 2, 448), (512, 4, 4, 1056)])
def test_rows_and_columns_beyond_whole_tiles(gpu, k_split, dim, heads, kv_heads, hidden):
    # row counts that are no multiples of 16, 64 or 128; K with half a chunk and an odd number of chunks
    cfg = config(dim, hidden, heads, kv_heads, 260)
    gpu.set_tuning(gpu.TUNE_GEMM_K_SPLIT, k_split)
    try:
        compare(gpu, cfg, weights(cfg, "q8_0", True), LlamaModelType.Qwen2, 210)
    finally:
        gpu.set_tuning(gpu.TUNE_GEMM_K_SPLIT, 0)


@pytest.mark.parametrize("n,start", [(300, 0), (100, 37), (272, 41)])
@pytest.mark.parametrize("head_size", [16, 32, 48, 64, 80, 96, 112, 128])
def test_attention_in_four_and_in_eight_waves(gpu, head_size, n, start):
    """16 tokens per workgroup, of four waves where heads x blocks of tokens are at least as many as the 256 compute units
    (16 heads, 300 and 272 tokens: 304 and 272) and of eight below (100 tokens: 112), against a workgroup per token."""
    cfg = config(16 * head_size, 256, 16, 4, 400)
    w = weights(cfg, "q8_0", False)
    toks = W.prompt_tokens(9, start + n, cfg.vocab_size)
    got = []
    for per_token in (0, 1):
        m = Llama2(gpu, cfg, LlamaModelType.Llama).load(w)
        gpu.set_tuning(gpu.TUNE_PREFILL_ATTENTION_PER_TOKEN, per_token)
        try:
            if start:
                m.prefill(toks[:start])
            m.prefill(toks[start:], start_pos=start)
        finally:
            gpu.set_tuning(gpu.TUNE_PREFILL_ATTENTION_PER_TOKEN, 0)
        got.append(state(m, cfg, start + n))
    for a, b in zip(*got):
        assert np.isfinite(a).all() and np.abs(a - b).max() <= 2e-4 * np.abs(b).max()
